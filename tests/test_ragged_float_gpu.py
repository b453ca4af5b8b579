"""Float B of any width on the LDS-DMA rings: padded copies, rows in place
whose last 16-byte chunk is cut off by N, unaligned outputs, and the SDDMM on
rows padded with zeros."""

import numpy as np
import pytest
import torch

import cases
import oracle
import void_amd
from void_amd import _runtime, tuning

pytestmark = pytest.mark.gpu
U = 2.0 ** -24
ROUND = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}
ABS = {torch.float32: 0.0, torch.bfloat16: 0.0, torch.float16: 2.0 ** -25}


@pytest.fixture(autouse=True)
def always_pad(monkeypatch):
    monkeypatch.setattr(_runtime, "PAD_FLOAT_MIN_WORK", 1)
    monkeypatch.setattr(tuning, "PAD_FLOAT", True)


def _views(b):
    """b contiguous, in a NaN-padded aligned pitch, shifted, and column-major."""
    K, N = b.shape
    yield b
    for pitch, shift in ((-(-N // 8) * 8 + 8, 0), (N + 1, 1)):
        flat = torch.full((K * pitch + shift,), float("nan"), dtype=b.dtype, device=b.device)
        v = flat[shift:].view(K, pitch)[:, :N]
        v.copy_(b)
        yield v
    yield b.t().contiguous().t()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(1, 3), (5, 8), (64, 33), (70, 129), (33, 250)])
def test_padded_rows(gpu, dtype, shape):
    t = torch.randn(shape, device=gpu).to(dtype)
    for v in _views(t):
        for zero in (False, True):
            out = _runtime.padded_rows(v, zero_tail=zero)
            assert torch.equal(out, v) and _runtime.aligned_rows(out)
            per = 16 // t.element_size()
            if zero and shape[1] % per:
                tail = out.as_strided((shape[0], -shape[1] % per), out.stride(), out.storage_offset() + shape[1])
                assert bool((tail == 0).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("N", [1, 3, 7, 33, 130, 257])
@pytest.mark.parametrize("kern", [None, "cgd", "cgdk"])
def test_spmm_any_width(gpu, monkeypatch, dtype, N, kern):
    """Output bound: recursive fp32 summation plus one rounding of the output;
    bias and GELU-free, per-row bias included; data around C untouched."""
    if kern:
        monkeypatch.setenv("VOID_AMD_KERNEL", kern)
    case = cases.uniform_blocks(170, 203, N, 25, seed=N)
    vt = cases.make_void_tensor(case, "cpu").to(gpu).to_dtype(dtype)
    b = torch.from_numpy(case.b).to(gpu).to(dtype)
    A = torch.from_numpy(oracle.densify(vt.values.float().cpu().numpy(), case.block_rows, case.block_cols,
                                        (170, 203)).astype(np.float64)).to(gpu)
    n = 32 * int(np.bincount(case.block_rows).max())
    ref, mag = A @ b.double(), A.abs() @ b.double().abs()
    tol = n * U * mag + ROUND[dtype] * ref.abs() + ABS[dtype] + 1e-30
    wide = torch.full((170, N + 3), -7.0, device=gpu, dtype=dtype)
    for v in _views(b):
        assert bool(((void_amd.void_spmm(vt, v).double() - ref).abs() <= tol).all())
        void_amd.void_spmm(vt, v, out=wide[:, 1:N + 1])
        assert bool(((wide[:, 1:N + 1].double() - ref).abs() <= tol).all())
        assert bool((wide[:, 0] == -7).all()) and bool((wide[:, N + 1:] == -7).all())


@pytest.mark.parametrize("b_dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("N", [1, 7, 37, 130, 257])
def test_fp8_any_width(gpu, b_dtype, N):
    case = cases.uniform_blocks(100, 203, N, 14, seed=N)
    f8 = void_amd.void_tensor_to_fp8(cases.make_void_tensor(case, "cpu"))
    b = torch.from_numpy(case.b).to(gpu).to(b_dtype)
    t = f8.values_fp8.double() * f8.scaling_info.scale.double()[:, None, None]
    A = torch.zeros(128, 224, dtype=torch.float64)
    for i, (r, c) in enumerate(zip(case.block_rows, case.block_cols)):
        A[32 * r:32 * r + 32, 32 * c:32 * c + 32] = t[i]
    A = A[:100, :203].to(gpu)
    scale = torch.linspace(0.5, 2, N, device=gpu)
    ref, mag = (A @ b.double()) * scale.double(), (A.abs() @ b.double().abs()) * scale.double()
    wide = torch.full((100, N + 3), -7.0, device=gpu)
    for v in _views(b):
        void_amd.void_spmm_fp8(f8.to(gpu), v, output_dtype=torch.float32, b_scale=scale, out=wide[:, 1:N + 1])
        assert bool(((wide[:, 1:N + 1].double() - ref).abs() <= 2.0 ** -15 * mag + 1e-30).all())
        assert bool((wide[:, 0] == -7).all()) and bool((wide[:, N + 1:] == -7).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("tokens", [1, 7, 33, 130])
def test_training_step_any_width(gpu, dtype, tokens):
    """Gradients of input, tiles and bias with a token count that no chunk
    divides, for both layouts of the incoming gradient, against float64."""
    case = cases.uniform_blocks(130, 200, tokens, 20, seed=tokens)
    vt = cases.make_void_tensor(case, "cpu").to(gpu).to_dtype(dtype)
    lin = void_amd.SparseLinear(200, 130, vt).to(gpu)
    x = torch.randn(tokens, 200, device=gpu).to(dtype).requires_grad_()
    gy = torch.randn(tokens, 130, device=gpu).to(dtype)
    W = torch.zeros(160, 224, dtype=torch.float64, device=gpu)
    for t, (r, c) in enumerate(zip(case.block_rows, case.block_cols)):
        W[32 * r:32 * r + 32, 32 * c:32 * c + 32] = vt.values[t].double()
    gp = torch.zeros(tokens, 160, dtype=torch.float64, device=gpu)
    xp = torch.zeros(tokens, 224, dtype=torch.float64, device=gpu)
    gp[:, :130], xp[:, :200] = gy.double(), x.detach().double()
    pick = lambda m: torch.stack([m[32 * r:32 * r + 32, 32 * c:32 * c + 32]
                                  for r, c in zip(case.block_rows, case.block_cols)])
    refs = [(xp @ W.t())[:, :130], (gp @ W)[:, :200], pick(gp.t() @ xp), gp[:, :130].sum(0)]
    mags = [(xp.abs() @ W.abs().t())[:, :130], (gp.abs() @ W.abs())[:, :200], pick(gp.abs().t() @ xp.abs()),
            gp[:, :130].abs().sum(0)]
    for g in (gy, gy.t().contiguous().t()):
        lin.zero_grad(set_to_none=True)
        x.grad = None
        y = lin(x)
        y.backward(g)
        outs = [y.detach(), x.grad, lin.sparse_weight.values.grad, lin.bias.grad]
        for k, (o, ref, mag) in enumerate(zip(outs, refs, mags)):
            assert bool(((o.double() - ref).abs() <= 300 * U * mag + ROUND[dtype] * ref.abs() + 1e-30).all()), k


def test_small_widths_keep_one_launch(gpu, monkeypatch):
    monkeypatch.undo()
    b = torch.randn(100, 37, device=gpu)
    assert _runtime.row_major(b, 60) is b
    out = _runtime.row_major(b, 600)
    assert _runtime.aligned_rows(out) and torch.equal(out, b)


@pytest.mark.parametrize("kind", ["int8", "int8_col", "float"])
def test_tall_b_is_read_in_place(gpu, monkeypatch, kind):
    """Few tiles over a tall B: nothing of B's size is allocated, and the
    result is right (int32 exact, fp32 within its summation bound)."""
    monkeypatch.undo()
    K, N, n = 1 << 20, 101, 40
    rng = np.random.default_rng(1)
    br, bc = np.arange(n) % 16, rng.choice(K // 32, n, replace=False)
    vt = void_amd.VOIDTensor(
        values=torch.from_numpy(rng.standard_normal((n, 32, 32)).astype(np.float32)).to(gpu),
        block_rows=torch.from_numpy(br.astype(np.int32)).to(gpu), block_cols=torch.from_numpy(bc.astype(np.int32)).to(gpu),
        morton_codes=torch.zeros(n, dtype=torch.int64, device=gpu), shape=(512, K), tile_size=(32, 32),
        nnz_original=n * 1024, n_blocks=n, density=0.0)
    if kind == "float":
        a, b = vt, torch.randn(K, N, device=gpu)
        run = lambda: void_amd.void_spmm(a, b)
        tiles = vt.values.double()
    else:
        a = void_amd.quantize_void_tensor(vt)
        b = torch.randint(-128, 128, (K, N), dtype=torch.int8, device=gpu)
        if kind == "int8_col":
            b = torch.cat([b.t().contiguous(), b.t()[:, :1].contiguous()], 1)[:, :K].t()  # columns of K + 1 bytes
        run = lambda: void_amd.void_spmm_int8(a, b, epilogue="raw_i32")
        tiles = a.values.double()
    run()
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    base = torch.cuda.memory_allocated()
    out = run()
    torch.cuda.synchronize()
    assert torch.cuda.max_memory_allocated() - base < b.numel() * b.element_size() // 8
    ref = torch.zeros(512, N, dtype=torch.float64, device=gpu)
    mag = torch.zeros_like(ref)
    for t in range(n):
        bt = b[32 * bc[t]:32 * bc[t] + 32].double()
        ref[32 * br[t]:32 * br[t] + 32] += tiles[t] @ bt
        mag[32 * br[t]:32 * br[t] + 32] += tiles[t].abs() @ bt.abs()
    assert bool(((out.double() - ref).abs() <= (96 * U * mag if kind == "float" else 0)).all())
