"""Backward of the float SpMM: the SDDMM kernels (void_sddmm_f32 and the
row-grouped void_sddmm_rows_f32) against
float64 products of the same operands, and the autograd wrappers
(VOIDSpMM, SparseLinear) against float64 dense gradients.  Bound: recursive
fp32 summation, (n-1) 2^-24 sum|x y| with n the reduction length."""

import numpy as np
import pytest
import torch

import cases
import oracle
import void_amd
from void_amd import _runtime, autograd

pytestmark = pytest.mark.gpu
U = 2.0 ** -24


@pytest.mark.parametrize("grouped", [None, "tile_rows", "ring", "rows"])
@pytest.mark.parametrize("M,K,N,n,seed", [(1024, 2048, 512, 600, 0), (100, 70, 36, 6, 1), (64, 96, 130, 5, 2),
                                          (256, 4096, 66, 300, 3), (96, 128, 1000, 12, 4), (70, 1000, 20, 40, 5),
                                          (500, 300, 8, 30, 6)])
def test_sddmm_tiles(gpu, M, K, N, n, seed, grouped, monkeypatch):
    # "ring" / "rows": void_sddmm_rows_f32 (tiles of a block-row share their
    # grad_c rows; the fourth shape has rows of up to 128 tiles, i.e. many
    # groups per row), on its LDS-DMA ring where the operands allow (N a
    # multiple of 4: chunks of 32 columns, the last one cut by N in several
    # shapes) or forced onto the register-staged kernel.  None /
    # "tile_rows": void_sddmm_f32 (tiles in the given order, 8 to a
    # workgroup on the per-tile ring with 16-column chunks, or one per
    # workgroup on the register-staged kernel).
    from void_amd.format import build_bsr_layout
    if grouped in ("rows", "tile_rows"):
        monkeypatch.setenv("VOID_AMD_SDDMM", "rows")
    elif grouped == "ring":  # the row-grouped ring even where the per-tile kernel would be chosen
        monkeypatch.setenv("VOID_AMD_SDDMM", "grouped")
    if grouped == "tile_rows":
        grouped = None
    rng = np.random.default_rng(seed)
    nbr, nbc = -(-M // 32), -(-K // 32)
    flat = rng.choice(nbr * nbc, min(n, nbr * nbc), replace=False)
    rows, cols = (flat // nbc).astype(np.int32), (flat % nbc).astype(np.int32)
    G = rng.standard_normal((M, N)).astype(np.float32)
    B = rng.standard_normal((K, N)).astype(np.float32)
    tr, tc = torch.from_numpy(rows).to(gpu), torch.from_numpy(cols).to(gpu)
    lay = build_bsr_layout(tr, tc, nbr, nbc, gpu) if grouped else None
    got = _runtime.sddmm_tiles(torch.from_numpy(G).to(gpu), torch.from_numpy(B).to(gpu), tr, tc, (M, K),
                               torch.float32, layout=lay)
    Gp = np.zeros((nbr * 32, N)); Gp[:M] = G
    Bp = np.zeros((nbc * 32, N)); Bp[:K] = B
    for t in range(len(rows)):
        x = Gp[rows[t] * 32:(rows[t] + 1) * 32]
        y = Bp[cols[t] * 32:(cols[t] + 1) * 32]
        ref = x @ y.T
        bound = N * U * (np.abs(x) @ np.abs(y).T)
        assert np.all(np.abs(got[t].cpu().numpy() - ref) <= bound + 1e-30), t



# One rounding of the output type on top of the fp32 bound (p significand
# bits: 8 for bf16, 11 for fp16, plus half of fp16's subnormal spacing).
_HALF = {torch.bfloat16: (2.0 ** -8, 0.0), torch.float16: (2.0 ** -11, 2.0 ** -25)}


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("grouped", [None, "tile_rows", "ring", "rows"])
def test_sddmm_tiles_half_outputs(gpu, out_dtype, grouped, monkeypatch):
    """The gradient tiles of a half-precision VOIDTensor come out in its
    dtype (autograd.py passes a_values.dtype): each kernel's bf16 and fp16
    stores."""
    from void_amd.format import build_bsr_layout
    if grouped in ("rows", "tile_rows"):
        monkeypatch.setenv("VOID_AMD_SDDMM", "rows")
    elif grouped == "ring":  # the row-grouped ring even where the per-tile kernel would be chosen
        monkeypatch.setenv("VOID_AMD_SDDMM", "grouped")
    if grouped == "tile_rows":
        grouped = None
    M, K, N = 640, 1024, 200
    rng = np.random.default_rng(7)
    nbr, nbc = M // 32, K // 32
    flat = rng.choice(nbr * nbc, 150, replace=False)
    rows, cols = (flat // nbc).astype(np.int32), (flat % nbc).astype(np.int32)
    G = rng.standard_normal((M, N)).astype(np.float32)
    B = rng.standard_normal((K, N)).astype(np.float32)
    tr, tc = torch.from_numpy(rows).to(gpu), torch.from_numpy(cols).to(gpu)
    lay = build_bsr_layout(tr, tc, nbr, nbc, gpu) if grouped else None
    got = _runtime.sddmm_tiles(torch.from_numpy(G).to(gpu), torch.from_numpy(B).to(gpu), tr, tc, (M, K),
                               out_dtype, layout=lay)
    assert got.dtype == out_dtype
    rel, ab = _HALF[out_dtype]
    G64, B64 = G.astype(np.float64), B.astype(np.float64)
    for t in range(len(rows)):
        x, y = G64[rows[t] * 32:(rows[t] + 1) * 32], B64[cols[t] * 32:(cols[t] + 1) * 32]
        ref = x @ y.T
        bound = N * U * (np.abs(x) @ np.abs(y).T) * (1 + rel) + rel * np.abs(ref) + ab
        assert np.all(np.abs(got[t].float().cpu().numpy() - ref) <= bound + 1e-30), t

@pytest.mark.parametrize("in_dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("same_out", [True, False], ids=["out16", "out32"])
@pytest.mark.parametrize("M,K,N,n,seed", [(1024, 2048, 512, 600, 0), (100, 70, 40, 6, 1), (64, 96, 136, 5, 2),
                                          (256, 4096, 72, 300, 3), (96, 128, 1000, 12, 4), (500, 300, 8, 30, 6),
                                          (70, 1000, 20, 40, 5)])
def test_sddmm16(gpu, in_dtype, same_out, M, K, N, n, seed):
    """16-bit grad_c and B of one dtype (the backward of a bf16 / fp16 VOID
    tensor): void_sddmm_rows_bf16 / _f16 on the 16-bit MFMA when N % 8 == 0
    (64-column chunks, the last cut by N), the fp32 kernel on widened copies
    otherwise (N = 20).  Same bound on the 16-bit values as the fp32 path,
    plus one rounding of a 16-bit output."""
    from void_amd.format import build_bsr_layout
    rng = np.random.default_rng(100 + seed)
    nbr, nbc = -(-M // 32), -(-K // 32)
    flat = rng.choice(nbr * nbc, min(n, nbr * nbc), replace=False)
    rows, cols = (flat // nbc).astype(np.int32), (flat % nbc).astype(np.int32)
    G = torch.from_numpy(rng.standard_normal((M, N)).astype(np.float32)).to(in_dtype)
    B = torch.from_numpy(rng.standard_normal((K, N)).astype(np.float32)).to(in_dtype)
    tr, tc = torch.from_numpy(rows).to(gpu), torch.from_numpy(cols).to(gpu)
    lay = build_bsr_layout(tr, tc, nbr, nbc, gpu)
    out_dtype = in_dtype if same_out else torch.float32
    got = _runtime.sddmm_tiles(G.to(gpu), B.to(gpu), tr, tc, (M, K), out_dtype, layout=lay)
    assert got.dtype == out_dtype
    rel, ab = _HALF[out_dtype] if same_out else (0.0, 0.0)
    Gp = np.zeros((nbr * 32, N)); Gp[:M] = G.double().numpy()
    Bp = np.zeros((nbc * 32, N)); Bp[:K] = B.double().numpy()
    for t in range(len(rows)):
        x, y = Gp[rows[t] * 32:(rows[t] + 1) * 32], Bp[cols[t] * 32:(cols[t] + 1) * 32]
        ref = x @ y.T
        bound = N * U * (np.abs(x) @ np.abs(y).T) * (1 + rel) + rel * np.abs(ref) + ab
        assert np.all(np.abs(got[t].float().cpu().numpy() - ref) <= bound + 1e-30), t


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
def test_voidspmm_gradients_16bit(gpu, dtype):
    """A bf16 / fp16 VOID tensor times an input of the same dtype: forward
    and the product for the input's gradient on the 16-bit SpMM, the tiles'
    gradient on the 16-bit SDDMM, each within the fp32 summation bound on the
    16-bit values plus one rounding of the 16-bit result."""
    case = cases.uniform_blocks(512, 1024, 96, 150, seed=5)
    vt = cases.make_void_tensor(case, "cpu").to_dtype(dtype).to(gpu)
    mod = void_amd.VOIDSpMM(vt).to(gpu)
    x = torch.randn(1024, 96, device=gpu).to(dtype).requires_grad_(True)
    w = torch.randn(512, 96, device=gpu).to(dtype)
    y = mod(x)
    assert y.dtype == dtype
    (y * w).sum().backward()
    rel, ab = _HALF[dtype]
    A = oracle.densify(vt.values.float().cpu().numpy(), case.block_rows, case.block_cols, (512, 1024)).astype(np.float64)
    X, W = x.detach().double().cpu().numpy(), w.double().cpu().numpy()
    n_row = np.bincount(case.block_rows, minlength=16).max()
    ref = A @ X
    assert np.all(np.abs(y.detach().double().cpu().numpy() - ref) <=
                  32 * n_row * U * (np.abs(A) @ np.abs(X)) + rel * np.abs(ref) + ab + 1e-30)
    gX = A.T @ W
    n_col = np.bincount(case.block_cols, minlength=32).max()
    assert np.all(np.abs(x.grad.double().cpu().numpy() - gX) <=
                  32 * n_col * U * (np.abs(A).T @ np.abs(W)) + rel * np.abs(gX) + ab + 1e-30)
    gA = W @ X.T
    tiles = mod.values.grad.double().cpu().numpy()
    bound_full = 96 * U * (np.abs(W) @ np.abs(X).T)
    rr, cc = vt.block_rows.cpu().numpy(), vt.block_cols.cpu().numpy()
    for t in range(len(tiles)):
        r, c = rr[t] * 32, cc[t] * 32
        g = gA[r:r + 32, c:c + 32]
        assert np.all(np.abs(tiles[t] - g) <= bound_full[r:r + 32, c:c + 32] + rel * np.abs(g) + ab + 1e-30)


def test_voidspmm_gradients(gpu):
    case = cases.uniform_blocks(512, 1024, 96, 150, seed=5)
    vt = cases.make_void_tensor(case, "cpu").to(gpu)
    mod = void_amd.VOIDSpMM(vt).to(gpu)
    x = torch.randn(1024, 96, device=gpu, requires_grad=True)
    w = torch.randn(512, 96, device=gpu)
    y = mod(x)
    (y * w).sum().backward()
    A = oracle.densify(case.tiles, case.block_rows, case.block_cols, (512, 1024)).astype(np.float64)
    X, W = x.detach().cpu().double().numpy(), w.cpu().double().numpy()
    assert np.all(np.abs(y.detach().cpu().numpy() - A @ X) <= 32 * 10 * U * (np.abs(A) @ np.abs(X)) + 1e-30)
    gX = A.T @ W  # dL/dB = A^T dL/dC
    n_col = np.bincount(case.block_cols, minlength=32).max()
    assert np.all(np.abs(x.grad.cpu().numpy() - gX) <= 32 * n_col * U * (np.abs(A).T @ np.abs(W)) + 1e-30)
    gA = W @ X.T  # dense dL/dA; only the tiles' entries are returned
    tiles = mod.values.grad.cpu().numpy()
    vals_rows, vals_cols = vt.block_rows.cpu().numpy(), vt.block_cols.cpu().numpy()
    bound_full = 96 * U * (np.abs(W) @ np.abs(X).T)
    for t in range(len(tiles)):
        r, c = vals_rows[t] * 32, vals_cols[t] * 32
        assert np.all(np.abs(tiles[t] - gA[r:r + 32, c:c + 32]) <= bound_full[r:r + 32, c:c + 32] + 1e-30)


def test_sparse_linear_training_step(gpu):
    case = cases.uniform_blocks(128, 256, 8, 12, seed=9)
    vt = cases.make_void_tensor(case, "cpu").to(gpu)
    layer = void_amd.SparseLinear(256, 128, vt).to(gpu)
    x = torch.randn(4, 5, 256, device=gpu)
    y = layer(x)
    assert y.shape == (4, 5, 128)
    loss = (y ** 2).mean()
    loss.backward()
    assert layer.sparse_weight.values.grad.shape == vt.values.shape and layer.bias.grad.shape == (128,)
    # an optimiser step changes the values in place; the next forward must see them
    with torch.no_grad():
        layer.sparse_weight.values.mul_(2.0)
        layer.bias.zero_()
    y2 = layer(x)
    W = oracle.densify(vt.values.cpu().numpy() * 2.0, case.block_rows, case.block_cols, (128, 256))
    ref = x.reshape(-1, 256).cpu().double().numpy() @ W.T.astype(np.float64)
    assert np.allclose(y2.detach().reshape(-1, 128).cpu().numpy(), ref, rtol=1e-5, atol=1e-4)



def test_inference_mode(gpu):
    """Tensors made under torch.inference_mode keep no version counter; the
    cached layouts then key on identity alone, and every entry point runs as
    outside that mode."""
    case = cases.uniform_blocks(256, 512, 64, 40, seed=8)
    x_host = torch.randn(512, 64)
    vt_ref = cases.make_void_tensor(case, "cpu").to(gpu)
    y_ref = void_amd.VOIDSpMM(vt_ref).to(gpu)(x_host.to(gpu)).detach()
    q_ref = void_amd.quantize_void_tensor(cases.make_void_tensor(case, "cpu")).to(gpu)
    bq, bs = oracle.quantize_i8_columns(case.b)
    z_ref = void_amd.void_spmm_int8(q_ref, torch.from_numpy(bq).to(gpu), b_scale=torch.from_numpy(bs).to(gpu))
    with torch.inference_mode():
        vt = cases.make_void_tensor(case, "cpu").to(gpu)
        mod = void_amd.VOIDSpMM(vt).to(gpu)
        x = x_host.to(gpu)
        assert torch.equal(mod(x), y_ref)
        assert torch.equal(void_amd.void_spmm(vt, x), y_ref)
        q = void_amd.quantize_void_tensor(cases.make_void_tensor(case, "cpu")).to(gpu)
        z = void_amd.void_spmm_int8(q, torch.from_numpy(bq).to(gpu), b_scale=torch.from_numpy(bs).to(gpu))
        assert torch.equal(z, z_ref)


def test_layout_plans_shared_and_streams(gpu):
    """One structure's plans serve every step, also from a second stream, with
    bit-identical results; capture is refused as before."""
    case = cases.uniform_blocks(256, 4096, 96, 700, seed=5)  # rows beyond 64 tiles: split plans
    vt = cases.make_void_tensor(case, "cpu").to(gpu)
    mod = void_amd.VOIDSpMM(vt)
    b = torch.from_numpy(case.b).to(gpu)

    def step():
        x = b.clone().requires_grad_()
        mod.zero_grad(set_to_none=True)
        y = mod(x)
        y.backward(torch.ones_like(y))
        return [y.detach().clone(), x.grad.clone(), mod.values.grad.clone()]

    ref = step()
    lay = autograd._layout(mod.block_rows, mod.block_cols, mod.shape)
    plan = lay.plans[64]
    assert plan.n_split_tiles > 0
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = step()
    torch.cuda.current_stream().wait_stream(side)
    for other in (got, step()):
        assert all(torch.equal(p, q) for p, q in zip(ref, other))
    assert lay.plans[64] is plan and len(plan.workspaces) == 2 and not plan.capture_spares
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with pytest.raises(RuntimeError, match="captured"):
        with torch.cuda.graph(g):
            mod(b)
    assert torch.equal(mod(b).detach(), ref[0])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n", [1, 3, 33, 1000])
def test_gather_tiles_transposed(gpu, dtype, n):
    v = torch.randn(n, 32, 32, device=gpu).to(dtype)
    order = torch.randperm(n, device=gpu)
    got = _runtime.gather_tiles_t(v, order).view(dtype).view(n, 32, 32)
    assert torch.equal(got, v[order].transpose(1, 2))
    shifted = torch.cat([v.reshape(-1)[:1], v.reshape(-1)])[1:].view(n, 32, 32)  # not 16-byte aligned
    assert torch.equal(_runtime.gather_tiles_t(shifted, order).view(dtype).view(n, 32, 32), got)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("tokens", [1, 7, 33, 260])
@pytest.mark.parametrize("token_major_grad", [True, False])
def test_linear_bias_fused_step(gpu, monkeypatch, dtype, tokens, token_major_grad):
    """SparseLinear on token-major input: output, gradients of input, tiles and
    bias against float64, with either layout of the incoming gradient; a
    forward hook on the weight module takes the unfused path to the same bits
    (the bias's gradient, summed in another order, within its bound)."""
    monkeypatch.setattr(_runtime, "TRANSPOSE_MIN_NUMEL", 1)
    monkeypatch.setattr(autograd, "BIAS_EPILOGUE_BYTES", {2: 0, 4: 0})
    case = cases.uniform_blocks(130, 200, tokens, 20, seed=tokens)
    vt = cases.make_void_tensor(case, "cpu").to(gpu).to_dtype(dtype)
    lin = void_amd.SparseLinear(200, 130, vt).to(gpu)
    g = torch.Generator(device=gpu).manual_seed(tokens)
    with torch.no_grad():
        lin.bias.copy_(torch.randn(130, generator=g, device=gpu))
    x = torch.randn(tokens, 200, generator=g, device=gpu).to(dtype).requires_grad_()
    gy = torch.randn(tokens, 130, generator=g, device=gpu).to(dtype)
    if not token_major_grad:
        gy = gy.t().contiguous().t()

    def step():
        lin.zero_grad(set_to_none=True)
        x.grad = None
        y = lin(x)
        y.backward(gy)
        return [y.detach(), x.grad, lin.sparse_weight.values.grad, lin.bias.grad]

    fused = step()
    assert fused[1].is_contiguous()
    handle = lin.sparse_weight.register_forward_hook(lambda m, i, o: None)
    plain = step()
    handle.remove()
    W = torch.zeros(160, 224, dtype=torch.float64, device=gpu)
    for t, (r, c) in enumerate(zip(case.block_rows, case.block_cols)):
        W[32 * r:32 * r + 32, 32 * c:32 * c + 32] = vt.values[t].double()
    gp = torch.zeros(tokens, 160, dtype=torch.float64, device=gpu)
    xp = torch.zeros(tokens, 224, dtype=torch.float64, device=gpu)
    gp[:, :130], xp[:, :200] = gy.double(), x.detach().double()
    gw = gp.t() @ xp
    gwa = gp.abs().t() @ xp.abs()
    pick = lambda m: torch.stack([m[32 * r:32 * r + 32, 32 * c:32 * c + 32]
                                  for r, c in zip(case.block_rows, case.block_cols)])
    b64 = lin.bias.detach().double()
    refs = [(xp @ W.t())[:, :130] + b64, (gp @ W)[:, :200], pick(gw), gp[:, :130].sum(0)]
    mags = [(xp.abs() @ W.abs().t())[:, :130] + b64.abs(), (gp.abs() @ W.abs())[:, :200], pick(gwa),
            gp[:, :130].abs().sum(0)]
    rnd = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8}[dtype]
    for k, (out, alt, ref, mag) in enumerate(zip(fused, plain, refs, mags)):
        # The output rounds twice: the product, at most mag, and the sum.
        tol = 300 * U * mag + rnd * ref.abs() + (rnd * mag if k == 0 else 0) + 1e-30
        assert bool(((out.double() - ref).abs() <= tol).all()), k
        assert bool(((alt.double() - ref).abs() <= tol).all()), k
        if k < 3:
            assert torch.equal(out, alt), k


def _linear(gpu, dtype, tokens, seed=3):
    case = cases.uniform_blocks(130, 200, tokens, 20, seed=seed)
    lin = void_amd.SparseLinear(200, 130, cases.make_void_tensor(case, "cpu").to(gpu).to_dtype(dtype)).to(gpu)
    g = torch.Generator(device=gpu).manual_seed(seed)
    with torch.no_grad():
        lin.bias.copy_(torch.randn(130, generator=g, device=gpu))
    return lin, torch.randn(tokens, 200, generator=g, device=gpu).to(dtype)


@pytest.mark.parametrize("kernel", ["", "cgd", "f32"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tokens", [1, 37, 64])
def test_linear_bias_is_an_addition(gpu, monkeypatch, dtype, tokens, kernel):
    """y = w(x) + b to the bit: the product is rounded to x's type, then the sum."""
    monkeypatch.setattr(autograd, "BIAS_EPILOGUE_BYTES", {2: 0, 4: 0})
    if kernel:
        monkeypatch.setenv("VOID_AMD_KERNEL", kernel)
    lin, x = _linear(gpu, dtype, tokens)
    with torch.no_grad():
        assert lin._bias_in_epilogue(x)
        assert torch.equal(lin(x), lin.sparse_weight(x.T).T + lin.bias)


def test_linear_bias_keeps_autograd(gpu, monkeypatch):
    """The bias alone: batched gradients, no SpMM in its backward, forward-mode
    tangents; and a frozen bias or weight."""
    import torch.autograd.forward_ad as fwd
    monkeypatch.setattr(autograd, "BIAS_EPILOGUE_BYTES", {2: 0, 4: 0})
    lin, x = _linear(gpu, torch.float32, 12)
    gy = torch.randn(4, 12, 130, device=gpu)
    y = lin(x)
    calls = []
    with monkeypatch.context() as m:
        m.setattr(autograd, "float_spmm", lambda *a, **k: calls.append(a))
        m.setattr(_runtime, "sddmm_tiles", lambda *a, **k: calls.append(a))
        (one,) = torch.autograd.grad(y, lin.bias, gy[0], retain_graph=True)
        (many,) = torch.autograd.grad(y, lin.bias, gy, is_grads_batched=True)
    assert not calls
    for got, ref in ((one, gy[0].double().sum(0)), (many, gy.double().sum(1))):
        assert got.shape == ref.shape and bool(((got.double() - ref).abs() <= 12 * U * gy.abs().sum(1).max()).all())
    with fwd.dual_level():
        bias = lin.bias
        del lin.bias
        tangent = torch.randn(130, device=gpu)
        lin.bias = fwd.make_dual(bias.detach(), tangent)
        with torch.no_grad():
            lin.sparse_weight.values.requires_grad_(False)
        assert torch.equal(fwd.unpack_dual(lin(x)).tangent, tangent.expand(12, 130))
    lin.bias = bias
    out = lin(x)  # only the bias trains
    out.backward(gy[0])
    assert torch.equal(lin.bias.grad, one) and lin.sparse_weight.values.grad is None
    lin.bias.requires_grad_(False)
    lin.bias.grad = None
    lin.sparse_weight.values.requires_grad_(True)
    lin(x).backward(gy[0])
    assert lin.bias.grad is None and lin.sparse_weight.values.grad is not None


def test_linear_create_graph_bias(gpu, monkeypatch):
    """With create_graph the bias gradient stays differentiable in the output gradient."""
    monkeypatch.setattr(autograd, "BIAS_EPILOGUE_BYTES", {2: 0, 4: 0})
    case = cases.uniform_blocks(64, 64, 5, 3, seed=2)
    lin = void_amd.SparseLinear(64, 64, cases.make_void_tensor(case, "cpu").to(gpu)).to(gpu)
    x = torch.randn(5, 64, device=gpu)
    gy = torch.randn(5, 64, device=gpu, requires_grad=True)
    (gb,) = torch.autograd.grad(lin(x), lin.bias, gy, create_graph=True)
    (gg,) = torch.autograd.grad(gb.sum(), gy)
    assert torch.equal(gg, torch.ones_like(gy))


@pytest.mark.parametrize("bad", [float("inf"), float("nan"), 1e38])
@pytest.mark.parametrize("grouped", ["tiles", "grouped"])
def test_sddmm_non_finite_follow_fp32(gpu, monkeypatch, bad, grouped):
    """A tile whose sums are not finite equals the fp32 MFMA's (the
    register-staged kernel's); the others stay within the fp32 bound."""
    from void_amd.format import build_bsr_layout
    case = cases.uniform_blocks(130, 200, 100, 20, seed=4)
    g = torch.randn(130, 100, device=gpu)
    b = torch.from_numpy(case.b).to(gpu)
    g[40, 7] = bad
    if bad == 1e38:
        g[40, 8] = -bad
        b *= 100
    rows, cols = torch.from_numpy(case.block_rows).to(gpu), torch.from_numpy(case.block_cols).to(gpu)
    lay = build_bsr_layout(rows, cols, 5, 7, gpu)
    out = {}
    for mode in (grouped, "rows"):
        monkeypatch.setenv("VOID_AMD_SDDMM", mode)
        out[mode] = _runtime.sddmm_tiles(g, b, rows, cols, (130, 200), torch.float32, layout=lay)
    a, r = out[grouped], out["rows"]
    assert not bool(torch.isfinite(r).all())
    assert torch.equal(torch.isnan(a), torch.isnan(r)) and torch.equal(torch.isinf(a), torch.isinf(r))
    ok = torch.isfinite(r).all(dim=2).all(dim=1)
    assert bool(ok.any()) and bool(((a - r)[ok].abs() <= 1e-5 * r[ok].abs().max()).all())


def test_layout_cache_eviction(gpu):
    """More structures than the cache holds, used on two streams in turn."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    for i in range(70):
        case = cases.uniform_blocks(64, 96, 40, 1 + i % 5, seed=i)
        vt = cases.make_void_tensor(case, "cpu").to(gpu)
        lin = void_amd.SparseLinear(96, 64, vt).to(gpu)
        x = torch.ones(40, 96, device=gpu)
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side if i % 2 else torch.cuda.current_stream()):
            y = lin(x)
        torch.cuda.current_stream().wait_stream(side)
        ref = vt.values.double().sum(2).new_zeros(64)
        for t, r in enumerate(case.block_rows):
            ref[32 * r:32 * r + 32] += vt.values[t].double().sum(1)
        assert bool(((y.double() - ref).abs() <= 1e-4).all()), i


@pytest.mark.parametrize("least", [0, 1 << 60])
def test_linear_output_in_place_and_shapes(gpu, monkeypatch, least):
    """The output takes in-place operations and 3-D and empty inputs as before,
    with the bias in the epilogue and as an addition."""
    monkeypatch.setattr(autograd, "BIAS_EPILOGUE_BYTES", {4: least})
    case = cases.uniform_blocks(64, 96, 40, 4, seed=9)
    lin = void_amd.SparseLinear(96, 64, cases.make_void_tensor(case, "cpu").to(gpu)).to(gpu)
    x = torch.randn(2, 5, 96, device=gpu, requires_grad=True)
    y = lin(x)
    assert y.shape == (2, 5, 64)
    z = lin(x).relu_()
    z.sum().backward()
    got = x.grad.clone()
    x.grad = None
    torch.relu(lin(x)).sum().backward()
    assert torch.equal(z.detach(), torch.relu(y).detach()) and torch.equal(got, x.grad)
    e = torch.randn(0, 96, device=gpu, requires_grad=True)
    out = lin(e)
    out.sum().backward()
    assert out.shape == (0, 64) and e.grad.shape == (0, 96)


@pytest.mark.parametrize("grouped", ["tiles", "grouped", "rows"])
@pytest.mark.parametrize("terms", [1, 2, 64])
@pytest.mark.parametrize("kind", ["normal", "constant", "tiny", "tinier"])
def test_sddmm_precision(gpu, monkeypatch, kind, terms, grouped):
    """fp32 products keep all 24 bits: one rounding for one term, n for n, also
    for operands far below one (still normal numbers) and for equal operands,
    whose errors would all have one sign."""
    from void_amd.format import build_bsr_layout
    monkeypatch.setenv("VOID_AMD_SDDMM", grouped)
    rng = np.random.default_rng(terms)
    N = max(terms, 4)
    case = cases.uniform_blocks(128, 192, N, 16, seed=4)
    G, B = rng.standard_normal((128, N)), rng.standard_normal((192, N))
    if kind == "constant":
        G[:], B[:] = (1 + 2.0 ** -7 - 2.0 ** -16,) * 2
    elif kind != "normal":
        G *= 2.0 ** (-118 if kind == "tiny" else -122)
        B *= 2.0 ** 100
    G, B = G.astype(np.float32), B.astype(np.float32)
    G[:, terms:] = 0
    rows, cols = torch.from_numpy(case.block_rows).to(gpu), torch.from_numpy(case.block_cols).to(gpu)
    lay = build_bsr_layout(rows, cols, 4, 6, gpu)
    got = _runtime.sddmm_tiles(torch.from_numpy(G).to(gpu), torch.from_numpy(B).to(gpu), rows, cols, (128, 192),
                               torch.float32, layout=lay).double().cpu().numpy()
    for t, (r, c) in enumerate(zip(case.block_rows, case.block_cols)):
        x, y = G[32 * r:32 * r + 32].astype(np.float64), B[32 * c:32 * c + 32].astype(np.float64)
        assert np.all(np.abs(got[t] - x @ y.T) <= terms * U * (np.abs(x) @ np.abs(y).T)), t


def test_layout_cache_threads_and_streams(gpu):
    """Two threads on streams of their own, each with more structures than the
    cache holds: dropped layouts' memory is recorded on both streams, and every
    result is right.  Outputs are checked at the end, without waits between."""
    import threading
    done, errors = [], []

    def work(k):
        try:
            stream = torch.cuda.Stream()
            with torch.cuda.stream(stream):
                for i in range(90):
                    case = cases.uniform_blocks(96, 160, 24, 3 + (i + k) % 9, seed=1000 * k + i)
                    vt = cases.make_void_tensor(case, "cpu").to(gpu)
                    lin = void_amd.SparseLinear(160, 96, vt).to(gpu)
                    x = torch.randn(24, 160, device=gpu, requires_grad=True)
                    gy = torch.randn(24, 96, device=gpu)
                    y = lin(x)
                    y.backward(gy)
                    done.append((case, vt, x, gy, y.detach(), x.grad))
                    assert stream.cuda_stream in autograd._layout(
                        lin.sparse_weight.block_rows, lin.sparse_weight.block_cols, lin.sparse_weight.shape).streams
            stream.synchronize()
        except Exception as e:  # reported by the main thread
            errors.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    torch.cuda.synchronize()
    assert len(done) == 180
    for case, vt, x, gy, y, gx in done:
        W = torch.zeros(96, 160, dtype=torch.float64, device=gpu)
        for t, (r, c) in enumerate(zip(case.block_rows, case.block_cols)):
            W[32 * r:32 * r + 32, 32 * c:32 * c + 32] = vt.values[t].double()
        for got, l, m in ((y, x.detach().double(), W.t()), (gx, gy.double(), W)):
            assert bool(((got.double() - l @ m).abs() <= 160 * U * (l.abs() @ m.abs()) + 1e-30).all())


def test_many_layers_plan_once(gpu, monkeypatch):
    """Two steps of more layers than the list of recent structures is long: the
    second orders, plans and uploads nothing."""
    layers = []
    for i in range(autograd.MAX_RECENT + 16):
        case = cases.uniform_blocks(96, 96, 8, 4, seed=i)
        layers.append(void_amd.SparseLinear(96, 96, cases.make_void_tensor(case, "cpu").to(gpu)).to(gpu))
    x = torch.randn(8, 96, device=gpu, requires_grad=True)
    calls = []

    def step():
        y = x
        for lin in layers:
            y = lin(y) + y
        y.sum().backward()

    step()
    for mod, name in ((autograd, "build_bsr_layout"), (_runtime, "build_bsr_layout"), (_runtime, "plan_rows")):
        fn = getattr(mod, name)
        monkeypatch.setattr(mod, name, lambda *a, fn=fn, name=name, **k: calls.append(name) or fn(*a, **k))
    step()
    assert not calls


def test_split_layers_share_one_workspace(gpu):
    """Layers whose plans split rows, of several sizes and widths in turn on one
    stream: one buffer in all, and every step repeats the first one's bits."""
    rng = np.random.default_rng(0)
    layers = []
    for i, (M, K) in enumerate([(96, 4096), (4096, 64), (160, 6000), (64, 8192)]):
        case = cases.uniform_blocks(M, K, 8, (M // 32) * (K // 32) * 3 // 4, seed=i)
        layers.append(void_amd.SparseLinear(K, M, cases.make_void_tensor(case, "cpu").to(gpu)).to(gpu))
    ins = [(lin, torch.from_numpy(rng.standard_normal((n, lin.in_features)).astype(np.float32)).to(gpu))
           for n in (40, 300, 7) for lin in layers]

    def step():
        out = []
        for lin, x in ins:
            x = x.clone().requires_grad_()
            y = lin(x)
            y.backward(torch.ones_like(y))
            out += [y.detach(), x.grad]
        return out

    _runtime.STEP_WORKSPACES.buffers.clear()
    ref = step()
    held = _runtime.STEP_WORKSPACES.buffers
    assert len(held) == 1
    for _ in range(3):
        assert all(torch.equal(p, q) for p, q in zip(ref, step()))
    assert len(held) == 1 and sum(b.numel() for b, _ in held.values()) <= _runtime.MAX_SPARE_WORKSPACE
    for (lin, x), y in zip(ins, ref[::2]):
        w = lin.sparse_weight
        W = torch.zeros(-(-lin.out_features // 32) * 32, -(-lin.in_features // 32) * 32, dtype=torch.float64, device=gpu)
        for t, (r, c) in enumerate(zip(w.block_rows.tolist(), w.block_cols.tolist())):
            W[32 * r:32 * r + 32, 32 * c:32 * c + 32] = w.values[t].detach().double()
        W = W[:lin.out_features, :lin.in_features]
        mag = x.double().abs() @ W.abs().t()
        assert bool(((y.double() - x.double() @ W.t()).abs() <= lin.in_features * U * mag + 1e-30).all())
