"""An 8-bit B of any width on the column-group kernels: aligned copies of
unaligned rows, padded quantisation of a float B, and rows whose last 16-byte
chunk is cut off by N."""

import numpy as np
import pytest
import torch

import cases
import oracle
import void_amd
from void_amd import _runtime, tuning

pytestmark = pytest.mark.gpu

WIDTHS = [1, 15, 17, 63, 65, 127, 129, 250, 513]


@pytest.fixture
def gpu():
    return torch.device("cuda:0")


@pytest.mark.parametrize("shape", [(1, 1), (3, 16), (70, 17), (33, 65), (129, 250), (64, 513)])
@pytest.mark.parametrize("shift", [0, 1, 7])
def test_aligned_copy_bytes(gpu, shape, shift):
    K, N = shape
    flat = torch.randint(-128, 128, (K * (N + 3) + shift,), dtype=torch.int8, device=gpu)
    b = flat[shift:].view(K, N + 3)[:, :N]
    out = _runtime.aligned_copy_b8(b, b.stride(0))
    assert out.stride(0) == tuning.aligned_pitch(N) and out.data_ptr() % 16 == 0
    assert torch.equal(out, b)


@pytest.mark.parametrize("N", WIDTHS)
def test_padded_quantisation_matches_flat(gpu, N):
    from void_amd.int_quant import IntFormat, IntQuantConfig, ScaleMode, _quantize_b_per_tensor, quantize_tensor
    b = torch.randn(77, N, generator=torch.Generator().manual_seed(N))
    cfg = IntQuantConfig(format=IntFormat.INT8, symmetric=True, scale_mode=ScaleMode.PER_TENSOR)
    ref, params = quantize_tensor(b, cfg)
    q, scale = _quantize_b_per_tensor(b.to(gpu))
    assert q.stride(0) % 16 == 0 and torch.equal(q.cpu(), ref)
    assert torch.equal(scale.cpu(), params.scale.reshape(1))


@pytest.mark.parametrize("kernel", ["default", "cg", "cgd", "cgd3", "cgdk", "bsr"])
@pytest.mark.parametrize("pad", ["0", "1", "pitch", "shift"])
@pytest.mark.parametrize("N", WIDTHS)
def test_int8_any_width(gpu, monkeypatch, kernel, pad, N):
    """Accumulators bit-exact for every kernel; columns past N hold other data."""
    if kernel != "default":
        monkeypatch.setenv("VOID_AMD_KERNEL", kernel)
    monkeypatch.setenv("VOID_AMD_PAD", "0" if pad == "0" else "1")
    case = cases.uniform_blocks(170, 203, N, 25, seed=N)
    q = void_amd.quantize_void_tensor(cases.make_void_tensor(case, "cpu"))
    rng = np.random.default_rng(N)
    bq = rng.integers(-128, 128, (203, N), dtype=np.int8)
    pitch, shift = (N + 31) // 16 * 16 if pad == "pitch" else N, 5 if pad == "shift" else 0
    flat = torch.full((203 * pitch + shift,), 99, dtype=torch.int8)
    b = flat[shift:].view(203, pitch)[:, :N]
    b.copy_(torch.from_numpy(bq))
    b = flat.to(gpu)[shift:].view(203, pitch)[:, :N]
    A = oracle.Bsr(q.values.numpy(), q.scales.numpy(), case.block_rows, case.block_cols, (170, 203))
    qd = q.to(gpu)
    got = void_amd.void_spmm_int8(qd, b, epilogue="raw_i32").cpu().numpy()
    assert np.array_equal(got, oracle.i8_acc(A, bq))
    # A misaligned output view as well.
    wide = torch.full((170, N + 3), -7, dtype=torch.int32, device=gpu)
    void_amd.void_spmm_int8(qd, b, epilogue="raw_i32", out=wide[:, 1:N + 1])
    assert np.array_equal(wide[:, 1:N + 1].cpu().numpy(), got)
    assert bool((wide[:, 0] == -7).all()) and bool((wide[:, N + 1:] == -7).all())


@pytest.mark.parametrize("N", WIDTHS)
def test_float_b_scale_stays_single(gpu, N):
    """Row-mean with the device scale of a float B, bit for bit the oracle's."""
    case = cases.uniform_blocks(170, 203, N, 25, seed=N + 1)
    q = void_amd.quantize_void_tensor(cases.make_void_tensor(case, "cpu"))
    bq, bs = oracle.quantize_i8_tensor(case.b)
    A = oracle.Bsr(q.values.numpy(), q.scales.numpy(), case.block_rows, case.block_cols, (170, 203))
    ref = oracle.row_mean(A, oracle.i8_acc(A, bq), bs)
    got = void_amd.void_spmm_int8(q.to(gpu), torch.from_numpy(case.b).to(gpu)).cpu().numpy()
    assert np.array_equal(got.view(np.int32), ref.view(np.int32))


@pytest.mark.parametrize("N", [17, 250])
def test_fp8_nan_codes_past_n(gpu, N):
    """Chunks cut off by N may hold NaN codes in the next columns: never stored, never mixed in."""
    case = cases.uniform_blocks(96, 200, N, 14, seed=N)
    f8 = void_amd.void_tensor_to_fp8(cases.make_void_tensor(case, "cpu"))
    pitch = (N + 31) // 16 * 16
    raw = torch.full((200, pitch), 0x7f, dtype=torch.uint8)
    codes = torch.from_numpy(case.b).clamp(-400, 400).to(torch.float8_e4m3fn)
    raw[:, :N] = codes.view(torch.uint8)
    b = raw.to(gpu).view(torch.float8_e4m3fn)[:, :N]
    out = void_amd.void_spmm_fp8(f8.to(gpu), b, output_dtype=torch.float32).double().cpu()
    dense = torch.zeros(96, 224, dtype=torch.float64)
    mag = torch.zeros(96, 224, dtype=torch.float64)
    t = f8.values_fp8.double() * f8.scaling_info.scale.double()[:, None, None]
    for i, (r, c) in enumerate(zip(case.block_rows, case.block_cols)):
        dense[32 * r:32 * r + 32, 32 * c:32 * c + 32] = t[i]
    mag = dense.abs()
    bd = codes.double()
    ref, bound = dense[:, :200] @ bd, mag[:, :200] @ bd.abs()
    assert bool(((out - ref).abs() <= 2.0 ** -13 * bound + 1e-30).all())


def _layouts(bq, gpu):
    """B as row- and column-major views: aligned, padded, and shifted by a byte."""
    K, N = bq.shape
    src = torch.from_numpy(bq)
    for col in (False, True):
        rows, cols = (N, K) if col else (K, N)
        for pitch, shift in ((cols, 0), ((cols + 31) // 16 * 16, 0), (cols + 1, 1)):
            flat = torch.full((rows * pitch + shift,), 0x7f, dtype=torch.int8)  # NaN as E4M3
            v = flat[shift:].view(rows, pitch)[:, :cols]
            v.copy_(src.t() if col else src)
            v = flat.to(gpu)[shift:].view(rows, pitch)[:, :cols]
            yield v.t() if col else v


@pytest.mark.parametrize("N", [1, 2, 15, 16, 17, 31, 32, 33, 48, 63, 64])
@pytest.mark.parametrize("K", [200, 256, 1])
@pytest.mark.parametrize("chunk", [None, 3])
def test_narrow_int8(gpu, N, K, chunk):
    """The narrow kernel: int32 and row-mean bit-exact and per-block within
    1e-5 on every layout, unsplit rows (one longer than 24 tiles where K
    allows) and split ones, empty rows and a misaligned output included."""
    n_bc = -(-K // 32)
    case = cases.uniform_blocks(300, K, N, min(6 * n_bc, 10 * n_bc - 1), seed=N)
    q = void_amd.quantize_void_tensor(cases.make_void_tensor(case, "cpu"))
    A = oracle.Bsr(q.values.numpy(), q.scales.numpy(), case.block_rows, case.block_cols, (300, K))
    bq, bs = oracle.quantize_i8_tensor(case.b)
    acc = oracle.i8_acc(A, bq)
    mean = oracle.row_mean(A, acc, bs)
    qd = q.to(gpu)
    wide = torch.full((300, N + 3), -7.0, device=gpu)
    for b in _layouts(bq, gpu):
        kw = dict(chunk_tiles=chunk)
        got = void_amd.void_spmm_int8(qd, b, epilogue="raw_i32", **kw)
        assert np.array_equal(got.cpu().numpy(), acc)
        got = void_amd.void_spmm_int8(qd, b, b_scale=float(bs), out=wide[:, 1:N + 1], **kw).cpu().numpy()
        assert np.array_equal(np.ascontiguousarray(got).view(np.int32), mean.view(np.int32))
        assert bool((wide[:, 0] == -7).all()) and bool((wide[:, N + 1:] == -7).all())
        first = void_amd.void_spmm_int8(qd, b, b_scale=float(bs), epilogue="per_block", **kw)
        again = void_amd.void_spmm_int8(qd, b, b_scale=float(bs), epilogue="per_block", **kw)
        assert torch.equal(first, again)
        t = q.values.double() * q.scales.double()[:, None, None]
        dense = torch.zeros(320, 32 * n_bc, dtype=torch.float64)
        for i, (r, c) in enumerate(zip(case.block_rows, case.block_cols)):
            dense[32 * r:32 * r + 32, 32 * c:32 * c + 32] = t[i]
        dense = dense[:300, :K]
        bd = torch.from_numpy(bq).double() * float(bs)
        assert bool(((first.double().cpu() - dense @ bd).abs() <= 1e-5 * (dense.abs() @ bd.abs()) + 1e-30).all())


@pytest.mark.parametrize("N", [1, 17, 32, 64])
@pytest.mark.parametrize("chunk", [None, 5])
def test_narrow_long_rows_and_activation(gpu, N, chunk):
    """Rows of up to 64 tiles, per-column scales, bias and GELU into bf16 and fp16."""
    case = cases.uniform_blocks(160, 4096, N, 300, seed=N)
    q = void_amd.quantize_void_tensor(cases.make_void_tensor(case, "cpu"))
    bq, bs = oracle.quantize_i8_columns(case.b)
    bias = torch.linspace(-1, 1, N)
    dense = torch.zeros(160, 4096, dtype=torch.float64)
    t = q.values.double() * q.scales.double()[:, None, None]
    for i, (r, c) in enumerate(zip(case.block_rows, case.block_cols)):
        dense[32 * r:32 * r + 32, 32 * c:32 * c + 32] = t[i]
    x = (dense @ (torch.from_numpy(bq).double() * torch.from_numpy(bs).double()) + bias.double()) * 0.02
    small = torch.from_numpy(bs * np.float32(0.02))
    ref = x * torch.sigmoid(2 * 0.7978845608 * (x + 0.044715 * x ** 3))
    for dtype, rnd in ((torch.bfloat16, 2.0 ** -8), (torch.float16, 2.0 ** -11)):
        for b in _layouts(bq, gpu):
            out = void_amd.void_spmm_int8(q.to(gpu), b, b_scale=small.to(gpu), bias=0.02 * bias.to(gpu),
                                          epilogue="per_block", out_dtype=dtype, activation="gelu", chunk_tiles=chunk)
            assert bool(((out.double().cpu() - ref).abs() <= rnd * ref.abs() + 1e-4).all())


@pytest.mark.parametrize("N", [1, 16, 33, 64])
def test_narrow_fp8(gpu, N):
    """E4M3 on every layout with NaN codes in the bytes around B."""
    case = cases.uniform_blocks(96, 200, N, 14, seed=N)
    f8 = void_amd.void_tensor_to_fp8(cases.make_void_tensor(case, "cpu"))
    codes = torch.from_numpy(case.b).clamp(-400, 400).to(torch.float8_e4m3fn)
    dense = torch.zeros(96, 224, dtype=torch.float64)
    t = f8.values_fp8.double() * f8.scaling_info.scale.double()[:, None, None]
    for i, (r, c) in enumerate(zip(case.block_rows, case.block_cols)):
        dense[32 * r:32 * r + 32, 32 * c:32 * c + 32] = t[i]
    dense = dense[:, :200]
    ref, bound = dense @ codes.double(), dense.abs() @ codes.double().abs()
    for b in _layouts(codes.view(torch.int8).numpy(), gpu):
        raw = b.view(torch.float8_e4m3fn) if b.stride(1) == 1 else b.t().view(torch.float8_e4m3fn).t()
        out = void_amd.void_spmm_fp8(f8.to(gpu), raw, output_dtype=torch.float32).double().cpu()
        assert bool(((out - ref).abs() <= 2.0 ** -13 * bound + 1e-30).all())


@pytest.mark.parametrize("K,N", [(203, 65), (256, 130), (200, 250), (96, 512), (1, 70), (33, 129)])
def test_column_major_any_alignment(gpu, K, N):
    """Column-major 8-bit B wider than the narrow kernel takes, at every
    alignment: copied to aligned rows where only single-byte loads are left."""
    case = cases.uniform_blocks(170, K, N, max(1, 5 * -(-K // 32) // 2), seed=N)
    q = void_amd.quantize_void_tensor(cases.make_void_tensor(case, "cpu")).to(gpu)
    A = oracle.Bsr(q.values.cpu().numpy(), q.scales.cpu().numpy(), case.block_rows, case.block_cols, (170, K))
    bq, _ = oracle.quantize_i8_tensor(case.b)
    acc = oracle.i8_acc(A, bq)
    for b in _layouts(bq, gpu):
        assert np.array_equal(void_amd.void_spmm_int8(q, b, epilogue="raw_i32").cpu().numpy(), acc)
        if b.stride(0) == 1 and K > 1:
            copy = _runtime.row_major_copy_b8(b, b.stride(1))
            assert copy.stride(0) % 16 == 0 and torch.equal(copy, b)


@pytest.mark.parametrize("M,N", [(512, 512), (4096, 2048)])
def test_narrow_named_on_a_wide_call(gpu, monkeypatch, M, N):
    """VOID_AMD_KERNEL=narrow on a call that is too wide for it: the default
    kernel, bit for bit (per-block sums in fp32 differ between ring shapes)."""
    case = cases.uniform_blocks(M, 1024, N, M // 32 * 16, seed=N)
    q = void_amd.quantize_void_tensor(cases.make_void_tensor(case, "cpu")).to(gpu)
    bq, bs = oracle.quantize_i8_columns(case.b)
    out = {}
    for kernel in (None, "narrow"):
        if kernel:
            monkeypatch.setenv("VOID_AMD_KERNEL", kernel)
        out[kernel] = void_amd.void_spmm_int8(q, torch.from_numpy(bq).to(gpu), b_scale=torch.from_numpy(bs).to(gpu),
                                              epilogue="per_block")
    assert torch.equal(out[None], out["narrow"])
