"""Workloads that a program built on void_amd runs, with sizes, inputs,
tolerances and 64-bit results.

A case is a dict of plain values.  ``kind`` names the entry point:

  int8   void_spmm_int8 / void_spmm_gelu on an INT8 weight (per-tile scales),
  fp8    void_spmm_fp8 on an E4M3 weight,
  float  void_spmm on a float weight,
  fused  FusedSparseLinear.forward (weight in its own dtype, GELU, row bias),
  train  SparseLinear forward and backward.

M, K, N: weight M x K, N columns of the dense operand (tokens).  ``pattern``
places the nonzero 32x32 tiles: "uniform" takes ``tiles`` positions at random,
"powerlaw" gives every block-row min(Zipf(1.5), K / 32) tiles.
"""

from __future__ import annotations

import math

import numpy as np
import torch

import void_amd

T = 32
DEV = "cuda"
DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
SIZE = {"fp32": 4, "bf16": 2, "fp16": 2, "int8": 1, "e4m3": 1}


def _case(name, kind, M, K, N, **kw):
    c = dict(name=name, kind=kind, M=M, K=K, N=N, pattern="uniform", b="", layout="row", out="fp32", act="none",
             bias=False)
    c.update(kw)
    return c


def listed():
    return [
        # The smallest call: a 512 x 512 matrix of which every tile is active,
        # the float operand quantised inside the call (the API's default form).
        _case("int8_small_float_b", "int8", 512, 512, 128, tiles=256, b="fp32"),
        # Decode: 16 tokens against a pruned FFN up-projection, activations
        # token-major with one scale per token, bias and GELU fused.
        _case("int8_decode_ffn", "int8", 14336, 4096, 16, tiles=14336, b="int8", layout="col", out="bf16",
              act="gelu", bias=True),
        # The headline matrix multiply: 4096 x 4096 at 90 % block sparsity.
        _case("int8_90pct", "int8", 4096, 4096, 512, tiles=1638, b="int8"),
        # A call with no size a multiple of anything, float operand quantised
        # inside it: a graph or embedding matrix of arbitrary shape.
        _case("int8_ragged_float_b", "int8", 5003, 3001, 730, tiles=2950, b="fp32"),
        # Long-tailed block-rows (graphs): the Stream-K partition with split rows.
        _case("int8_powerlaw", "int8", 16384, 16384, 256, pattern="powerlaw", b="int8"),
        # Prefill of the pruned FFN up-projection with GELU.
        _case("int8_prefill_ffn", "int8", 14336, 4096, 2048, tiles=14336, b="int8", out="bf16", act="gelu"),
        # E4M3 weights and activations at 80 % block sparsity.
        _case("fp8_80pct", "fp8", 4096, 4096, 512, tiles=3277, b="e4m3", out="bf16"),
        # The same weights with the API's default operand, a float32 matrix.
        _case("fp8_80pct_float_b", "fp8", 4096, 4096, 512, tiles=3277, b="fp32", out="fp16"),
        # Float SpMM in float32, the library's plainest call.
        _case("float32_80pct", "float", 4096, 4096, 1024, tiles=3277, b="fp32"),
        # Inference through the fused linear layer in bf16, token-major
        # activations as a model holds them.
        _case("fused_linear_bf16", "fused", 14336, 4096, 2048, tiles=14336, b="bf16", out="bf16", act="gelu",
              bias=True),
        # Fine-tuning a sparse layer in float32: forward and both gradients.
        _case("train_linear_fp32", "train", 4096, 4096, 1024, tiles=3277, b="fp32", bias=True),
        # The same in bf16 at the FFN's size.
        _case("train_linear_bf16", "train", 14336, 4096, 2048, tiles=14336, b="bf16", out="bf16", bias=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """A size in [lo, hi], log-uniform; a multiple of 32 half of the time."""
    v = _log(rng, lo, hi)
    return max(lo // T * T, v // T * T) if rng.random() < 0.5 else v


def draw(rng):
    kind = rng.choice(["int8", "int8", "int8", "fp8", "fp8", "float", "fused", "train"])
    M, K = _size(rng, 512, 16384), _size(rng, 512, 8192)
    N = rng.choice([_log(rng, 1, 64), _size(rng, 64, 2048), _size(rng, 64, 2048)])
    grid = -(-M // T) * -(-K // T)
    tiles = max(1, int(grid * math.exp(rng.uniform(math.log(0.05), math.log(0.4)))))
    # No more tile products than the largest listed case, scaled down for the
    # kinds that run several passes.
    most = 14336 * 2048 if kind in ("int8", "fused") else 14336 * 1024
    tiles = max(1, min(tiles, 14336, most // N))
    c = _case("", kind, M, K, N, tiles=tiles)
    del c["name"]
    if kind == "int8":
        c["b"] = rng.choice(["int8", "int8", "fp32"])
        if c["b"] == "int8":
            c["layout"] = rng.choice(["row", "row", "col"])
            c["out"] = rng.choice(["fp32", "bf16", "fp16"])
            c["act"] = rng.choice(["none", "gelu"])
            c["bias"] = rng.random() < 0.5
            if rng.random() < 0.2:
                c["pattern"], c["K"], c["M"] = "powerlaw", 8192, min(M, 8192)
                c["N"] = min(N, 512)
                del c["tiles"]
    elif kind == "fp8":
        c["b"] = rng.choice(["e4m3", "fp32", "bf16"])
        c["out"] = rng.choice(["fp32", "bf16", "fp16"])
    else:
        c["b"] = rng.choice(["fp32", "bf16", "fp16"]) if kind != "train" else rng.choice(["fp32", "bf16"])
        c["out"] = c["b"]
        c["act"] = rng.choice(["gelu", "relu"]) if kind == "fused" else "none"
        c["bias"] = kind != "float"
    return c


# ---- inputs ---------------------------------------------------------------

def _counts(case):
    """Tiles per block-row of a power-law matrix (part of the case, not of the seed)."""
    n_br, n_bc = -(-case["M"] // T), -(-case["K"] // T)
    return np.minimum(np.random.default_rng(0).zipf(1.5, size=n_br), n_bc)


def _n_tiles(case):
    return int(_counts(case).sum()) if case["pattern"] == "powerlaw" else case["tiles"]


def _positions(case, seed):
    rng = np.random.default_rng(seed)
    n_br, n_bc = -(-case["M"] // T), -(-case["K"] // T)
    if case["pattern"] == "powerlaw":
        counts = _counts(case)
        key = rng.random((n_br, n_bc))
        order = np.argsort(key, axis=1)
        br = np.repeat(np.arange(n_br), counts)
        bc = np.concatenate([order[r, :c] for r, c in enumerate(counts)])
    else:
        pick = rng.choice(n_br * n_bc, case["tiles"], replace=False)
        br, bc = pick // n_bc, pick % n_bc
    morton = void_amd.morton_encode_batch(br, bc).astype(np.int64)
    o = np.argsort(morton, kind="stable")
    return br[o].astype(np.int32), bc[o].astype(np.int32), morton[o]


def _raw(case, seed):
    """The float inputs: tile positions, tiles, dense operand, bias and (train) output gradient."""
    M, K, N = case["M"], case["K"], case["N"]
    br, bc, morton = _positions(case, seed)
    g = torch.Generator(device=DEV)
    g.manual_seed(seed + 1)
    randn = lambda *s: torch.randn(*s, generator=g, device=DEV)
    layer = case["kind"] in ("fused", "train")
    std = 0.02 if layer or case["act"] != "none" else 1.0
    tiles = randn(len(br), T, T) * std
    # Parts of edge tiles outside the matrix are zero, as the conversions leave them.
    rows = torch.from_numpy(br).to(DEV)[:, None] * T + torch.arange(T, device=DEV)
    cols = torch.from_numpy(bc).to(DEV)[:, None] * T + torch.arange(T, device=DEV)
    tiles *= (rows < M)[:, :, None] & (cols < K)[:, None, :]
    dense = randn(N, K) if layer or case["layout"] == "col" else randn(K, N)
    bias = randn(M if layer else N) * 0.1 if case["bias"] else None
    grad = randn(N, M) if case["kind"] == "train" else None
    return br, bc, morton, tiles, dense, bias, grad


def _void_tensor(case, br, bc, morton, tiles, dtype):
    n_br, n_bc = -(-case["M"] // T), -(-case["K"] // T)
    return void_amd.VOIDTensor(
        values=tiles.to(dtype), block_rows=torch.from_numpy(br).to(DEV), block_cols=torch.from_numpy(bc).to(DEV),
        morton_codes=torch.from_numpy(morton).to(DEV), shape=(case["M"], case["K"]), tile_size=(T, T),
        nnz_original=len(br) * T * T, n_blocks=len(br), density=len(br) / (n_br * n_bc), dtype=dtype)


def _quantize_columns(x, dim):
    """Symmetric INT8 with one scale per column of the dense operand (per token)."""
    scale = torch.clamp(x.abs().amax(dim=dim, keepdim=True) / 128, min=1e-8)
    return (x / scale).round().clamp(-128, 127).to(torch.int8), scale.reshape(-1)


def prepare(case, seed):
    br, bc, morton, tiles, dense, bias, grad = _raw(case, seed)
    kind = case["kind"]
    st = {"case": case}
    if kind == "int8":
        st["a"] = void_amd.quantize_void_tensor(_void_tensor(case, br, bc, morton, tiles, torch.float32))
        if case["b"] == "int8":
            q, s = _quantize_columns(dense, 1 if case["layout"] == "col" else 0)
            st["b"], st["scale"] = (q.t() if case["layout"] == "col" else q), s
        else:
            st["b"], st["scale"] = dense, None
        st["bias"] = bias
    elif kind == "fp8":
        st["a"] = void_amd.void_tensor_to_fp8(_void_tensor(case, br, bc, morton, tiles, torch.float32))
        if case["b"] == "e4m3":
            s = float(dense.abs().max()) / 448
            st["b"], st["scale"] = (dense / s).clamp(-448, 448).to(torch.float8_e4m3fn), s
        else:
            st["b"], st["scale"] = dense.to(DTYPES[case["b"]]), None
    elif kind == "float":
        dt = DTYPES[case["b"]]
        st["a"], st["b"] = _void_tensor(case, br, bc, morton, tiles, dt), dense.to(dt)
    elif kind == "fused":
        dt = DTYPES[case["b"]]
        layer = void_amd.FusedSparseLinear(case["K"], case["M"], _void_tensor(case, br, bc, morton, tiles, dt),
                                           activation=case["act"]).to(DEV)
        with torch.no_grad():
            layer.bias.copy_(bias)
        st["layer"], st["x"] = layer, dense.to(dt)
    else:
        dt = DTYPES[case["b"]]
        layer = void_amd.SparseLinear(case["K"], case["M"], _void_tensor(case, br, bc, morton, tiles, dt)).to(DEV)
        with torch.no_grad():
            layer.bias.copy_(bias)
        st["layer"], st["x"], st["grad"] = layer, dense.to(dt).requires_grad_(), grad.to(dt)
    return st


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "int8":
        if case["act"] == "gelu":
            return void_amd.void_spmm_gelu(state["a"], state["b"], state["bias"], b_scale=state["scale"],
                                           out_dtype=DTYPES[case["out"]])
        if case["b"] == "int8":
            return void_amd.void_spmm_int8(state["a"], state["b"], b_scale=state["scale"], bias=state["bias"],
                                           epilogue="per_block", out_dtype=DTYPES[case["out"]])
        return void_amd.void_spmm_int8(state["a"], state["b"])
    if kind == "fp8":
        return void_amd.void_spmm_fp8(state["a"], state["b"], DTYPES[case["out"]], b_scale=state["scale"])
    if kind == "float":
        return void_amd.void_spmm(state["a"], state["b"])
    layer, x = state["layer"], state["x"]
    if kind == "fused":
        with torch.no_grad():
            return layer(x)
    layer.zero_grad(set_to_none=True)
    x.grad = None
    y = layer(x)
    y.backward(state["grad"])
    return [y.detach(), x.grad, layer.sparse_weight.values.grad, layer.bias.grad]


def work(case):
    M, K, N, nb = case["M"], case["K"], case["N"], _n_tiles(case)
    kind = case["kind"]
    esz = SIZE[case["b"]]
    flops = 2 * nb * T * T * N
    a = nb * T * T * (1 if kind in ("int8", "fp8") else esz) + 8 * nb
    b, c = K * N * esz, M * N * SIZE[case["out"]]
    if kind != "train":
        return {"bytes": a + b + c + (4 * N if case["b"] == "int8" else 0), "flops": flops}
    # Forward reads the tiles and x and writes y; backward reads y's gradient
    # and writes the gradients of x, the tiles and the bias.
    return {"bytes": 2 * a + 2 * b + 2 * c + M * esz, "flops": 3 * flops}


def tolerance(case):
    # About four times the measured difference from the 64-bit result.
    if case["out"] != "fp32":
        # Rounding of the output: 1.7e-3 (bf16), 2.1e-4 (fp16); a bf16 layer
        # with a separate bias rounds twice (2.3e-3).
        return {"rel": {"bf16": 9e-3 if case["kind"] == "train" else 7e-3, "fp16": 9e-4}[case["out"]]}
    if case["kind"] == "fp8":
        # The fp8 matrix cores' sums: 1.5e-5; a float32 operand in two bf16
        # parts: 4.9e-6; a bf16 operand: 32-bit sums of exact products.
        return {"rel": {"e4m3": 6e-5, "fp32": 2e-5, "bf16": 1e-6}[case["b"]]}
    if case["kind"] == "int8":
        return {"rel": 1e-6}  # 1.9e-7: exact sums, a few 32-bit multiplications
    return {"rel": 3.5e-6}  # 8.1e-7: 32-bit sums over up to 2048 terms


# ---- 64-bit results -------------------------------------------------------

def _dense_a(case, br, bc, tiles):
    n_br, n_bc = -(-case["M"] // T), -(-case["K"] // T)
    grid = torch.zeros(n_br * n_bc, T, T, dtype=torch.float64, device=DEV)
    grid[torch.from_numpy(br.astype(np.int64) * n_bc + bc).to(DEV)] = tiles.double()
    return grid.view(n_br, n_bc, T, T).permute(0, 2, 1, 3).reshape(n_br * T, n_bc * T)[:case["M"], :case["K"]]


def _act(x, name):
    if name == "relu":
        return torch.relu(x)
    if name == "gelu":
        return x * torch.sigmoid(2 * 0.7978845608 * (x + 0.044715 * x * x * x))
    return x


def exact(case, seed):
    br, bc, _, tiles, dense, bias, grad = _raw(case, seed)
    kind = case["kind"]
    if kind == "int8":
        s = torch.clamp(tiles.abs().amax(dim=(1, 2)) / 128, min=1e-8)
        q = (tiles / s[:, None, None]).round().clamp(-128, 127).double()
        if case["b"] == "int8":
            bq, bs = _quantize_columns(dense, 1 if case["layout"] == "col" else 0)
            bd = bq.double() * bs.double()[:, None] if case["layout"] == "col" else bq.double() * bs.double()
            a = _dense_a(case, br, bc, q * s.double()[:, None, None])
            c = a @ (bd.t() if case["layout"] == "col" else bd)
            if bias is not None:
                c = c + bias.double()
            return _act(c, case["act"])
        # Row-mean epilogue: integer sums times the mean scale of the block-row.
        bs = torch.clamp(dense.abs().max() / 128, min=1e-8)
        bq = (dense / bs).round().clamp(-128, 127).double()
        n_br = -(-case["M"] // T)
        rows = torch.from_numpy(br).long().to(DEV)
        total = torch.zeros(n_br, dtype=torch.float64, device=DEV).index_add_(0, rows, s.double() * bs.double())
        count = torch.zeros(n_br, dtype=torch.float64, device=DEV).index_add_(0, rows, torch.ones_like(s).double())
        mean = (total / count.clamp(min=1)).repeat_interleave(T)[:case["M"]]
        return (_dense_a(case, br, bc, q) @ bq) * mean[:, None]
    if kind == "fp8":
        amax = tiles.abs().amax(dim=(1, 2))
        s = torch.clamp((amax.double() / 448).float(), min=1e-12)
        q = (tiles * (torch.ones_like(s) / s)[:, None, None]).clamp(-448, 448).to(torch.float8_e4m3fn)
        a = _dense_a(case, br, bc, q.float().double() * s.double()[:, None, None])
        if case["b"] == "e4m3":
            bs = float(dense.abs().max()) / 448
            bd = (dense / bs).clamp(-448, 448).to(torch.float8_e4m3fn).float().double() * bs
        else:
            bd = dense.to(DTYPES[case["b"]]).double()
        return a @ bd
    dt = DTYPES[case["b"]]
    a = _dense_a(case, br, bc, tiles.to(dt))
    if kind == "float":
        return a @ dense.to(dt).double()
    x = dense.to(dt).double()
    if kind == "fused":
        return _act(x @ a.t() + bias.double(), case["act"])
    y = x @ a.t() + bias.to(dt).double()
    gy = grad.to(dt).double()
    M, K, N = case["M"], case["K"], case["N"]
    n_br, n_bc = -(-M // T), -(-K // T)
    gpad = torch.zeros(N, n_br * T, dtype=torch.float64, device=DEV)
    xpad = torch.zeros(N, n_bc * T, dtype=torch.float64, device=DEV)
    gpad[:, :M], xpad[:, :K] = gy, x
    gv = (gpad.t() @ xpad).view(n_br, T, n_bc, T).permute(0, 2, 1, 3)
    gv = gv[torch.from_numpy(br).long().to(DEV), torch.from_numpy(bc).long().to(DEV)].contiguous()
    return [y, gy @ a, gv, gy.sum(0)]
