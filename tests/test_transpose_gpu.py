"""void_transpose through contiguous_2d: exact copies at tile edges, remainders
and unaligned columns, and the operand layouts that keep torch's own copy."""

import pytest
import torch

from void_amd import _runtime

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(1, 2), (2, 1), (7, 9), (64, 64), (65, 63), (128, 72), (200, 1000), (1001, 66)])
@pytest.mark.parametrize("pad,shift", [(0, 0), (5, 0), (8, 1)])
def test_column_major_copy(gpu, monkeypatch, dtype, shape, pad, shift):
    monkeypatch.setattr(_runtime, "TRANSPOSE_MIN_NUMEL", 1)
    R, C = shape
    flat = torch.randn(C * (R + pad) + shift, device=gpu).to(dtype)
    flat[shift] = float("nan")
    t = flat[shift:].view(C, R + pad)[:, :R].t()
    out = _runtime.contiguous_2d(t)
    assert out.is_contiguous() and out.shape == t.shape
    bits = {2: torch.int16, 4: torch.int32}[t.element_size()]
    assert torch.equal(out.view(bits), t.contiguous().view(bits))


def test_other_layouts(gpu, monkeypatch):
    monkeypatch.setattr(_runtime, "TRANSPOSE_MIN_NUMEL", 1)
    x = torch.randn(6, 8, device=gpu)
    assert _runtime.contiguous_2d(x) is x
    for t in (x[::2], x.t().expand(8, 6)[::2], x[:, :1].expand(6, 5), torch.empty(0, 4, device=gpu).t(),
              x.double().t()):
        assert torch.equal(_runtime.contiguous_2d(t), t.contiguous())
        assert _runtime.contiguous_2d(t).is_contiguous()
