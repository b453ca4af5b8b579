"""How the host lays out dense operands for the ring kernels, from sizes and
strides alone (no GPU): what is used in place, copied, and to which pitch."""

import pytest

from void_amd import _runtime

LIM = _runtime.RING_LIMIT


@pytest.mark.parametrize("R,C,s0,esz,want", [
    (100, 40, 40, 4, (True, 40)),         # aligned rows in place
    (100, 37, 40, 4, (True, 40)),         # any width inside an aligned pitch
    (100, 37, 37, 4, (False, 64)),        # whole 128-byte lines
    (100, 5, 5, 4, (False, 8)),           # up to one line: 16-byte chunks
    (100, 37, 37, 2, (False, 40)),
    (100, 65, 65, 2, (False, 128)),
    (8192, 37, 65536, 4, (False, 64)),    # a narrow view whose span is 2 GiB
    (8192, 65510, 65510, 4, (False, 65512)),  # whole lines would reach 2 GiB
    (16384, 32741, 32741, 4, (False, 32744)),
    (8192, 65536, 65536, 4, None),        # no pitch fits
    (8180, 65533, 65533, 4, None),        # rows count in whole tiles
])
def test_padded_layout(R, C, s0, esz, want):
    assert _runtime.padded_layout(R, C, s0, 1, 0, esz, limit=LIM) == want
    if want is not None:
        assert -(-R // 32) * 32 * want[1] * esz < LIM and want[1] * esz % 16 == 0 and want[1] >= C


def test_padded_layout_in_place_needs():
    assert _runtime.padded_layout(64, 40, 40, 1, 4, 4) == (False, 64)       # shifted view
    assert _runtime.padded_layout(64, 40, 1, 64, 0, 4) == (False, 64)       # column-major
    assert _runtime.padded_layout(64, 40, 0, 1, 0, 4) == (False, 64)        # one row broadcast
    assert _runtime.padded_layout(64, 37, 40, 1, 0, 4, zero_tail=True) == (False, 64)
    assert _runtime.padded_layout(64, 40, 40, 1, 0, 4, zero_tail=True) == (True, 40)
    assert _runtime.padded_layout(8192, 65536, 65536, 1, 0, 4) == (True, 65536)  # no limit asked for
