"""How the host lays out dense operands for the ring kernels, from sizes and
strides alone (no GPU): what is used in place, copied, and to which pitch."""

import pytest

from void_amd import _runtime, tuning

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


@pytest.fixture(autouse=True)
def no_forcing(monkeypatch):
    for name in ("VOID_AMD_PAD", "VOID_AMD_BT"):
        monkeypatch.delenv(name, raising=False)


@pytest.mark.parametrize("n,max_row,K,N,row8,col8,f32", [
    (46, 4, 512, 155, True, True, False),          # a small matrix: byte loads lose, fp32 in place does not
    (400, 23, 4099, 101, True, True, True),
    (2950, 26, 3001, 730, True, True, True),
    (200, 5, 4099, 101, True, True, False),        # short rows
    (50, 7, 1 << 20, 730, False, False, False),    # 1.2 MB gathered of a 0.8 GB B
    (3200, 25, 1 << 20, 730, False, False, False),
    (400, 23, 262147, 101, True, True, False),
])
def test_copy_rules_weigh_the_pass_over_b(n, max_row, K, N, row8, col8, f32):
    """A copy is made where what the tiles gather outweighs the pass over B
    (both sides measured; the figures stand at the rules)."""
    assert tuning.copy_unaligned_b(n, K, N, False, max_row) == row8
    assert tuning.copy_col_major_b(n, K, True, N, max_row) == col8
    assert tuning.pad_float_b(n, max_row, K, N, -(-N // 32) * 32, 4, True) == f32


def test_copy_rules_forced(monkeypatch):
    monkeypatch.setenv("VOID_AMD_PAD", "1")
    assert tuning.copy_unaligned_b(1, 1 << 20, 101, False, 1)
    monkeypatch.setenv("VOID_AMD_PAD", "0")
    assert not tuning.copy_unaligned_b(14336, 4096, 2004, True, 64)
    for forced in (True, False):
        monkeypatch.setattr(tuning, "PAD_FLOAT", forced)
        assert _runtime._pad_forced(1, 1) is forced and _runtime._pad_forced(14336, 2004) is forced


def test_sddmm_copies_weigh_the_passes():
    pads = lambda n, K, N, esz, in_place: tuning.pad_float_sddmm(
        n, N, esz, [(r, -(-N * esz // 128) * 128 // esz, in_place) for r in (4096, K)])
    assert not pads(400, 4099, 101, 4, True) and pads(3200, 4099, 101, 4, True)
    assert pads(3200, 4099, 730, 4, True) and not pads(3200, 262147, 730, 4, True)
    assert pads(400, 262147, 730, 4, False)       # copied either way (token-major operands)
    assert not pads(400, 4099, 101, 2, True) and pads(3200, 262147, 730, 2, True)
