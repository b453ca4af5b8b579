"""Fixed gfx950 launch configuration (replaces the reference's autotuner).

The reference searches TILE_N x num_warps x num_stages at run time and keeps
a JSON cache (void/autotune.py:39-104, 345-381).  On MI355X the kernel shape
is fixed by the hardware instead:

* one workgroup = 4 wave64s, one 32-row block-row x 128-column panel of C,
  each wave owning 32 columns; the LDS-DMA column-group kernel uses 40 KB of
  LDS and about 100 registers per lane -> 4 workgroups per CU;
* 256 CUs in 8 XCDs -> 1024 resident workgroups;
* the only shape-dependent knob is the Stream-K chunk: the most tiles one
  work item may take before its block-row is split.  The column-group
  kernel takes items of at most 64 tiles (an item's block columns and
  scales sit one per lane), and a split row pays a partial-tile round trip
  through L2 (coherent 16-byte stores, an atomic, coherent loads):
  - every block-row fits in 64 tiles: chunk 64, nothing is split;
  - some block-row is longer: 1.3 times the average work per resident
    workgroup slot, clamped to [32, 64].  Plans with split rows run the
    two-ring kernel (8-wave workgroups, 2 per CU), so a slot is 1/512 of
    the chip.  Measured on the power-law config (Zipf rows up to 512 tiles,
    cold): two-ring kernel at chunk 32 / 46 / 64: 33.4-33.9 / 29.5-30.0 /
    27.8-28.1 us; the one-ring kernel at 32 / 46 / 64: 30.9-31.0 / 29.4-29.5
    / 28.5-28.7 us.
"""

from __future__ import annotations

import math
import os

GFX950_CUS = 256
GFX950_XCDS = 8
WAVES_PER_WORKGROUP = 4
WORKGROUPS_PER_CU = 4
PANEL_COLUMNS = 128
TILE = 32

MIN_SPLIT_CHUNK = 32

# (name, longest item of the column-group kernel, factor on the per-slot average)
CHUNK_TABLE = {
    "int8": (64, 1.3),
    "fp8": (64, 1.3),
}


# Longest work item of the kernels that stage fp32 B slabs (the float SpMM
# and the E4M3 x fp32 SpMM): they hold an item's block columns one per lane.
FP32_B_MAX_CHUNK = 64


def resident_workgroups() -> int:
    return GFX950_CUS * WORKGROUPS_PER_CU


# Workgroups per CU of the two-ring kernel that plans with split rows run.
SPLIT_WORKGROUPS_PER_CU = 2


def n_panels(N: int) -> int:
    return (N + PANEL_COLUMNS - 1) // PANEL_COLUMNS


def select_chunk(kind: str, n_blocks: int, N: int, max_row: int = 0) -> int:
    """Stream-K chunk (max tiles per work item) for a problem whose longest
    block-row has max_row tiles."""
    cg_max, factor = CHUNK_TABLE[kind]
    if max_row <= cg_max:
        return cg_max
    per_slot = n_blocks * n_panels(max(N, 1)) / (GFX950_CUS * SPLIT_WORKGROUPS_PER_CU)
    return min(cg_max, max(MIN_SPLIT_CHUNK, int(math.ceil(per_slot * factor))))


# Up to this many columns (with and without split rows) an 8-bit B runs the
# narrow kernel, which reads any layout and alignment in place: no copy of B
# is made for it.  The line is the library's own (void_spmm.hip, with what
# both sides measured).
NARROW_COLUMNS = (32, 64)


def narrow(N: int, n_split_tiles: int) -> bool:
    return N <= NARROW_COLUMNS[0 if n_split_tiles else 1]


def aligned_pitch(N: int) -> int:
    """Row pitch of an aligned copy of an 8-bit B: whole 128-byte lines, so
    that a panel's slab rows start on a line (N up to 64: whole 16-byte
    chunks, one line holding several rows)."""
    return (N + 127) // 128 * 128 if N > 64 else (N + 15) // 16 * 16


# ---- Copies of B for the LDS-DMA rings ------------------------------------
#
# A copy costs a launch and one pass over all of B; what it saves grows with
# the tiles: the chain of the longest block-row and the values gathered
# (tiles x 32 x N).  Both sides below in us, fitted to eager calls with 50, 400
# and 3200 tiles (about 3 to 20 a row), N = 101 and 730, K from 4099 to
# 1048579.  VOID_AMD_BT=0 / 1 forces the copy of a column-major 8-bit B off / on,
# VOID_AMD_PAD=0 / 1 that of a row-major one.


def _forced(name: str):
    env = os.environ.get(name)
    return env == "1" if env in ("0", "1") else None


def _pass_us(rows: int, read: int, written: int, bytes_per_us: float) -> float:
    """Time of a pass that reads and writes so many bytes a row."""
    return rows * (read + written) / bytes_per_us


# A column-major B (X.t() of token-major activations) runs the register-staged
# column-group loop, whose 16-byte loads from one column each use a quarter
# of a 128-byte line; the LDS-DMA ring reads row-major B in whole lines.  When
# the tiles gather B this many times over (32 n_blocks rows of N against K), a
# row-major copy of B (one pass over it) pays for itself: on the FFN config
# the SpMM with GELU took 183 us with B column-major against 91 us
# row-major.
COL_MAJOR_COPY_RATIO = 32


def copy_col_major_b(n_blocks: int, K: int, bytewise: bool = False, N: int = 0, max_row: int = 0) -> bool:
    """Whether an 8-bit column-major B is copied to row-major.  ``bytewise``:
    its columns are not 16-byte aligned (or K not a multiple of 32), which
    leaves single-byte loads (K = 4099, N = 101: 50 tiles 29 us in place, 17 with
    the copy; 400 tiles 55 and 17; K = 262147: 29 and 33, 57 and 36; K = 1048579:
    29 and 97, 57 and 99)."""
    forced = _forced("VOID_AMD_BT")
    if forced is not None:
        return forced
    if 32 * n_blocks >= COL_MAJOR_COPY_RATIO * max(K, 1):
        return True
    saved = 8 + 1.5 * min(max_row, 64) + 1.9e-6 * 32 * n_blocks * N  # (an item's chain: 64 tiles at most)
    return bytewise and saved > _pass_us(K, N, aligned_pitch(N), 2.6e6)


# An 8-bit row-major B whose rows are not 16-byte aligned (N or the row pitch
# not a multiple of 16, or a shifted view) cannot feed the LDS-DMA ring; the
# general kernel gathers it by 4-byte loads where rows and C allow that
# (``dword``), byte by byte otherwise.  Against the bytewise loads (us in place,
# with the copy; N = 101): K = 4099 50 tiles 24 and 17, 400 tiles 45 and 17;
# K = 262147 24 and 20, 45 and 22; K = 1048579 24 and 49, 45 and 51; N = 730,
# 3200 tiles: K = 4099 101 and 19, K = 1048579 143 and 433.  Against the 4-byte
# loads it pays where the slabs gathered exceed 32 times B over more than one
# panel (14336 x 4096, 14336 tiles, N = 500: 51 -> 43 us, N = 2004: 161 -> 121 us;
# 4096 x 4096, 1638 tiles (13 x B), N = 500: 10.2 against 14.1 us with the copy;
# 14336 tiles, N = 100: 15.8 against 16.4).
def copy_unaligned_b(n_blocks: int, K: int, N: int, dword: bool, max_row: int = 0) -> bool:
    forced = _forced("VOID_AMD_PAD")
    if forced is not None:
        return forced
    if dword:
        return N > PANEL_COLUMNS and 32 * n_blocks >= COL_MAJOR_COPY_RATIO * max(K, 1)
    saved = 10 + 1.1 * min(max_row, 64) + 1.2e-6 * 32 * n_blocks * N
    return saved > _pass_us(K, N, aligned_pitch(N), 4.2e6)


# A float B (or gradient) whose rows are not whole 16-byte chunks: copied to
# padded rows for the rings, or left to the element-wise fp32 kernels, which
# read an fp32 B in place and a 16-bit one widened (a pass of its own).  Below
# this many tiles times columns the element-wise kernels take no longer.
PAD_FLOAT_MIN_WORK = 1 << 14
PAD_FLOAT = None  # True / False forces these copies on / off (comparisons and tests)


def pad_float_b(n_blocks: int, max_row: int, K: int, N: int, pitch: int, esz: int, in_place: bool) -> bool:
    """Whether the copy to padded rows pays for a float SpMM.  ``in_place``: an
    fp32 B that would otherwise be read where it is; any other is written once
    either way.  (us without and with the copy: fp32 N = 101, K = 4099 200 tiles
    in 128 rows 13.5 and 20.4, 400 tiles in 25 rows 30 and 22, K = 262147 33 and 54;
    bf16 K = 4099 34 and 19, K = 262147 59 and 32; fp32 N = 730, 3200 tiles, K = 4099
    121 and 72, K = 262147 132 and 447.)"""
    gathered = 32e-6 * n_blocks * N
    if esz == 2:
        widened = _pass_us(K, 2 * N, 4 * N, 5.2e6)
        return 1.0 * min(max_row, 64) - 8 + 1.1 * gathered + widened > _pass_us(K, 2 * N, 2 * pitch, 4.2e6)
    saved = 1.0 * min(max_row, 64) - 4.5 + 0.5 * gathered
    return saved > (6.5 + _pass_us(K, 4 * N, 4 * pitch, 4.4e6) if in_place else 0)


def pad_float_sddmm(n_blocks: int, N: int, esz: int, operands) -> bool:
    """Whether copies to padded rows pay for an SDDMM of n_blocks tiles;
    operands: (rows, pitch, in_place) of those that would be copied.  (us without
    and with the copies: fp32 K = 4099 N = 101, 400 tiles 12.6 and 25, 3200 tiles 46
    and 23; N = 730, 400 tiles 62 and 51, 3200 tiles 287 and 68, K = 262147 396 and
    444; bf16 N = 101, 400 tiles 19.5 and 22, 3200 tiles 52 and 22.)"""
    saved = 1e-4 * n_blocks * N
    for rows, pitch, in_place in operands:
        if esz == 2:
            saved += _pass_us(rows, 2 * N, 4 * N, 5.2e6) - _pass_us(rows, 2 * N, 2 * pitch, 4.2e6)
        elif in_place:
            saved -= 6.5 + _pass_us(rows, 4 * N, 4 * pitch, 4.4e6)
    return saved + (0.02 * N - 3.5 * len(operands) if esz == 2 else -1) > 0
