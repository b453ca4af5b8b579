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


# A column-major B (X.t() of token-major activations) runs the register-staged
# column-group loop, whose 16-byte loads from one column each use a quarter
# of a 128-byte line; the LDS-DMA ring reads row-major B in whole lines.  When
# the slabs gathered (32 N bytes per tile) exceed 32 times B itself, a
# row-major copy of B (one pass over it) pays for itself: on the FFN config
# the SpMM with GELU took 183 us with B column-major against 91 us
# row-major.  VOID_AMD_BT=0 / 1 forces the copy off / on.


# Columns that are not 16-byte aligned (or K not a multiple of 32) leave only
# single-byte loads (``bytewise``): there the copy always pays (4615 x 646,
# 554 tiles, N = 1248: 150 -> 19 us).
COL_MAJOR_COPY_RATIO = 32


def copy_col_major_b(n_blocks: int, K: int, bytewise: bool = False) -> bool:
    env = os.environ.get("VOID_AMD_BT")
    if env in ("0", "1"):
        return env == "1"
    return bytewise or 32 * n_blocks >= COL_MAJOR_COPY_RATIO * max(K, 1)


# An 8-bit row-major B whose rows are not 16-byte aligned (N or the row pitch
# not a multiple of 16, or a shifted view) cannot feed the LDS-DMA ring; the
# general kernel gathers it by 4-byte loads where rows and C allow that
# (``dword``), byte by byte otherwise.  A copy to aligned rows costs a launch
# and one pass over B (2-4 us).  Against the bytewise loads it always pays
# (46 tiles, N = 155: 24.1 -> 8.2 us; 2950 tiles, N = 730: 131 -> 19.6 us with
# the copy).  Against the 4-byte loads it pays where the slabs gathered exceed
# 32 times B over more than one panel (14336 x 4096, 14336 tiles, N = 500:
# 51 -> 43 us, N = 2004: 161 -> 121 us; 4096 x 4096, 1638 tiles (13 x B), N = 500:
# 10.2 against 14.1 us with the copy; 14336 tiles, N = 100: 15.8 against 16.4).
# VOID_AMD_PAD=0 / 1 forces it off / on.
def aligned_pitch(N: int) -> int:
    """Row pitch of an aligned copy of an 8-bit B: whole 128-byte lines, so
    that a panel's slab rows start on a line (N up to 64: whole 16-byte
    chunks, one line holding several rows)."""
    return (N + 127) // 128 * 128 if N > 64 else (N + 15) // 16 * 16


def copy_unaligned_b(n_blocks: int, K: int, N: int, dword: bool) -> bool:
    env = os.environ.get("VOID_AMD_PAD")
    if env in ("0", "1"):
        return env == "1"
    if K * aligned_pitch(N) >= 1 << 31:  # past the ring's 31-bit offsets
        return False
    return not dword or (N > PANEL_COLUMNS and 32 * n_blocks >= COL_MAJOR_COPY_RATIO * max(K, 1))
