"""gfx950 matmul tile policy.

Replaces the reference's Apple tile picker (reference:
src/compute/matmul/config.py:40-51: 32x32x16 .. 128x64x32 tiles, four
32-wide simdgroups).  Here a workgroup of ``sg_M x sg_N`` wave64s computes a
``tile_M x tile_N`` output tile with MFMAs (32x32 blocks); each wave owns a
``(tile_M/sg_M) x (tile_N/sg_N)`` sub-tile, i.e. ``WM x WN`` accumulator
blocks of 16 registers.  A and B k-chunks of ``tile_K`` are double-buffered
in LDS: dense, XOR-swizzled tiles filled by direct-to-LDS loads, or rows
padded by ``a_pad``/``b_pad`` floats when filled through registers (see
``TileConfig.a_layout`` / ``b_layout``).

``select_tile_config`` scores each candidate by tile area x resident waves per
SIMD x useful fraction x grid fill (``tile_score``) and takes the best; the
16-wave tiles are candidates only when the caller says the operands leave the
registers for them (``wide``).  Large problems then run as persistent
workgroups (``persistent_workgroups``) with a stream-K last round
(``uses_stream_k``).
"""

from __future__ import annotations

import functools
from dataclasses import dataclass

NUM_CUS = 256  # MI355X compute units (8 XCDs x 32)


@dataclass(frozen=True)
class TileConfig:
    tile_M: int
    tile_N: int
    tile_K: int
    sg_M: int  # waves along M
    sg_N: int  # waves along N
    a_pad: int = 4
    b_pad: int = 4
    stages: int = 2
    c_pad: int = 4  # row padding of an LDS C tile (MatmulAccumToTgFragment)
    # LDS layouts of the operand tiles.  "pad": rows padded by a_pad / b_pad,
    # filled from registers.  Filled by direct-to-LDS loads instead (dense
    # rows): A "swz" = [tile_M][tile_K] with XOR-swizzled 16-byte slots;
    # B "dense" = [tile_K][tile_N]; B "nswz" = n-major [tile_N][tile_K],
    # swizzled like A (a transposed view such as K^T, read along K).
    a_layout: str = "pad"
    b_layout: str = "pad"

    @property
    def num_threads(self) -> int:
        return 64 * self.sg_M * self.sg_N

    @property
    def tg_x(self) -> int:
        return self.num_threads

    @property
    def tg_y(self) -> int:
        return 1

    @property
    def wave_M(self) -> int:
        return self.tile_M // self.sg_M

    @property
    def wave_N(self) -> int:
        return self.tile_N // self.sg_N

    @property
    def WM(self) -> int:
        return self.wave_M // 32

    @property
    def WN(self) -> int:
        return self.wave_N // 32

    @property
    def lda(self) -> int:
        return self.tile_K if self.a_layout == "swz" else self.tile_K + self.a_pad

    @property
    def ldb(self) -> int:
        """Row pitch of the B tile: along N (k-major layouts) or along K
        (the n-major layout)."""
        if self.b_layout == "dense":
            return self.tile_N
        if self.b_layout == "nswz":
            return self.tile_K
        return self.tile_N + self.b_pad

    def a_tile_shape(self) -> tuple[int, ...]:
        return (self.stages, self.tile_M, self.lda)

    def b_tile_shape(self) -> tuple[int, ...]:
        if self.b_layout == "nswz":
            return (self.stages, self.tile_N, self.tile_K)
        return (self.stages, self.tile_K, self.ldb)

    def validate(self) -> None:
        if self.wave_M % 32 or self.wave_N % 32 or self.tile_M % self.sg_M or self.tile_N % self.sg_N:
            raise ValueError(f"wave tile must be a multiple of 32x32: {self}")
        if self.tile_K % 8:
            raise ValueError(f"tile_K must be a multiple of 8: {self}")
        if self.lda % 4:
            raise ValueError(f"A tile row pitch must be a multiple of 4 floats (128-bit reads): {self}")
        if self.num_threads > 1024:
            raise ValueError(f"at most 1024 lanes per workgroup: {self}")
        if self.a_layout not in ("pad", "swz") or self.b_layout not in ("pad", "dense", "nswz"):
            raise ValueError(f"unknown operand tile layout: {self}")
        if (self.a_layout == "swz" or self.b_layout == "nswz") and self.tile_K not in (16, 32):
            raise ValueError(f"swizzled tiles are defined for tile_K 16 and 32: {self}")


def ceil_div(a: int, b: int) -> int:
    return (a + b - 1) // b


def is_aligned_shape(M: int, K: int, N: int, config: TileConfig) -> bool:
    return M % config.tile_M == 0 and N % config.tile_N == 0 and K % config.tile_K == 0


def grid_for(M: int, N: int, config: TileConfig) -> tuple[int, int, int]:
    return (ceil_div(N, config.tile_N), ceil_div(M, config.tile_M), 1)


# Candidate tiles.  One accumulator set: wave tiles up to 128x64 (128 acc
# registers); two sets (multi-anchor): up to 64x64 per anchor.
SINGLE_ANCHOR_TILES = (
    TileConfig(256, 256, 32, 2, 4),
    TileConfig(256, 128, 32, 4, 2),
    TileConfig(128, 256, 32, 2, 4),
    TileConfig(256, 128, 32, 2, 2),
    TileConfig(128, 256, 32, 2, 2),
    TileConfig(128, 128, 32, 4, 2),
    TileConfig(128, 128, 32, 2, 2),
    TileConfig(128, 64, 32, 2, 2),
    TileConfig(64, 128, 32, 2, 2),
    TileConfig(64, 64, 32, 2, 2),
    TileConfig(32, 32, 32, 1, 1),
)

# 16-wave tiles (4 waves per SIMD): offered when the operand chunks leave the
# registers for it (no full-size gathered prologue operands).  4x4 waves of
# 64x64 on 256x256: a wave splits the operand fragments it multiplies into
# bf16 parts, (64 + 64) x 32 elements a chunk for square wave tiles against
# (128 + 32) x 32 for 2x8 waves of 128x32 (measured on MI355X, 4096^3: 750
# against 787 us; 8 waves of 128x64 731 us).
WIDE_TILES = (
    TileConfig(256, 256, 32, 4, 4),
    TileConfig(256, 128, 32, 4, 4),
)

DUAL_ANCHOR_TILES = (
    TileConfig(256, 128, 32, 4, 2),
    TileConfig(128, 128, 32, 2, 2),
    TileConfig(128, 64, 32, 2, 2),
    TileConfig(64, 128, 32, 2, 2),
    TileConfig(64, 64, 32, 2, 2),
    TileConfig(32, 32, 32, 1, 1),
)

LDS_BYTES = 163_840
VGPRS_PER_LANE = 512  # unified VGPR+AGPR file per SIMD lane (gfx950)

FORCE_TILE: TileConfig | None = None  # tuning override (measurement scripts)


def _pow2_at_least(x: int) -> int:
    p = 32
    while p < x:
        p *= 2
    return p


def tile_lds_bytes(t: TileConfig, anchors: int = 1) -> int:
    return 4 * t.stages * (t.tile_M * t.lda + anchors * t.tile_K * t.ldb)


def estimated_vgprs(t: TileConfig, anchors: int = 1) -> int:
    """Accumulators + prefetch registers + ~48 for addressing/operands."""
    acc = 16 * t.WM * t.WN * anchors
    prefetch = (t.tile_M * t.tile_K + anchors * t.tile_K * t.tile_N) // t.num_threads
    return acc + prefetch + 48


def tile_score(t: TileConfig, M: int, N: int, anchors: int = 1, batch: int = 1) -> tuple[float, float]:
    """(score, waves per SIMD).  Score = tile area (operand reuse per byte
    loaded) x resident waves per SIMD (latency hiding, capped at 4; from the
    LDS and register limits and the number of workgroups available) x the
    fraction of the tile that is real output x how well the grid fills the
    256 CUs."""
    wgs = batch * ceil_div(M, t.tile_M) * ceil_div(N, t.tile_N)
    waves = t.sg_M * t.sg_N
    by_lds = LDS_BYTES // tile_lds_bytes(t, anchors)
    by_vgpr = max(1, (4 * (VGPRS_PER_LANE // estimated_vgprs(t, anchors))) // waves)
    per_cu = max(1, min(by_lds, by_vgpr, ceil_div(wgs, NUM_CUS)))
    wps = per_cu * waves / 4
    useful = (M * N) / (ceil_div(M, t.tile_M) * t.tile_M * ceil_div(N, t.tile_N) * t.tile_N)
    fill = min(1.0, wgs / NUM_CUS)
    return t.tile_M * t.tile_N * min(wps, 4.0) * useful * fill, wps


@dataclass(frozen=True)
class FillTile:
    """A tile for problems whose best-scored tile leaves compute units idle, with
    what one 32-wide k-chunk of it costs on MI355X in microseconds: ``alone`` with
    at most one workgroup on every other compute unit, where it waits for its own
    loads and barriers; ``base + each * n`` with n workgroups on every unit, but not
    below ``shared * n``, the unit's rate.  ``registers``: factor when an operand of
    sizes it divides, or of a product in parts, goes through registers (no
    direct-to-LDS loads); ``odd``: the factors for other sizes (bounds, masked loads)
    with up to one workgroup a unit and with more.  Fitted to 10 whole shapes from
    256^3 to 2048 x 4096 x 1024, every tile in 1 to 16 parts (the pick within 10 % of
    the best), and ``odd`` to 90 more of 65 to 4096 rows, 128 to 4096 k's and 64 to
    8192 columns, where one wave of 32x32 is the worst off (2145 of them 37 us, 561 tiles of 64x64 26 us)."""

    tile: TileConfig
    alone: float
    base: float
    each: float
    registers: float = 1.05
    shared: float = 0.0
    odd: tuple[float, float] = (1.0, 1.0)


FILL_TILES = (
    FillTile(TileConfig(256, 256, 32, 4, 4), 4.0, 0.0, 5.2, 1.4, odd=(1.75, 1.5)),
    FillTile(TileConfig(256, 128, 32, 4, 4), 2.5, 0.2, 3.4, 1.1, odd=(1.25, 1.0)),
    FillTile(TileConfig(128, 256, 32, 4, 4), 2.5, 0.2, 3.4, 1.1, odd=(1.3, 1.0)),
    FillTile(TileConfig(128, 128, 32, 2, 2), 1.5, 0.25, 1.55, 1.1, odd=(1.65, 1.15)),
    FillTile(TileConfig(128, 64, 32, 2, 2), 1.0, 0.3, 0.85, odd=(1.65, 1.3)),
    FillTile(TileConfig(64, 128, 32, 2, 2), 1.0, 0.25, 0.83, odd=(1.7, 1.15)),
    FillTile(TileConfig(64, 64, 32, 2, 2), 0.65, 0.3, 0.43, 1.25, shared=0.5, odd=(1.55, 1.3)),
    FillTile(TileConfig(32, 64, 32, 1, 2), 0.5, 0.45, 0.165, shared=0.32, odd=(2.1, 1.4)),
    FillTile(TileConfig(32, 32, 32, 1, 1), 0.5, 0.42, 0.07, shared=0.175, odd=(2.25, 1.75)),
)
FILL_MAX_PARTS = 16
# Products of fewer k's keep one sum in one order: as the product of a pair or
# with a row reduction their kernels give the same bits.
FILL_PARTS_MIN_K = 1024
FILL_WORKSPACE = 64 << 20  # bytes of partial sums a split may need (both anchors' of a pair)


def fill_time(tiles: int, chunks: int, parts: int, f: FillTile, slow: tuple[float, float] = (1.0, 1.0)) -> float:
    """Microseconds of ``tiles`` tiles in ``parts`` parts each: the chunks the
    busiest compute unit walks (``slow``: factors with up to one workgroup a unit and
    with more), and for a split the partial sums (5 TB/s out, and the last workgroup
    reads its tile's at about 80 GB/s; 2 us to meet)."""
    groups = tiles * parts
    n = ceil_div(groups, NUM_CUS)
    chunk = f.alone if 2 * groups <= NUM_CUS else max(f.base + f.each * n, f.shared * n)
    time = ceil_div(chunks, parts) * chunk * slow[n > 1]
    if parts == 1:
        return time
    tile_bytes = 4 * f.tile.tile_M * f.tile.tile_N
    return time + 2.0 + groups * tile_bytes / 5e6 + parts * tile_bytes / 80e3


def _fill_candidates(M: int, N: int, min_waves: int, anchors: int) -> list[FillTile]:
    fit = [f for f in FILL_TILES if f.tile.tile_M <= _pow2_at_least(M) and f.tile.tile_N <= _pow2_at_least(N)
           and (anchors == 1 or 16 * f.tile.WM * f.tile.WN * anchors <= 128)]
    return [f for f in fit if f.tile.sg_M * f.tile.sg_N >= min_waves] or fit


@functools.lru_cache(maxsize=1024)
def filled_parts(M: int, K: int, N: int, batch: int = 1) -> int:
    """Workgroups per tile of the least ``fill_time`` (one for batched programs and
    fewer than FILL_PARTS_MIN_K k's).  It depends on the sizes alone, so that a
    product adds its terms in the same order with any epilogue and as one of a pair
    that shares its left operand.  Not where another kernel takes it: up to 64 rows
    alone (skinny) but not as one of a pair, a prologue that divides by rows (never
    in parts), a batch, 128 columns on row waves."""
    chunks = ceil_div(K, 32)
    best = (float("inf"), 1)
    for f in _fill_candidates(M, N, 1, 1):
        t = f.tile
        tiles = ceil_div(M, t.tile_M) * ceil_div(N, t.tile_N)
        for parts in range(1, FILL_MAX_PARTS + 1):
            if parts > 1 and (
                batch != 1 or K < FILL_PARTS_MIN_K or 2 * parts > chunks or tiles >= STREAM_K_MAX_WORKGROUPS
                or 2 * tiles * parts * t.tile_M * t.tile_N * 4 > FILL_WORKSPACE
            ):
                break
            best = min(best, (fill_time(batch * tiles, chunks, parts, f), parts))
    return best[1]


@functools.lru_cache(maxsize=1024)  # fusion assembles a vertex several times
def select_filled(M: int, K: int, N: int, batch: int = 1, splittable: bool = True, registers: bool = False,
                  min_waves: int = 1, anchors: int = 1) -> tuple[TileConfig, int]:
    """(tile, parts): ``filled_parts`` workgroups per tile, and the tile of least
    ``fill_time`` for them; tiles of at least ``min_waves`` waves, if M and N reach
    such a tile's size."""
    parts = filled_parts(M, K, N, batch) if splittable else 1
    chunks = ceil_div(K, 32)

    def time(f: FillTile) -> float:
        t = f.tile
        tiles = ceil_div(M, t.tile_M) * ceil_div(N, t.tile_N)
        if parts > 1 and (tiles >= STREAM_K_MAX_WORKGROUPS
                          or anchors * tiles * parts * t.tile_M * t.tile_N * 4 > FILL_WORKSPACE):
            return float("inf")
        whole = parts > 1 or is_aligned_shape(M, K, N, t)
        slow = f.odd if not whole else (f.registers, f.registers) if registers else (1.0, 1.0)
        return fill_time(batch * tiles, chunks, parts, f, slow)

    return min(_fill_candidates(M, N, min_waves, anchors), key=time).tile, parts


def fills(M: int, N: int, t: TileConfig, batch: int = 1) -> bool:
    """Whether tile ``t`` occupies at least three quarters of the compute units in
    every round of workgroups (a persistent loop, whose last round is shared out,
    always does)."""
    if persistent_workgroups(M, N, t, batch) is not None:
        return True
    tiles = batch * ceil_div(M, t.tile_M) * ceil_div(N, t.tile_N)
    return 4 * tiles >= 3 * NUM_CUS * ceil_div(tiles, NUM_CUS)


PERSISTENT = True  # tuning switch for the persistent tile loop
PERSISTENT_CAPACITY: int | None = None  # override of resident workgroups (tests)
# Split the last partial round of a persistent loop by k-chunks (stream-K)
# instead of leaving workgroups idle; single (unbatched) problems only, and
# at most STREAM_K_MAX_WORKGROUPS workgroups (the workspace head holds one
# flag word per workgroup and the error word: MT_WS_HEAD - 1 flags).
STREAM_K = True
STREAM_K_MAX_WORKGROUPS = 1023


def resident_workgroups(t: TileConfig, anchors: int = 1, extra_lds: int = 0) -> int:
    """Workgroups of tile ``t`` one compute unit holds at once, from the LDS
    size (operand tiles plus ``extra_lds`` bytes the kernel declares beside
    them) and the register estimate (4 SIMDs x 512 registers per lane)."""
    by_lds = LDS_BYTES // (tile_lds_bytes(t, anchors) + extra_lds)
    by_vgpr = (4 * (VGPRS_PER_LANE // estimated_vgprs(t, anchors))) // (t.sg_M * t.sg_N)
    return max(1, min(by_lds, by_vgpr))


LOOK_LDS_BYTES = 512  # the words of waves looking for each other, as LDS is allocated


def look_words_fit(t: TileConfig, anchors: int = 1, extra_lds: int = 0) -> bool:
    """Whether those words leave a compute unit as many workgroups of tile ``t``: the
    operand tiles of 64x64 fill its LDS five times, a pair's of 64x128 twice and of
    128x256 once."""
    lds = tile_lds_bytes(t, anchors) + extra_lds
    return LDS_BYTES // lds == LDS_BYTES // (lds + LOOK_LDS_BYTES)


def persistent_workgroups(M: int, N: int, t: TileConfig, batch: int = 1, anchors: int = 1) -> int | None:
    """Workgroups per problem for a persistent tile loop, or None when every
    tile of every problem gets a resident workgroup in one round anyway."""
    if not PERSISTENT or t.stages != 2:
        return None
    tiles = ceil_div(M, t.tile_M) * ceil_div(N, t.tile_N)
    capacity = PERSISTENT_CAPACITY or NUM_CUS * resident_workgroups(t, anchors)
    if tiles * batch <= capacity:
        return None
    return min(tiles, max(1, capacity // batch))


def uses_stream_k(M: int, K: int, N: int, t: TileConfig, workgroups: int | None, batch: int = 1) -> bool:
    """A persistent loop of ``workgroups`` whose tiles are not a whole
    number of rounds: the last round runs as stream-K -- when its k-chunks
    are at least as many as the workgroups, so every workgroup's range holds
    work and a split tile's contributors are the workgroups just below its
    owner (the kernel's fixup relies on that)."""
    if not STREAM_K or workgroups is None or batch != 1 or workgroups > STREAM_K_MAX_WORKGROUPS:
        return False
    rem = (ceil_div(M, t.tile_M) * ceil_div(N, t.tile_N)) % workgroups
    return rem != 0 and rem * ceil_div(K, t.tile_K) >= workgroups


def select_tile_config(
    M: int, K: int, N: int, anchors: int = 1, batch: int = 1, wide: bool = False
) -> TileConfig:
    """Highest ``tile_score``; ties go to more resident waves, then more
    workgroups.  ``batch``
    identical problems launched together (grid z) count toward filling the
    GPU.  Tiles wider than the (power-of-two rounded) output are skipped.
    ``wide`` adds the 16-wave tiles (single anchor only).
    Measured on MI355X: 256x256 for 4096^3 and the C4/C5 Q.K^T GEMMs
    (16 waves when wide, else 8); 256x128 as 16 waves (wide) or 128x128 as
    8 waves for the C5 P.V GEMM (N = 128, batched heads)."""
    return FORCE_TILE or _best_scored(M, N, anchors, batch, wide)


@functools.lru_cache(maxsize=1024)
def _best_scored(M: int, N: int, anchors: int, batch: int, wide: bool) -> TileConfig:
    pool = SINGLE_ANCHOR_TILES if anchors == 1 else DUAL_ANCHOR_TILES
    if wide and anchors == 1:
        pool = WIDE_TILES + pool
    cands = [t for t in pool if t.tile_M <= _pow2_at_least(M) and t.tile_N <= _pow2_at_least(N)]
    best = None
    best_key = None
    for i, t in enumerate(cands):
        score, wps = tile_score(t, M, N, anchors, batch)
        wgs = ceil_div(M, t.tile_M) * ceil_div(N, t.tile_N)
        key = (score, wps, wgs, -i)
        if best_key is None or key > best_key:
            best, best_key = t, key
    return best
