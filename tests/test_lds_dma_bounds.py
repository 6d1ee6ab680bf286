"""CPU replay of the direct global-to-LDS loads (ld16_to_lds, csrc/lrq_common.h).

Seven kernels move 16 bytes per lane from global memory straight into LDS with
__builtin_amdgcn_global_load_lds: k_encode_rows, k_encode_tiles and k_encode_any (csrc/lrq_encode.hip),
k_softmax_rows (csrc/lrq_rowops.hip), k_wht_rows (csrc/lrq_wht.hip), k_legacy_encode and
k_legacy_apply (csrc/lrq_legacy.hip).  This file restates, in numpy, the
host launch arithmetic (grid, row blocks per workgroup) and each kernel's source and
destination address arithmetic, and checks for every instance and launch shape that the
library's callers use (bench.py's configurations and the GPU tests' shapes) that

  * every global byte read lies inside the caller's tensor (rows clamped to the last row),
  * every LDS byte written lies inside the workgroup's allocation and inside the wave's own
    region (encode) or the block's tile (softmax, rotation),
  * no two lanes of one workgroup write the same LDS bytes for one row block.

For the kernels whose LDS is swizzled (k_encode_tiles, k_encode_any, k_legacy_encode and
k_legacy_apply) the replay also checks that every read-back finds every column where the loads put it.

No GPU is needed; a change to any of these kernels' addressing must be mirrored here.
"""

from __future__ import annotations

import numpy as np
import pytest

LDS_BYTES = 160 * 1024
CU_COUNTS = (256, 304, 80)  # MI355X, and two other counts the launch arithmetic must also survive


def _rows_per_wg(nrb: int, wgs: int) -> tuple[int, int]:
    rbw = (nrb + wgs - 1) // wgs
    return rbw, (nrb + rbw - 1) // rbw


def _blocks(grid: int, rbw: int, nrb: int):
    """Row blocks each workgroup loads: rb0 .. rb0 + nblk - 1 (the kernels return early when
    rb0 >= nrb, and their next-block loads stay below rb0 + nblk)."""
    for wg in range(grid):
        rb0 = wg * rbw
        if rb0 >= nrb:
            continue
        yield np.arange(rb0, rb0 + min(rbw, nrb - rb0))


def _check(gsrc, ldst, *, gbytes, lds_alloc, lo, hi, what):
    """gsrc / ldst: int64 arrays of the first byte each lane moves (16 bytes each)."""
    assert gsrc.min() >= 0 and (gsrc + 16).max() <= gbytes, f"{what}: global read out of the tensor"
    assert ldst.min() >= 0 and (ldst + 16).max() <= lds_alloc, f"{what}: LDS write out of the allocation"
    assert (ldst >= lo).all() and (ldst + 16 <= hi).all(), f"{what}: LDS write out of its region"


# ----------------------------------------------------------------------------- k_encode_rows
def encode_rows_replay(M, N, ldx, cus, bits=4, group=64, rank=16, upw=4, nw=8):
    """k_encode_rows<bits, group, rank, nw, upw> as launch_rows() launches it."""
    NP, RT = 8 // bits, rank // 16
    PIECE = upw * group * 2
    PITCH = NP * PIECE + 16
    REGION = 16 * PITCH
    PPL = 1024 // PIECE
    LPL = 64 // PPL
    NLD = 16 * NP // PPL
    PART = nw * RT * 64 * 16
    LDS = nw * REGION + 2 * PART
    assert LDS <= LDS_BYTES
    if PPL != NP:
        return 0  # this instance stages through registers (no direct loads)
    RPL = PPL // NP
    nrb = (M + 15) // 16
    rbw = (nrb + cus - 1) // cus
    grid = (nrb + rbw - 1) // rbw
    lane = np.arange(64)
    lpc, loff = lane // LPL, (lane % LPL) * 16
    lrow = lpc // NP
    checked = 0
    for w in range(nw):
        ub = w * upw
        xlane = ((lpc % NP) * (N // NP) + ub * group) * 2 + loff        # unit_base(p, ub) * 2 + loff
        for rbs in _blocks(grid, rbw, nrb):
            rb = rbs[:, None, None]
            i = np.arange(NLD)[None, :, None]
            r0 = rb * 16 + RPL * i
            full = r0 + RPL <= M
            row = np.where(full, r0 + lrow, np.minimum(r0 + lrow, M - 1))
            gsrc = row * ldx * 2 + xlane                                 # gaddr()
            ldst = np.broadcast_to(w * REGION + i * PITCH + lane * 16, gsrc.shape)  # region + i*PITCH, lane*16
            _check(gsrc, ldst, gbytes=((M - 1) * ldx + N) * 2, lds_alloc=LDS, lo=w * REGION,
                   hi=(w + 1) * REGION, what=f"k_encode_rows M={M} N={N} ldx={ldx} cus={cus} w={w}")
            # within one block the waves' lanes write disjoint bytes
            if w == 0 and rbs[0] == 0:
                allw = (np.arange(nw)[:, None, None] * REGION + np.arange(NLD)[None, :, None] * PITCH
                        + lane[None, None, :] * 16).ravel()
                assert np.unique(allw).size == allw.size
            checked += gsrc.size
    return checked


ENCODE_SHAPES = [  # (rows, ldx extra columns): bench north_star / c1 / lora, GPU-test shapes
    (16384, 0), (2048, 0), (1, 0), (5, 0), (16, 0), (17, 0), (37, 0), (64, 0), (96, 0), (100, 0),
    (4100, 0), (9000, 0), (100, 64), (33, 8),
]


@pytest.mark.parametrize("cus", CU_COUNTS)
def test_encode_rows_direct_loads_stay_in_bounds(cus):
    n = 0
    for rows, extra in ENCODE_SHAPES:
        n += encode_rows_replay(rows, 4096, 4096 + extra, cus)
    assert n > 0
    # the 2-unit-per-wave instance (hidden 2048) stages through registers: nothing to check
    assert encode_rows_replay(64, 2048, 2048, 256, upw=2) == 0


# ----------------------------------------------------------------------------- k_encode_tiles
def encode_tiles_replay(M, N, ldx, cus, upw=5, nw=8):
    """k_encode_tiles<upw, rot> as encode_tiles_dispatch() launches it (int4/g64: units of 128
    columns, tiles of 16 rows x 128 columns, 4 KB)."""
    NT, TILE = nw * upw, 16 * 256
    LDS = NT * TILE
    assert N == NT * 128 and LDS <= LDS_BYTES
    nrb = (M + 15) // 16
    rbw = (nrb + cus - 1) // cus
    grid = (nrb + rbw - 1) // rbw
    lane = np.arange(64)
    lr, lq = lane >> 4, lane & 15
    checked = 0
    for rbs in _blocks(grid, rbw, nrb):
        for rb in (rbs[0], rbs[-1]):
            dst_all, col_at = [], np.full(LDS // 16, -1, dtype=np.int64)  # LDS chunk -> (row, global chunk)
            for w in range(nw):
                for i in range(upw):
                    t = w + nw * i
                    for k in range(4):
                        r = 4 * k + lr
                        row = np.minimum(rb * 16 + r, M - 1)
                        gsrc = row * ldx * 2 + 256 * t + 16 * (lq ^ r)        # issue_one()
                        ldst = t * TILE + 1024 * k + 16 * lane
                        _check(gsrc, ldst, gbytes=((M - 1) * ldx + N) * 2, lds_alloc=LDS, lo=t * TILE,
                               hi=(t + 1) * TILE, what=f"k_encode_tiles M={M} N={N} ldx={ldx} cus={cus} w={w}")
                        assert ((gsrc % (ldx * 2)) // 256 == t).all(), "a tile holds columns of another tile"
                        dst_all.append(ldst)
                        col_at[ldst // 16] = r * 1000 + (gsrc % (ldx * 2)) // 16
                        checked += gsrc.size
            d = np.concatenate(dst_all)
            assert np.unique(d).size == d.size == LDS // 16, "every LDS chunk written exactly once per block"
            # read-back: lane (j, g) of wave w reads unit u = w*upw + uu, plane p, chunk
            # 8(u%2) + 2g + k of tile p*NT/2 + u/2, row j, at position chunk ^ j
            j, g = lane & 15, lane >> 4
            for w in range(nw):
                for uu in range(upw):
                    u = w * upw + uu
                    for p in range(2):
                        tp = p * (NT // 2) + u // 2
                        for k in range(2):
                            c = 8 * (u % 2) + 2 * g + k
                            pos = (tp * TILE + 256 * j + 16 * (c ^ j)) // 16
                            want_col = (p * (N // 2) + 64 * u + 16 * g + 8 * k)   # unit_base(p, u) + 16g + 8k
                            assert (col_at[pos] == j * 1000 + want_col // 8).all(), "read-back finds other columns"
                # the rotation's layout: lane (j, g) chunks 4g + c of its tiles' row j
                for i in range(upw):
                    t = w + nw * i
                    for c in range(4):
                        pos = (t * TILE + 256 * j + 16 * ((4 * g + c) ^ j)) // 16
                        assert (col_at[pos] == j * 1000 + (128 * t) // 8 + 4 * g + c).all()
    return checked


@pytest.mark.parametrize("cus", CU_COUNTS)
def test_encode_tiles_direct_loads_stay_in_bounds(cus):
    n = 0
    for rows, extra in [(16384, 0), (1, 0), (5, 0), (16, 0), (37, 0), (48, 0), (64, 0), (100, 0), (4100, 0),
                        (5000, 0), (64, 64), (33, 8)]:
        n += encode_tiles_replay(rows, 5120, 5120 + extra, cus)
    assert n > 0


# ----------------------------------------------------------------------------- k_softmax_rows
def softmax_rows_replay(M, N, lddp, cus, bits, group):
    """k_softmax_rows<bits, group, rank, NW> as softmax_units() / softmax_rows_launch() launch it."""
    NP = 8 // bits
    units = N // (group * NP)
    UB = group * NP * 2
    if units not in (8, 16) or (units * UB) % 1024:
        return 0
    NW = units
    ROWB = NW * group * NP * 2
    PITCH = ROWB + 16
    TILE = 16 * PITCH
    CPR = ROWB // 1024
    DPW = 16 * CPR // NW
    LDS = 2 * TILE + NW * 16 * 4
    if LDS > LDS_BYTES:
        return 0  # softmax_units() has no instance for this width (its compile-time LDS check)
    assert (16 * CPR) % NW == 0
    nrb = (M + 15) // 16
    per_cu = max(1, min(4, LDS_BYTES // LDS))
    wgs = max(1, min(nrb, cus * per_cu))
    rbw, grid = _rows_per_wg(nrb, wgs)
    lane = np.arange(64)
    checked = 0
    for rbs in _blocks(grid, rbw, nrb):
        for tb in (0, 1):
            dsts = []
            for w in range(NW):
                q = w * DPW + np.arange(DPW)[:, None]
                r, c = q // CPR, q % CPR
                row = np.minimum(rbs[:, None, None] * 16 + r[None], M - 1)
                gsrc = row * lddp * 2 + c[None] * 1024 + lane * 16
                ldst = np.broadcast_to(tb * TILE + r * PITCH + c * 1024 + lane * 16, (DPW, 64))
                _check(gsrc, ldst, gbytes=((M - 1) * lddp + N) * 2, lds_alloc=LDS, lo=tb * TILE,
                       hi=tb * TILE + TILE, what=f"k_softmax_rows M={M} N={N} bits={bits} w={w}")
                # a row's chunks stay inside the row's ROWB bytes of the tile
                assert ((ldst - tb * TILE) % PITCH + 16 <= ROWB).all()
                dsts.append(ldst.ravel())
                checked += gsrc.size
            d = np.concatenate(dsts)
            assert np.unique(d).size == d.size
    return checked


@pytest.mark.parametrize("cus", CU_COUNTS)
@pytest.mark.parametrize("bits,group,N", [(4, 64, 2048), (4, 64, 1024), (8, 128, 2048), (8, 128, 1024),
                                          (8, 64, 1024), (4, 128, 4096)])
def test_softmax_rows_direct_loads_stay_in_bounds(cus, bits, group, N):
    n = 0
    for rows in (1, 16, 40, 64, 100, 9000):
        n += softmax_rows_replay(rows, N, N, cus, bits, group)
    if (bits, group, N) == (4, 64, 2048):
        n += softmax_rows_replay(2 * 32 * 2048, N, N, cus, bits, group)  # config 5
    assert (n > 0) == ((bits, group, N) != (4, 128, 4096))  # 16 units of 512 B rows: no tile fits


# ----------------------------------------------------------------------------- k_wht_rows
def wht_rows_replay(M, N, ldx, cus):
    """k_wht_rows as lrq_wht128 launches it (hidden % 512 == 0)."""
    PITCH = 1024 + 16
    TILE = 16 * PITCH
    LDS = 2 * TILE
    nrb = (M + 15) // 16
    slabs = N // 512
    ranges = max(1, min(nrb, cus * 4 // slabs))
    rbw = (nrb + ranges - 1) // ranges
    grid = (nrb + rbw - 1) // rbw
    lane = np.arange(64)
    checked = 0
    for by in range(slabs):
        c0 = by * 512
        for rbs in _blocks(grid, rbw, nrb):
            for tb in (0, 1):
                dsts = []
                for w in range(4):
                    r = 4 * w + np.arange(4)[:, None]
                    row = np.minimum(rbs[:, None, None] * 16 + r[None], M - 1)
                    gsrc = c0 * 2 + row * ldx * 2 + lane * 16
                    ldst = np.broadcast_to(tb * TILE + r * PITCH + lane * 16, (4, 64))
                    _check(gsrc, ldst, gbytes=((M - 1) * ldx + N) * 2, lds_alloc=LDS, lo=tb * TILE,
                           hi=tb * TILE + TILE, what=f"k_wht_rows M={M} N={N} slab={by} w={w}")
                    dsts.append(ldst.ravel())
                    checked += gsrc.size
                d = np.concatenate(dsts)
                assert np.unique(d).size == d.size
    return checked


@pytest.mark.parametrize("cus", CU_COUNTS)
def test_wht_rows_direct_loads_stay_in_bounds(cus):
    n = 0
    for rows, N, extra in [(16384, 5120, 0), (20000, 512, 0), (64, 1024, 0), (33, 2048, 0), (100, 4096, 8),
                           (1, 512, 0), (5000, 5120, 0)]:
        n += wht_rows_replay(rows, N, N + extra, cus)
    assert n > 0


# ----------------------------------------------------------------------------- k_encode_any
def encode_any_replay(M, N, ldx, cus, bits, rank):
    """k_encode_any as encode_any_dispatch() launches it: X's and V^T's tiles, and the read-back of every
    unit's columns and of every projection step's operands (which cover the columns in the chains of the
    two-pass encode)."""
    TILE, NP, U, NW = 4096, 8 // bits, N // 128, 8
    even, upw, RT = U % 2 == 0, (U + 7) // 8, max(1, rank // 16)
    nch = 0 if rank == 0 else U // 2 if even else 4
    QR = 8 if (upw == 3 if rank == 16 else rank == 32 and upw == 2) else 0
    vlds = rank > 0 and (upw <= 2 or (rank == 16 and upw == 3))
    t0 = 0 if QR == 0 else 16 if even else QR
    nv = max(0, U - t0) * RT if vlds else 0
    vbase = U * TILE + nch * RT * 1024
    alloc = vbase + nv * TILE
    assert alloc <= LDS_BYTES and nv >= 0
    nrb = (M + 15) // 16
    rbw, grid = _rows_per_wg(nrb, cus * (2 if upw == 1 and rank <= 16 else 1))
    lane = np.arange(64)
    lr, lq, j, g = lane >> 4, lane & 15, lane & 15, lane >> 4
    checked = 0
    # V^T tiles: chunk held at each (tile, rank row, position)
    vheld = np.full((max(nv, 1), 16, 16), -1, dtype=np.int64)
    for v in range(nv):
        for k in range(4):
            r = 4 * k + lr
            src = (v % RT) * 16 * N * 2 + 256 * (t0 + v // RT) + (r * N + 8 * (lq ^ r)) * 2
            dst = vbase + v * TILE + 1024 * k + 16 * lane
            _check(src, dst, gbytes=rank * N * 2, lds_alloc=alloc, lo=vbase + v * TILE, hi=vbase + (v + 1) * TILE,
                   what=f"k_encode_any V^T {N} rank {rank}")
            vheld[v, r, lq] = src % (2 * N) // 16  # 16-byte chunk of the V^T row
    # the projection: wave w's steps in order; the chains cover every 32 columns once, as the two passes do
    chains = {}
    for w in range(NW):
        nq = 0 if w >= nch else (nch - w + NW - 1) // NW * 8 if even else U
        for q in range(nq):
            col = 256 * (w + NW * (q >> 3)) + 32 * (q & 7) if even else 32 * w + 128 * q
            chains.setdefault(w + 8 * (q >> 3) if even else w, []).append(col)
            c = col >> 5
            if vlds and q >= QR:
                for t in range(RT):
                    v = ((c >> 2) - t0) * RT + t
                    assert (vheld[v, j, (4 * (c & 3) + g) ^ j] == (col + 8 * g) // 8).all()
    if rank:
        want = {c: [256 * c + 32 * k for k in range(8)] for c in range(U // 2)} if even else \
            {c: [32 * k for k in range(c, 4 * U, 4)] for c in range(4)}
        assert chains == want
    for rbs in _blocks(grid, rbw, nrb):
        for rb in rbs:
            lim = M - 1 - rb * 16
            held = np.full((U, 16, 16), -1, dtype=np.int64)  # (tile, row, position) -> chunk of the row
            dsts = []
            for t in range(U):
                for k in range(4):
                    r = 4 * k + lr
                    gsrc = (rb * 16 * ldx) * 2 + 256 * t + np.minimum(r, lim) * ldx * 2 + 16 * (lq ^ r)
                    ldst = t * TILE + 1024 * k + 16 * lane
                    _check(gsrc, ldst, gbytes=((M - 1) * ldx + N) * 2, lds_alloc=alloc, lo=t * TILE, hi=(t + 1) * TILE,
                           what=f"k_encode_any {M}x{N}")
                    dsts.append(ldst)
                    checked += 64
                    held[t, r, lq] = (gsrc - np.minimum(rb * 16 + r, M - 1) * ldx * 2) // 16
            d = np.concatenate(dsts)
            assert np.unique(d).size == d.size
            for u in range(U):
                for p in range(NP):
                    c = p * U + u if NP == 2 else 2 * u
                    for k in range(4 // NP):
                        chunk = 8 * (c & 1) + (4 // NP) * g + k
                        want = p * (N // NP) + u * (128 // NP) + (32 // NP) * g + 8 * k
                        assert (held[c // 2, j, chunk ^ j] == want // 8).all()
            for c in range(4 * U if rank else 0):  # a projection step's 32 columns
                assert (held[c >> 2, j, (4 * (c & 3) + g) ^ j] == (32 * c + 8 * g) // 8).all()
    return checked


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("cus", CU_COUNTS)
def test_encode_any_direct_loads_stay_in_bounds(cus, bits):
    n = 0
    for M, N, extra, rank in [(1, 128, 0, 16), (33, 896, 8, 16), (40, 1152, 0, 32), (33, 1024, 0, 32), (40, 2048, 0, 32),
                              (40, 1920, 0, 32), (100, 3072, 0, 16), (20, 2944, 0, 16), (33, 2048, 0, 16), (47, 3584, 0, 16),
                              (47, 4736, 0, 16), (50, 4992, 0, 0)]:
        n += encode_any_replay(M, N, N + extra, cus, bits, rank)
    assert n > 0


# ----------------------------------------------------------------------------- k_legacy_encode
def _legacy_run_blocks(groups, nrb, cus):
    """legacy_run_blocks(): row blocks per run."""
    best, least = 1, None
    for r in range(1, 17):
        per_cu = -(-groups * -(-nrb // r) // cus)
        if r > 1 and per_cu < (3 if groups * nrb >= 24 * cus else 2):
            break
        if least is None or per_cu * (4 * r + 3) < least:
            best, least = r, per_cu * (4 * r + 3)
    return best


def legacy_ring_replay(B, M, N, ldx_m, ldx_b, cus, bits, WAVE, what):
    """k_legacy_encode (its x) and k_legacy_apply (its y) as legacy_launch() launches them, WAVE bytes of
    LDS per wave with the ring first: every request of every wave, and the read-back of every slot (lane
    (j, g): columns 16g .. 16g + 15 of row j) from what the slot holds at that step."""
    NP = 8 // bits
    NB = N // NP
    RING, SLOT = 4, 16 * 128
    nrb, nu = (M + 15) // 16, NB // 64
    ug = (nu + 3) // 4
    rbw = _legacy_run_blocks(B * ug, nrb, cus)
    nrun = (nrb + rbw - 1) // rbw
    lane = np.arange(64)
    j, g = lane & 15, lane >> 4
    checked = 0
    assert 4 * WAVE <= LDS_BYTES
    for t in range(nrun * ug * B):
        run, b = (t // ug) % nrun, t // (ug * nrun)
        rb0 = run * rbw
        nblk = min(rbw, nrb - rb0)
        assert nblk >= 1
        for w in range(4):
            u = (t % ug) * 4 + w
            if u * 64 >= NB:
                continue
            steps = [(min(st // NP, nblk - 1), st % NP, st) for st in range(RING)]
            steps += [(min(i + (p + RING) // NP, nblk - 1), (p + RING) % NP, (i * NP + p) % RING)
                      for i in range(nblk) for p in range(NP)]
            held = {}  # slot -> (block, plane, first column, chunk held at each position of each row)

            def read_back(i, p, slot):
                hi, hp, col0, col = held[slot]
                assert (hi, hp) == (i, p) and col0 == u * 64 + p * NB, "the slot holds another step"
                for h in range(2):
                    assert (col[j, (2 * g + h) ^ (j & 7)] == 2 * g + h).all()

            for n, (i, p, slot) in enumerate(steps):
                if n >= RING:  # (each step reads its slot, then requests it again)
                    read_back((n - RING) // NP, (n - RING) % NP, slot)
                col = np.empty((16, 8), dtype=np.int64)  # chunk held at each position of each row
                for k in range(2):
                    r = 8 * k + lane // 8
                    row = np.minimum((rb0 + i) * 16 + r, M - 1)
                    c = u * 64 + 8 * ((lane & 7) ^ (lane >> 3)) + p * NB
                    gsrc = (b * ldx_b + row * ldx_m + c) * 2
                    assert (gsrc % 16 == 0).all()
                    ldst = w * WAVE + slot * SLOT + 1024 * k + 16 * lane
                    _check(gsrc, ldst, gbytes=((B - 1) * ldx_b + (M - 1) * ldx_m + N) * 2, lds_alloc=4 * WAVE,
                           lo=w * WAVE + slot * SLOT, hi=w * WAVE + (slot + 1) * SLOT, what=f"{what} {M}x{N} {bits}")
                    col[r, lane & 7] = (c - u * 64 - p * NB) // 8
                    checked += 64
                held[slot] = (i, p, u * 64 + p * NB, col)
    return checked


# (batches, rows, columns, row padding): one row, ragged blocks, unit counts that are no multiple of four,
# several blocks per run
RING_SHAPES = [(1, 1, 512, 0), (2, 100, 1024, 8), (1, 40, 1536, 0), (3, 37, 2048, 0), (1, 2100, 512, 0), (2, 5003, 512, 8)]


@pytest.mark.parametrize("bits", [1, 2, 4, 8])
@pytest.mark.parametrize("cus", CU_COUNTS)
def test_legacy_encode_direct_loads_stay_in_bounds(cus, bits):
    n = 0
    NP = 8 // bits
    for B, M, N, extra in RING_SHAPES:
        for K in (16, 32) if bits == 1 else (16,):  # (the rank changes the layout at 1 bit only)
            wave = 4 * 2048 + NP * 64 * 4 + 16 * NP * 8 + (2 * 4 * 64 * 16 if bits == 1 and K == 32 else 0)
            n += legacy_ring_replay(B, M, N, N + extra, M * (N + extra), cus, bits, wave, "k_legacy_encode")
    assert n > 0


@pytest.mark.parametrize("bits", [1, 2, 4, 8])
@pytest.mark.parametrize("cus", CU_COUNTS)
def test_legacy_apply_direct_loads_stay_in_bounds(cus, bits):
    """The consumers' y (contiguous rows and batches) through the ring; behind it the scale table and the
    result tile."""
    n = 0
    for B, M, N, _ in RING_SHAPES:
        n += legacy_ring_replay(B, M, N, N, M * N, cus, bits, 4 * 2048 + 8 // bits * 64 * 4 + 2048, "k_legacy_apply")
    assert n > 0


@pytest.mark.parametrize("B,M,N,bits", [(4, 3072, 3072, 1), (4, 3072, 3072, 2), (4, 3072, 3072, 4), (4, 3072, 3072, 8),
                                        (2, 5253, 2560, 1), (2, 5253, 2560, 8), (4, 1024, 1024, 8), (4, 8192, 8192, 1)])
def test_legacy_runs_spread_over_the_cus(B, M, N, bits):
    """The run length of k_legacy_encode and k_legacy_apply leaves the busiest of 256 CUs at most half more
    than the mean number of row blocks, a run's set-up counted as 3/4 of one (lengths from the mean alone
    came to 1.75 times)."""
    groups, nrb = B * ((N * bits // 8 // 64 + 3) // 4), (M + 15) // 16
    r = _legacy_run_blocks(groups, nrb, 256)
    busiest = -(-groups * -(-nrb // r) // 256) * (r + 0.75)
    assert 1 <= r <= 16 and busiest <= 1.5 * groups * nrb / 256


def test_replay_catches_a_planted_overrun():
    """The check is live: a replay whose row clamp is dropped (rows past the end read) fails."""
    M, N = 37, 4096
    nrb = (M + 15) // 16
    row = np.arange(nrb * 16)  # no clamp
    gsrc = row * N * 2
    with pytest.raises(AssertionError):
        _check(gsrc, np.zeros_like(gsrc), gbytes=((M - 1) * N + N) * 2, lds_alloc=LDS_BYTES, lo=0, hi=LDS_BYTES,
               what="planted")
