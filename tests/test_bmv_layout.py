"""CPU model of the batched mat-vec on the int8 matrix cores
(qwen3-4b-q4_k_m-inference-engine_amd/csrc/bmv.hip, bmv.hpp), M = 2..8.

For each shape the model restates the launcher's plan (workgroups per
matrix, superblock runs per row group, LDS size with the slots, which launches
are made at all) and the kernel's cursors, then checks every global load of
every lane of every wave of every workgroup (inside its superblock and its
matrix, including the ring's refills past a wave's last tile; Q6_K in mode 0:
the chunks of a tile's rows, up to the zeros past the descriptor's end), every
LDS read and write against its region, and that each (part, row, superblock)
is computed by exactly one tile and each unit's sums slot written once. A lane-level emulation of the arithmetic (the block-
diagonal A tiles as the lanes read them from the LDS image, the B operands as
the lanes build them, v_mfma_i32_16x16x64_i8 as an integer product with the
probed lane layout: lane l holds A[l%16][16(l/16)+t], B[16(l/16)+t][l%16] and
receives C[4(l/16)+i][l%16]) is compared with the oracle's product, with
garbage planted in the LDS rows the kernel leaves unwritten. The model is its
own code restating the kernel's integer arithmetic; a change to either file
must be mirrored here."""
import numpy as np
import pytest

CUS, MAX_LDS, WAVES = 256, 160 * 1024, 16
BYTES = {12: 144, 14: 210}
P = {12: 2, 14: 1}
SLOT_CHUNKS, SLOT_LOADS = 14, 3
SLOT_ROWS = 64 * SLOT_LOADS // SLOT_CHUNKS


def sums_end(K, stride, parts, groups, ranges):
    return 8 * stride + 16 + 4 * K + parts * groups * 16 * ranges * 32


def slot_bytes(rows):
    return 16 * SLOT_CHUNKS * rows


def wave_tiles(rows, parts, S, ranges):
    if rows <= 0:
        return 0
    groups = -(-rows // 16)
    units = parts * groups * ranges
    return -(-units // WAVES) * -(-S // ranges)


def counts(rows, types, mode):
    """Workgroups of each matrix, or None past the CUs."""
    if mode == 1 or len(rows) == 1:
        return [min(CUS, rows[0])]
    for groups in (1, 2):
        need = [-(-r // (SLOT_ROWS if t == 14 else 16 * groups)) for r, t in zip(rows, types)]
        if sum(need) <= CUS:
            byt = [r * BYTES[t] for r, t in zip(rows, types)]
            left = CUS - sum(need)
            return [min(r, c + int(left * x / sum(byt))) for r, c, x in zip(rows, need, byt)]
    return None


def fits(rows, types, K, mode):
    """bmv_plan: (workgroups per matrix, ranges, groups_max, lds, rows of a
    slot, tiles on the busiest wave, the same with any LDS), or None."""
    nseg = 1 if mode == 1 else len(rows)
    parts = 2 if mode == 1 else 1
    S, stride = K // 256, K + 16
    count = counts(rows, types, mode)
    if count is None:
        return None
    most = [-(-rows[j] // count[j]) for j in range(nseg)]
    slot_rows = max([most[j] for j in range(nseg) if mode == 0 and types[j] == 14], default=0)
    if slot_rows > SLOT_ROWS:
        return None
    groups_max = max(-(-m // 16) for m in most)
    best, all_tiles = None, None
    for r in range(1, S + 1):
        lds = sums_end(K, stride, parts, groups_max, r) + WAVES * slot_bytes(slot_rows)
        if lds > MAX_LDS and best is None:
            return None
        tiles = max(wave_tiles(m, parts, S, r) for m in most)
        units = max(-(-(parts * -(-m // 16) * r) // WAVES) for m in most)
        all_tiles = tiles if all_tiles is None else min(all_tiles, tiles)
        if lds <= MAX_LDS and (best is None or 8 * tiles + units < best[0]):
            best = (8 * tiles + units, r, lds, tiles)
    return count, best[1], groups_max, best[2], slot_rows, best[3], all_tiles


def pays(rows, types, K, M):
    """bmv_pays: the lines of mode 0."""
    total, S, q4, q6 = sum(rows), K // 256, 12 in types, 14 in types
    if len(rows) == 1:
        if q4:
            return M >= 3 or K <= 8192
        if M < 3:
            return False
        if M <= 4:
            return K <= 8192 or total > 8 * CUS
        return M <= 6 or total > 3 * CUS or (M == 7 and K > 8192)
    if S < 9 or M >= 5:
        return S >= 9
    if S % 8 == 0 and ((q4 and q6) or total > (24 if K <= 4096 else 20) * CUS):
        return False
    if not q6:
        return M >= 3 or K <= (6400 if total > 16 * CUS else 8192)
    if q4:
        return M >= 3 and total > (16 if K < 3328 else 8) * CUS
    return M >= 3 and (K <= 8192 or total > 8 * CUS)


def plan(rows, types, K, mode, M):
    """The launch's plan, or None when the launcher declines."""
    if not 2 <= M <= 8 or mode not in (0, 1):
        return None
    if mode == 0 and not pays(rows, types, K, M):
        return None
    cfg = fits(rows, types, K, mode)
    if cfg is None or mode == 1:
        return cfg
    if (len(rows) == 1 and cfg[2] > 1) or cfg[5] > (1 if M <= 4 else 2) * cfg[6]:
        return None
    return cfg


class Share:
    def __init__(self, r0, nrows, S, ranges, parts):
        self.r0, self.nrows, self.S, self.ranges, self.parts = r0, nrows, S, ranges, parts
        self.groups = (nrows + 15) >> 4
        self.run_q, self.run_r = S // ranges, S % ranges

    def run_begin(self, rr):
        return rr * self.run_q + min(rr, self.run_r)


class Cursor:
    def __init__(self, sh, u, left):
        self.sh = sh
        self.rr = u % sh.ranges
        pg = u // sh.ranges
        self.part = pg // sh.groups
        self.g = pg - self.part * sh.groups
        self.s, self.s_end = sh.run_begin(self.rr), sh.run_begin(self.rr + 1)
        self.left = left

    def copy(self):
        c = Cursor.__new__(Cursor)
        c.__dict__.update(self.__dict__)
        return c

    def next(self):
        sh = self.sh
        if self.left > 1:
            self.left -= 1
            self.s += 1
            if self.s == self.s_end:
                self.rr += 1
                if self.rr == sh.ranges:
                    self.rr = 0
                    self.g += 1
                    if self.g == sh.groups:
                        self.g = 0
                        self.part += 1
                self.s, self.s_end = sh.run_begin(self.rr), sh.run_begin(self.rr + 1)


def wave_streams(sh, wave, depth):
    """(compute tiles, load tiles) of a wave: tiles as (part, g, rr, s, last_of_unit)."""
    units = sh.parts * sh.groups * sh.ranges
    u_lo, u_hi = units * wave // WAVES, units * (wave + 1) // WAVES
    ntiles = sum(sh.run_begin(u % sh.ranges + 1) - sh.run_begin(u % sh.ranges) for u in range(u_lo, u_hi))
    start = Cursor(sh, u_lo if u_lo < u_hi else 0, ntiles)
    lc, cc = start.copy(), start.copy()
    loads, comps = [], []
    for _ in range(depth):
        loads.append((lc.part, lc.g, lc.rr, lc.s))
        lc.next()
    for base in range(0, ntiles, depth):
        for j in range(depth):
            if base + j < ntiles:
                comps.append((cc.part, cc.g, cc.rr, cc.s, cc.s + 1 == cc.s_end))
                cc.next()
            loads.append((lc.part, lc.g, lc.rr, lc.s))
            lc.next()
    return comps, loads


LANE = np.arange(64)
LN, LKQ = LANE & 15, LANE >> 4


def load_ranges(qtype, sb):
    """Byte ranges [a, b) each lane reads of its superblock at offset sb (array per lane)."""
    kq = LKQ
    if qtype == 12:
        return [(sb, sb + 16), (sb + 16 + 16 * kq, sb + 32 + 16 * kq), (sb + 80 + 16 * kq, sb + 96 + 16 * kq)]
    return [(sb + 16 * kq, sb + 16 + 16 * kq), (sb + 64 + 16 * kq, sb + 80 + 16 * kq),
            (sb + 128 + 16 * (kq & 1), sb + 144 + 16 * (kq & 1)),
            (sb + 160 + 16 * (kq & 1), sb + 176 + 16 * (kq & 1)), (sb + 192, sb + 208), (sb + 208, sb + 210)]


def workgroups(rows, types, K, mode, cfg):
    count, ranges = cfg[:2]
    nseg = 1 if mode == 1 else len(rows)
    parts = 2 if mode == 1 else 1
    for j in range(nseg):
        per, rem = rows[j] // count[j], rows[j] % count[j]
        for g in range(count[j]):
            yield j, Share(g * per + min(g, rem), per + (1 if g < rem else 0), K // 256, ranges, parts)


def check_indices(rows, types, K, mode, M, bases):
    """Workgroups of one segment with the same row count differ only by their
    first row, so beyond 32 workgroups the first of each row count and the
    last are checked lane by lane; the shares' partition of the rows is
    checked for all of them."""
    cfg = plan(rows, types, K, mode, M)
    assert cfg is not None
    count, ranges, groups_max, lds, slot_rows = cfg[:5]
    S, stride = K // 256, K + 16
    Z = 8 * stride + 16
    parts = 2 if mode == 1 else 1
    nseg = 1 if mode == 1 else len(rows)
    end = sums_end(K, stride, parts, groups_max, ranges)  # the slots of the waves follow
    assert end + WAVES * slot_bytes(slot_rows) == lds <= MAX_LDS and sum(count[:nseg]) <= CUS
    chosen = set()
    for j in range(nseg):
        per, rem = rows[j] // count[j], rows[j] % count[j]
        shares = [(g * per + min(g, rem), per + (1 if g < rem else 0)) for g in range(count[j])]
        assert shares[0][0] == 0 and shares[-1][0] + shares[-1][1] == rows[j]
        assert all(a + n == b for (a, n), (b, _) in zip(shares, shares[1:])), "shares partition the rows"
        assert all(1 <= n <= 16 * groups_max for _, n in shares)
        if count[j] <= 32:
            chosen |= {(j, r0) for r0, _ in shares}
        else:
            chosen |= {(j, shares[0][0]), (j, shares[rem - 1][0] if rem else 0), (j, shares[rem][0] if rem < count[j] else 0),
                       (j, shares[-1][0])}
    seen = {}
    for j, sh in workgroups(rows, types, K, mode, cfg):
        if (j, sh.r0) not in chosen:
            continue
        qtype = types[j]
        B = BYTES[qtype]
        rb = S * B
        through_slots = qtype == 14 and mode == 0
        slots = {}
        for wave in range(WAVES):
            comps, loads = wave_streams(sh, wave, P[qtype])
            if through_slots:
                assert sh.nrows <= slot_rows <= SLOT_ROWS and sh.groups == 1
                chunks = SLOT_CHUNKS * sh.nrows
                end4 = (rows[j] * rb + 3) & ~3
                c = np.minimum(LANE[:, None] + 64 * np.arange(SLOT_LOADS), chunks - 1)
                assert set(c.ravel()) == set(range(chunks))  # every chunk of the tile is loaded
                at = end + wave * slot_bytes(slot_rows) + 16 * c
                assert np.all(at % 16 == 0) and np.all(at + 16 <= end + (wave + 1) * slot_bytes(slot_rows))
                for s in {load[3] for load in loads}:
                    first = (sh.r0 + np.arange(sh.nrows)) * rb + s * B
                    off = ((first & ~3)[:, None] + 16 * np.arange(SLOT_CHUNKS))[c // SLOT_CHUNKS, c % SLOT_CHUNKS]
                    assert np.all(off >= 0) and np.all(off + 16 <= end4 + 16) and np.all(off % 4 == 0)
                    # the superblock's bytes lie in its row's chunks, the 54 dwords read in its part of the slot
                    assert np.all((first & 3) + B <= 16 * SLOT_CHUNKS) and 4 * 54 <= 16 * SLOT_CHUNKS
                    assert np.all(first + B <= rows[j] * rb)
                loads = []
            for part, g, rr, s in loads:
                w = bases[1] if (mode == 1 and part) else bases[j]
                n_mat = rows[1] if (mode == 1 and part) else rows[j]
                row = np.minimum(16 * g + LN, sh.nrows - 1)
                sb = w + (sh.r0 + row) * rb + s * B
                for a, b in load_ranges(qtype, sb):
                    assert np.all(a >= sb) and np.all(b <= sb + B), "read outside the superblock"
                    assert np.all(a >= w) and np.all(b <= w + n_mat * rb), "read outside the matrix"
                    if qtype == 12 and (b - a)[0] == 16:
                        assert np.all(a % 16 == 0), "Q4_K loads are 16-byte aligned"
            for part, g, rr, s, last in comps:
                for rw in range(16 * g, min(16 * g + 16, sh.nrows)):
                    key = (j, part, sh.r0 + rw, s)
                    assert key not in seen, "tile computed twice"
                    seen[key] = True
                # LDS reads of the tile
                khi, klo = LKQ >> 1, LKQ & 1
                if qtype == 12:
                    valid = (LN < 8) == (LKQ < 2)
                    base = (LN & 7) * stride + 16 * klo
                    for h in range(2):
                        for nib in range(2):
                            jj = 4 * h + nib + 2 * khi
                            aoff = np.where(valid, base + 256 * s + 32 * jj, 8 * stride)
                            assert np.all(aoff + 16 <= 8 * stride + 16) and np.all(aoff % 16 == 0)
                            assert np.all(np.where(valid, aoff + 16 <= 8 * stride, True))
                            for reg in (0, K):  # xs, xss
                                off = Z + reg + 4 * ((8 * s + jj) * 8 + 4 * klo)
                                assert np.all(off >= Z + reg) and np.all(off + 16 <= Z + reg + K)
                else:
                    for h in range(2):
                        for nib in range(2):
                            blk = 4 * h + 2 * nib + khi
                            for p in range(2 if M > 4 else 1):
                                if M > 4:  # two products of the same Q8 block
                                    valid = ((LN >> 3) == khi) & (klo == p)
                                    base, m0, sb16 = (LN & 7) * stride + 16 * LKQ, 4 * klo, 2 * blk + p
                                else:
                                    valid = (LN >> 2) == LKQ
                                    base, m0, sb16 = (LN & 3) * stride + 16 * LKQ, 0, 8 * h + 4 * nib + LKQ
                                aoff = np.where(valid, base + 256 * s + 128 * h + 64 * nib, 8 * stride)
                                assert np.all(aoff % 16 == 0) and np.all(aoff + 16 <= 8 * stride + 16)
                                assert np.all(np.where(valid, aoff + 16 <= 8 * stride, True))
                                off = Z + 4 * ((8 * s + blk) * 8 + m0)
                                assert np.all(off + 16 <= Z + K)
                                off = Z + 2 * K + 4 * ((16 * s + sb16) * 8 + m0)
                                assert np.all(off >= Z + 2 * K) and np.all(off + 16 <= Z + 4 * K)
                if last:
                    assert (part, g, rr) not in slots, "unit flushed twice"
                    slots[(part, g, rr)] = True
                    slot = ((part * groups_max + g) * 16 + LN) * ranges + rr
                    off = Z + 4 * K + 4 * (slot * 8)
                    assert np.all(off + 32 <= end)
        assert len(slots) == parts * sh.groups * ranges, "every unit flushed"
        # totals read every run of every valid row
        for part in range(parts):
            for rw in range(sh.nrows):
                for rr in range(ranges):
                    off = Z + 4 * K + 4 * ((((part * groups_max) * 16 + rw) * ranges + rr) * 8 + 7)
                    assert off + 4 <= end
    for j, sh in workgroups(rows, types, K, mode, cfg):
        if (j, sh.r0) in chosen:
            for part in range(parts):
                for rw in range(sh.r0, sh.r0 + sh.nrows):
                    for s in range(S):
                        assert (j, part, rw, s) in seen, "tile never computed"
    return cfg


SHAPES = [  # rows, types, K, mode, M
    ([4096, 1024, 1024], [12, 12, 14], 2560, 0, 8),   # attn q/k/v
    ([4096, 1024, 1024], [12, 12, 14], 2560, 0, 3),
    ([4096, 1024, 1024], [12, 12, 12], 2560, 0, 2),
    ([9728, 9728], [12, 12], 2560, 1, 8),               # ffn gate/up
    ([9728, 9728], [12, 12], 2560, 1, 5),
    ([9728, 9728], [14, 14], 2560, 1, 6),
    ([9728, 9728], [14, 14], 2560, 1, 3),
    ([300, 300], [12, 12], 512, 1, 2),
    ([2560], [14], 9728, 0, 8),                         # ffn_down
    ([2560], [14], 9728, 0, 4),
    ([2560], [12], 9728, 0, 8),
    ([4096], [12], 11008, 0, 3),
    ([4096], [12], 8192, 0, 2),                         # 16 rows on every CU
    ([17], [12], 256, 0, 5),
    ([3328], [14], 8192, 0, 8),                         # 13 rows of Q6_K on every CU
    ([2560], [14], 10240, 0, 5),                        # LDS bounds the runs
    ([19], [14], 9728, 0, 7),
    ([45], [14], 768, 0, 3),
    ([101], [14], 1280, 0, 5),
    ([300, 17], [14, 12], 2304, 0, 8),
    ([1700, 33, 1560, 17], [14, 12, 14, 12], 2560, 0, 5),  # 256 workgroups
    ([8160, 32], [12, 12], 2560, 0, 4),
    ([700, 700], [14, 14], 4352, 0, 3),
]


@pytest.mark.parametrize("rows,types,K,mode,M", SHAPES)
def test_bmv_indices_in_bounds(rows, types, K, mode, M):
    bases = [(1 << 30) * (i + 1) + (4 if t == 14 else 0) for i, t in enumerate(types)]
    check_indices(rows, types, K, mode, M, bases)


def test_bmv_plan_for_qwen3_shapes():
    """LDS plans of the decode batch's launches (one workgroup per CU)."""
    down = plan([2560], [14], 9728, 0, 8)                         # 8 x 9728 codes + scales + slots
    assert down[:3] == ([256], 13, 1) and down[3:] == (159376, 10, 3, 3)
    assert plan([9728, 9728], [12, 12], 2560, 1, 8)[0] == [256]
    qkv = plan([4096, 1024, 1024], [12, 12, 14], 2560, 0, 8)
    assert sum(qkv[0]) <= 256 and qkv[2] == 2 and qkv[4] <= SLOT_ROWS
    assert plan([2560], [12], 4096, 0, 1) is None                 # M = 1: the whole-share kernels
    assert plan([2560], [12], 4096, 0, 9) is None                 # M > 8: the prefill GEMM


@pytest.mark.parametrize("rows,types,K,M", [
    ([151936], [14], 2560, 8), ([4097], [12], 9728, 5), ([3329], [14], 9728, 8),       # more rows than a group or slot
    ([8160, 33], [12, 12], 2560, 4), ([1700, 33, 1700, 17], [14, 12, 14, 12], 2560, 5),  # past the CUs
    ([1024], [14], 12288, 8), ([2560], [14], 10240, 4), ([300], [12], 13568, 3),         # LDS holds too few runs
    ([2560], [14], 9728, 2), ([1024], [14], 9728, 4), ([4096, 1024, 1024], [12, 12, 12], 2048, 8),
])
def test_bmv_plan_declines(rows, types, K, M):
    assert plan(rows, types, K, 0, M) is None


# ---------------------------------------------------------------- arithmetic

def _u32(b):
    return np.frombuffer(np.ascontiguousarray(b, dtype=np.uint8).tobytes(), dtype=np.uint32)


def _f16(bits):
    return float(np.array([bits], dtype=np.uint16).view(np.float16)[0])


def emulate(oracle, rows, types, K, mode, M, weights, x, rng):
    """The kernel's arithmetic at lane level; returns y per segment (mode 0) or h (mode 1)."""
    cfg = fits(rows, types, K, mode)
    ranges, groups_max = cfg[1:3]
    S, stride = K // 256, K + 16
    parts = 2 if mode == 1 else 1
    codes_q, scales_q = oracle.quantize_q8(x)
    codes_q = codes_q.reshape(M, K)
    scales_q = scales_q.reshape(M, K // 32)
    # LDS image: written rows from the oracle's Q8, garbage elsewhere
    codes = rng.integers(-128, 128, size=(8, stride), dtype=np.int64)
    codes[:M, :K] = codes_q
    zero = np.zeros(16, dtype=np.int64)
    xs = rng.standard_normal((K // 32, 8)) * 1e3
    xss = rng.standard_normal((K // 32, 8)) * 1e3
    xf = rng.integers(-(1 << 20), 1 << 20, size=(K // 16, 8), dtype=np.int64)
    c32 = codes_q.reshape(M, K // 32, 32).astype(np.int64)
    xs[:, :M] = scales_q.T
    xss[:, :M] = (scales_q * c32.sum(axis=2)).T
    xf[0::2, :M] = (-32 * c32[:, :, :16].sum(axis=2)).T  # int32: the Q6_K MFMA's accumulator input
    xf[1::2, :M] = (-32 * c32[:, :, 16:].sum(axis=2)).T

    def a_tile(offs):  # A[r][16kq+t] from lane (r, kq) = (l%16, l/16) reading 16 bytes at offs[l]
        A = np.zeros((16, 64), dtype=np.int64)
        for l in range(64):
            o = offs[l]
            if o == 8 * stride:
                vals = zero
            else:
                m, k = divmod(int(o), stride)
                vals = codes[m, k:k + 16]
            A[l % 16, 16 * (l // 16):16 * (l // 16) + 16] = vals
        return A

    def b_tile(byte_rows):  # B[16kq+t][n] from lane (n, kq) holding 16 bytes byte_rows[l]
        Bm = np.zeros((64, 16), dtype=np.int64)
        for l in range(64):
            Bm[16 * (l // 16):16 * (l // 16) + 16, l % 16] = byte_rows[l]
        return Bm

    def lane_c(C):  # lane l's four results C[4(l/16)+i][l%16]
        return np.stack([C[4 * (LANE // 16) + i, LANE % 16] for i in range(4)], axis=1)

    nseg = 1 if mode == 1 else len(rows)
    out = [np.full((M, rows[j]), np.nan) for j in range(nseg)]
    for j, sh in workgroups(rows, types, K, mode, cfg):
        qtype = types[j]
        B = BYTES[qtype]
        sums = np.full((parts, groups_max, 16, ranges, 8), np.nan)
        for wave in range(WAVES):
            comps, _ = wave_streams(sh, wave, P[qtype])
            acc = np.zeros((64, 4))
            for part, g, rr, s, last in comps:
                w = weights[1] if (mode == 1 and part) else weights[j]
                row = np.minimum(16 * g + LN, sh.nrows - 1) + sh.r0
                sbs = w.reshape(-1, S, B)[row, s]  # [64 lanes][B bytes]
                kq, khi, klo = LKQ, LKQ >> 1, LKQ & 1
                if qtype == 12:
                    head = np.stack([_u32(sbs[l, :16]) for l in range(64)])
                    qa = np.stack([sbs[l, 16 + 16 * kq[l]:32 + 16 * kq[l]] for l in range(64)]).astype(np.int64)
                    qb = np.stack([sbs[l, 80 + 16 * kq[l]:96 + 16 * kq[l]] for l in range(64)]).astype(np.int64)
                    valid = (LN < 8) == (kq < 2)
                    base = (LN & 7) * stride + 16 * klo
                    mainv, minv = np.zeros((64, 4)), np.zeros((64, 4))
                    for h in range(2):
                        for nib in range(2):
                            jj = 4 * h + nib + 2 * khi
                            A = a_tile(np.where(valid, base + 256 * s + 32 * jj, 8 * stride))
                            q = qb if h else qa
                            Bm = b_tile((q >> 4) & 15 if nib else q & 15)
                            C = lane_c(A @ Bm)
                            o = 8 * (nib + 2 * khi)
                            s0, s1, s2 = head[:, 1], head[:, 2], head[:, 3]
                            if h == 0:
                                sc, mn = (s0 >> o) & 63, (s1 >> o) & 63
                            else:
                                sc = ((s2 >> o) & 15) | (((s0 >> (o + 6)) & 3) << 4)
                                mn = ((s2 >> (o + 4)) & 15) | (((s1 >> (o + 6)) & 3) << 4)
                            x4 = np.stack([xs[8 * s + jj[l], 4 * klo[l]:4 * klo[l] + 4] for l in range(64)])
                            y4 = np.stack([xss[8 * s + jj[l], 4 * klo[l]:4 * klo[l] + 4] for l in range(64)])
                            mainv += C * x4 * sc[:, None]
                            minv += mn[:, None] * y4
                    d = np.array([_f16(v & 0xFFFF) for v in head[:, 0]])
                    dmin = np.array([_f16(v >> 16) for v in head[:, 0]])
                    acc += d[:, None] * mainv - dmin[:, None] * minv
                else:
                    ql = [np.stack([sbs[l, 64 * h + 16 * kq[l]:64 * h + 16 * kq[l] + 16] for l in range(64)]).astype(np.int64) for h in range(2)]
                    qh = [np.stack([sbs[l, 128 + 32 * h + 16 * klo[l]:128 + 32 * h + 16 * klo[l] + 16] for l in range(64)]).astype(np.int64) for h in range(2)]
                    scb = np.stack([sbs[l, 192:208] for l in range(64)]).view(np.int8).astype(np.int64)
                    d = np.array([_f16(int(sbs[l, 208]) | int(sbs[l, 209]) << 8) for l in range(64)])
                    accsb = np.zeros((64, 4))
                    for h in range(2):
                        for nib in range(2):
                            # the kernel's dword ops: lo nibbles, qh rotated right by
                            # sh = 28 + 2*khi (nib 0) or 2*khi (nib 1), bits 4-5 inserted
                            sh_r = (28 + 2 * khi) if nib == 0 else 2 * khi
                            codes16 = np.zeros((64, 16), dtype=np.int64)
                            for l in range(64):
                                lw = _u32(ql[h][l].astype(np.uint8)).astype(np.uint64)
                                hw = _u32(qh[h][l].astype(np.uint8)).astype(np.uint64)
                                lo = ((lw >> 4) if nib else lw) & 0x0F0F0F0F
                                r = int(sh_r[l])
                                hs = ((hw >> r) | (hw << (32 - r))) & 0xFFFFFFFF if r else hw
                                word = (hs & 0x30303030) | (lo & ~np.uint64(0x30303030) & 0xFFFFFFFF)
                                codes16[l] = np.frombuffer(word.astype(np.uint32).tobytes(), dtype=np.uint8)
                            Bm = b_tile(codes16)
                            blk = 4 * h + 2 * nib + khi
                            k0 = 256 * s + 128 * h + 64 * nib
                            for p in range(2 if M > 4 else 1):
                                if M > 4:  # products of the two sub-blocks of one Q8 block
                                    valid = ((LN >> 3) == khi) & (klo == p)
                                    base, m0, sb16 = (LN & 7) * stride + 16 * kq, 4 * klo, 2 * blk + p
                                else:
                                    valid = (LN >> 2) == kq
                                    base, m0, sb16 = (LN & 3) * stride + 16 * kq, 0 * klo, 8 * h + 4 * nib + kq
                                A = a_tile(np.where(valid, base + k0, 8 * stride))
                                n4 = np.stack([xf[16 * s + sb16[l], m0[l]:m0[l] + 4] for l in range(64)])
                                C = lane_c(A @ Bm) + n4  # D = A B + C, exact in int32
                                x4 = np.stack([xs[8 * s + blk[l], m0[l]:m0[l] + 4] for l in range(64)])
                                accsb += scb[LANE, sb16][:, None] * (x4 * C)
                    acc += d[:, None] * accsb
                if last:
                    v = acc + acc[LANE ^ 32]
                    lanes = 32  # activation rows 4 (kq & 1).. in lanes of kq < 2
                    if qtype == 14 and M <= 4:
                        v, lanes = v + v[LANE ^ 16], 16
                    for l in range(lanes):
                        sums[part, g, l & 15, rr, 4 * (l >> 4):4 * (l >> 4) + 4] = v[l]
                    acc[:] = 0.0
        for m in range(M):
            for rw in range(sh.nrows):
                a = sums[0, rw >> 4, rw & 15, :, m].sum()
                if mode == 0:
                    out[j][m, sh.r0 + rw] = a
                else:
                    b = sums[1, rw >> 4, rw & 15, :, m].sum()
                    out[j][m, sh.r0 + rw] = a / (1.0 + np.exp(-a)) * b
    return out


EMULATED = [  # rows, types, K, mode, M
    ([40], [12], 512, 0, 8),
    ([37], [14], 768, 0, 8),
    ([23], [14], 512, 0, 3),
    ([20, 9, 13], [12, 12, 14], 256, 0, 5),
    ([33, 33], [12, 12], 512, 1, 2),
]


@pytest.mark.parametrize("rows,types,K,mode,M", EMULATED)
def test_bmv_arithmetic_matches_oracle(oracle, rows, types, K, mode, M):
    rng = np.random.default_rng(5)
    x = oracle.synth_normal(M * K, 20261300 + K + M)
    nmat = len(rows)
    weights = [oracle.synth_superblocks(types[i], rows[i], K, 20261400 + i, 0.01 if types[i] == 12 else 0.005, 0.01)
               for i in range(nmat)]
    got = emulate(oracle, rows, types, K, mode, M, weights, x, rng)
    if mode == 0:
        for j in range(nmat):
            ref = oracle.reference_product(x, weights[j], types[j], K, rows[j])
            assert oracle.row_norm_error(got[j], ref) <= 1e-6
    else:
        g = oracle.reference_product(x, weights[0], types[0], K, rows[0])
        u = oracle.reference_product(x, weights[1], types[1], K, rows[1])
        ref = g / (1.0 + np.exp(-g)) * u
        assert oracle.row_norm_error(got[0], ref) <= 1e-6


def _owner(r, per, rem):
    big = rem * (per + 1)
    return r // (per + 1) if r < big else rem + (r - big) // per


@pytest.mark.parametrize("N,M,count", [(9728, 8, 256), (9728, 2, 256), (512, 5, 7), (2048, 8, 100),
                                       (96, 3, 50), (6144, 8, 256), (256, 8, 256)])
def test_bmv_q8h_blocks_close_once(N, M, count):
    """Q8(h) in the gate/up launch (bmv_close_blocks): whatever order the
    workgroups arrive in, each 32-value block of h is completed by exactly one
    workgroup, after every workgroup owning one of its rows arrived, every
    counter is back at zero for the next launch, and the closing quads fit the
    workgroup (the launcher's bound on blocks per share holds)."""
    count = min(count, N)
    per, rem = divmod(N, count)
    rows_max = per + (1 if rem else 0)
    bound = (rows_max + 30) // 32 + 1
    if not (N % 32 == 0 and bound <= 16 and 4 * bound * M <= 64 * WAVES):
        return  # the launcher declines; the separate quantise launch runs
    rng = np.random.default_rng(N + M + count)
    for trial in range(3):
        arrive = np.zeros(N // 32, dtype=np.int64)
        closed = np.zeros(N // 32, dtype=np.int64)
        arrived = np.zeros(N // 32, dtype=np.int64)
        for g in rng.permutation(count):
            r0, nrows = g * per + min(g, rem), per + (1 if g < rem else 0)
            b0 = r0 >> 5
            nb = ((r0 + nrows - 1) >> 5) - b0 + 1
            assert nb <= bound
            for i in range(nb):
                b = b0 + i
                first, last = _owner(32 * b, per, rem), _owner(min(32 * b + 31, N - 1), per, rem)
                assert first <= g <= last
                arrive[b] += 1
                arrived[b] += 1
                if arrive[b] == last - first + 1:
                    arrive[b] = 0
                    closed[b] += 1
                    assert arrived[b] == last - first + 1  # every owner's h is stored
                    quads = [(i * M + m) for m in range(M)]
                    assert max(quads) * 4 + 3 < 64 * WAVES
        assert np.all(closed == 1) and np.all(arrive == 0)
    # the owner function restates the cut
    for r in range(0, N, max(1, N // 97)):
        g = _owner(r, per, rem)
        assert g * per + min(g, rem) <= r < g * per + min(g, rem) + per + (1 if g < rem else 0)


@pytest.mark.parametrize("K", [256, 2560])
def test_q6k_pair_tile_model(K):
    """Q6_K at M = 5..8 (bmv_half6<2>): product p's A rows 4g..4g+3 hold
    activation rows 4(g & 1).. against k-quarter 2(g >> 1) + p, so that lane
    (n, kq) gets both sub-blocks of Q8 block 4h + 2nib + (kq >> 1) for activation
    rows 4(kq & 1)..; every read stays in its LDS array, the integer sums stay
    below 2^24 at the extreme codes and scales, and the lanes' sums are the
    product's."""
    stride, Z, S = K + 16, 8 * (K + 16) + 16, K // 256
    rng = np.random.default_rng(K)
    x = rng.integers(-127, 128, (8, K))
    q, sc = rng.integers(0, 64, (16, K)), rng.integers(-128, 128, (16, K // 16))
    x[:, :32], q[:, :32], sc[:, :2] = -127, 0, -128  # the extreme: 16 * 127 * 32 * 128, twice
    xs = rng.standard_normal((K // 32, 8))
    lds = np.zeros((8, stride), np.int64)
    lds[:, :K] = x
    lds = np.concatenate([lds.ravel(), np.zeros(16, np.int64)])
    neg = -32 * x.reshape(8, -1, 16).sum(2).T  # [K / 16][8]
    acc = np.zeros((64, 4))
    klo, khi = LKQ & 1, LKQ >> 1
    for s in range(S):
        for h in range(2):
            for nib in range(2):
                k0 = 256 * s + 128 * h + 64 * nib
                blk = 4 * h + 2 * nib + khi
                total = np.zeros((64, 4), np.int64)
                for p in range(2):
                    valid = ((LN >> 3) == khi) & (klo == p)
                    aoff = np.where(valid, (LN & 7) * stride + 16 * LKQ + k0, 8 * stride)
                    assert np.all(aoff % 16 == 0) and np.all(aoff + 16 <= 8 * stride + 16)
                    A, Bm = np.zeros((16, 64), np.int64), np.zeros((64, 16), np.int64)
                    for l in range(64):
                        A[LN[l], 16 * LKQ[l]:16 * LKQ[l] + 16] = lds[aoff[l]:aoff[l] + 16]
                        Bm[16 * LKQ[l]:16 * LKQ[l] + 16, LN[l]] = q[LN[l], k0 + 16 * LKQ[l]:k0 + 16 * LKQ[l] + 16]
                    D = A @ Bm
                    off = Z + 2 * K + 4 * ((16 * s + 2 * blk + p) * 8 + 4 * klo)
                    assert np.all(off >= Z + 2 * K) and np.all(off + 16 <= Z + 4 * K)
                    sb = 16 * s + 2 * blk + p
                    for l in range(64):
                        dot = D[4 * LKQ[l]:4 * LKQ[l] + 4, LN[l]] + neg[sb[l], 4 * klo[l]:4 * klo[l] + 4]
                        assert np.all(np.abs(dot) < 1 << 23)
                        total[l] += dot * sc[LN[l], sb[l]]
                assert np.abs(total).max() <= 1 << 24
                off = Z + 4 * ((8 * s + blk) * 8 + 4 * klo)
                assert np.all(off + 16 <= Z + K)
                for l in range(64):
                    acc[l] += xs[8 * s + blk[l], 4 * klo[l]:4 * klo[l] + 4] * total[l]
    v = acc + acc[LANE ^ 32]
    want = np.einsum("mk,nk->nm", x * np.repeat(xs.T, 32, 1), (q - 32) * np.repeat(sc, 16, 1))
    for l in range(32):
        assert np.allclose(v[l], want[LN[l], 4 * LKQ[l]:4 * LKQ[l] + 4], rtol=1e-12)


@pytest.mark.parametrize("N,S", [(2560, 38), (3328, 10), (2561, 7), (3, 1), (40, 41)])
def test_bmv_q6k_slots(N, S):
    """Q6_K in mode 0: the tile's chunks (dword-aligned 16-byte loads, at most
    three a lane) put every superblock of the share's rows into the wave's slot
    whole, where ws_tile6 reads its 54 dwords; no load passes the matrix's last
    dword except into the descriptor's zeros, no write passes the slot."""
    CH, LOADS = SLOT_CHUNKS, SLOT_LOADS
    count = min(CUS, N)
    rows_max = -(-N // count)
    assert rows_max <= SLOT_ROWS
    rb, total = S * 210, N * S * 210
    end4 = (total + 3) & ~3
    per, rem = N // count, N % count
    mat = np.zeros(end4 + 64, np.uint8)
    mat[:total] = np.arange(total, dtype=np.int64) * 2654435761 % 251 + 1
    for g in {0, rem, count - 1}:
        r0, nrows = g * per + min(g, rem), per + (1 if g < rem else 0)
        n = CH * nrows
        c = np.minimum(np.arange(64 * LOADS), n - 1)
        assert n <= 64 * LOADS and 16 * n <= 16 * CH * rows_max
        for s in range(S):
            off = (((r0 + c // CH) * rb + s * 210) & ~3) + 16 * (c % CH)
            slot = np.zeros(16 * n, np.uint8)
            for o, k in zip(off, c):
                assert o % 4 == 0
                slot[16 * k:16 * k + 16] = np.where(o + np.arange(16) < end4, mat[np.minimum(o + np.arange(16), end4)], 0)
            for row in range(nrows):
                first = (r0 + row) * rb + s * 210
                o = 16 * CH * row + (first & 3)
                assert (first & 3) in (0, 2) and 4 * 54 <= 16 * CH
                assert np.array_equal(slot[o:o + 210], mat[first:first + 210])
