// Batched mat-vec on the int8 matrix cores: M = 2..8 activation rows (the
// decode batch of several sequences), fp32 activations quantised in the
// kernel or Q8 blocks copied in. Replaces quantize + project<Q4_K/Q6_K> with gridDim.y = rows
// (src/cuda/matmul.cu:8-22, 86-125, 151-158), which re-reads every weight row
// once per activation row.
//
// With integer dots on the vector ALU every lane needs the activation bytes
// that match its weights, so an M-row launch reads M activation fragments
// from LDS per weight piece (96 bytes per 64 weights per row): at M = 8 the
// LDS, not HBM, bounds it. Here one v_mfma_i32_16x16x64_i8 takes 16 weight
// rows (B columns) against an activation tile (A rows) that all 16 rows
// share. Sub-block scales (32 weights for Q4_K, 16 for Q6_K) and the Q8
// block scales (32 activations) vary along k, so each MFMA spans exactly the
// sub-blocks whose products it keeps apart: its A tile is block-diagonal.
//   Q4_K: k 0..31 = sub-block j1, k 32..63 = j2 (the low or high nibbles of
//         64 qs bytes); A rows 0..7 = activation rows 0..7 against j1, rows
//         8..15 = the same rows against j2, zero elsewhere.
//   Q6_K: k = 4 sub-blocks of 16 (one nibble of 64 ql bytes with their qh
//         bit pairs); M <= 4: A rows 4b..4b+3 = the activation rows against
//         sub-block b; M > 4: two MFMAs on the same B, in product p A rows
//         4b..4b+3 = activation rows 4*(b&1)..+3 against sub-block 2*(b>>1)+p.
// Lane l holds A[l%16][16(l/16)..+16], B[16(l/16)..+16][l%16] and receives
// C[4(l/16)+i][l%16], i < 4 (probed on gfx950), so lane (n, kq) = (l%16, l/16)
// loads the 16 weight bytes of row n for k-quarter kq straight from memory,
// and its four integer results belong to one sub-block and four activation
// rows: they are scaled by that sub-block's scale and the rows' Q8 scales in
// fp32 (Q4_K: d*sc*xs*dot - dmin*m*xs*sum(codes); Q6_K: d*sc*xs*(dot - 32
// sum(codes)), src/cuda/matmul.cu:24-84).
//
// A workgroup (one per CU) owns a contiguous range of rows of one matrix (mode
// 1: of gate and of up); its rows are cut into groups of 16 and each group's superblock columns
// into `ranges` runs. Work units (part, group, run) are dealt to the waves in
// contiguous blocks; a wave streams its units' tiles (16 rows x one
// superblock) through a ring of P register buffers, P tiles ahead, so
// memory stays busy while earlier tiles are computed. Each unit's sums go to
// LDS; after a barrier one thread per (row, activation row) adds the runs in
// order and stores (results do not depend on timing).
#pragma once

#include <type_traits>

#include "gemv_stream.hpp"

namespace qk {

// 16 waves with shallow rings: a wave has 1 to 4 tiles, so deep rings mostly
// load tiles again past its end, and four waves a SIMD hide the LDS reads and
// the MFMAs of each other's tiles. Measured, gate/up (Q4_K) at M = 3 / 8: 8
// waves with rings of 6 13.6 / 14.7 us, 16 waves with rings of 4 12.4 / 13.0, of
// 2 11.0 / 11.8 (of 1: equal); Q6_K 26.1 / 27.3 -> 22.0 / 23.2.
constexpr int kBmvWaves = 16;   // waves per workgroup (one workgroup per CU)
// activation tasks (Q8 blocks) per lane whose loads are issued before the
// weights
constexpr int kBmvXStaged = 2;
constexpr int kBmvQ8Staged = 2;
constexpr int kBmvP4 = 2;       // Q4_K tiles in flight per wave
constexpr int kBmvP6 = 1;       // Q6_K tiles in flight per wave (mode 1)
// Q6_K in mode 0: a tile's rows go through a slot of the wave in LDS
constexpr int kBmvSlotChunks = 14;  // 16-byte chunks that cover a superblock from the dword boundary below it
constexpr int kBmvSlotLoads = 3;    // chunks per lane and tile
constexpr int kBmvSlotRows = 64 * kBmvSlotLoads / kBmvSlotChunks;  // rows of a workgroup at most: 13
constexpr int kBmvSlotP = 1;        // tiles in flight per wave
constexpr int kBmvMaxGroups = 2;    // row groups a workgroup in a launch of several matrices (q/k/v)
// Q8 blocks of h one workgroup may complete (M activation rows each, a quad
// per block row): the launcher checks blocks * M * 4 <= threads.
constexpr int kBmvMaxCloseBlocks = 16;

struct BmvParams {
  const float* x;       // [M x K], or null:
  const qk_q8_block* q8;  // [M x K/32] (mode 0)
  float* h;             // mode 1 output [M x N]
  qk_q8_block* hq;      // mode 1, optional: Q8 of h [M][N/32], formed in the launch
  uint32_t* arrive;     // with hq: per-block arrival counters [N/32], zero between launches
  int32_t M, K, S;
  int32_t stride;      // LDS bytes per activation row of codes (K + 16)
  int32_t ranges;      // superblock runs per row group
  int32_t groups_max;  // row groups of the largest workgroup share
  int32_t rows_max;    // rows of the largest share that goes through slots
  int32_t pad;
  int32_t nseg, pad2;
  StreamSegment seg[kMaxSegments];  // mode 0: the matrices; mode 1: gate and up
};

// LDS image (byte offsets; K a multiple of 256):
//   codes [8][stride] int8         at 0 (rows m >= M are never written)
//   zero  16 bytes                 at 8*stride
//   xs    [K/32][8] fp32 Q8 scale  at Z = 8*stride + 16
//   xss   [K/32][8] fp32 scale*sum(codes)          at Z + K
//   xf    [K/16][8] int32 -32*(sum of 16 codes)    at Z + 2K (the Q6_K offset,
//                                                  the MFMA's accumulator input)
//   sums  [parts][groups_max][16][ranges][8] fp32  at Z + 4K
//   slots [waves][rows][14 chunks]                 after the sums (Q6_K, mode 0)
// Rows m >= M of every array are left unwritten: they feed only results for
// activation rows that are never stored.
__host__ __device__ constexpr int bmv_lds_z(int stride) { return 8 * stride + 16; }
__host__ __device__ constexpr int bmv_lds_bytes(int K, int stride, int parts, int groups, int ranges) {
  return bmv_lds_z(stride) + 4 * K + parts * groups * 16 * ranges * 32;
}
__host__ __device__ constexpr int bmv_slot_bytes(int rows) { return 16 * kBmvSlotChunks * rows; }

typedef __attribute__((address_space(3))) f32x4 lds_f32x4;

typedef int32_t i32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i32x4 lds_i32x4;
typedef __attribute__((address_space(3))) int32_t lds_i32;

// Task t (8 activations of the [M][K] stream): codes to row t / (K/8), the
// block's scales by lane 0 of its quad.
__device__ __forceinline__ void bmv_quantize_task(f32x4 a, f32x4 b, int t, int groups, int stride,
                                                  lds_u8* codes, lds_f32* xs, lds_f32* xss, lds_f32* xf) {
  const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
  const Q8Quarter q = quantize_quarter(v);
  const int m = t / groups, k0 = 8 * (t - m * groups);
  *reinterpret_cast<lds_u32x2*>(codes + m * stride + k0) = u32x2{q.lo, q.hi};
  if ((t & 3) == 0) {
    const int blk = k0 >> 5;
    xs[blk * 8 + m] = q.scale;
    xss[blk * 8 + m] = q.scale * static_cast<float>(q.pair + q.other);
    lds_i32* xi = reinterpret_cast<lds_i32*>(xf);
    xi[(2 * blk) * 8 + m] = -32 * q.pair;
    xi[(2 * blk + 1) * 8 + m] = -32 * q.other;
  }
}

// Block b of caller-provided Q8 blocks [M][K/32] (its three 16-byte words:
// codes 0..15, codes 16..31, then scale / scale*sum / -32*sum(0..15) /
// -32*sum(16..31)) into the LDS image bmv_quantize_task writes: the same
// codes, the same scale, the same fp32 product scale*sum and the same
// integer offsets. The record is bit cast as a whole vector: a bit cast of
// one subscripted element (rec.y) was compiled as the vector's first element.
__device__ __forceinline__ void bmv_store_block(u32x4 c0, u32x4 c1, u32x4 rec, int b, int bpr, int stride,
                                                lds_u8* codes, lds_f32* xs, lds_f32* xss, lds_f32* xf) {
  const int m = b / bpr, blk = b - m * bpr;
  lds_u8* row = codes + m * stride + 32 * blk;
  *reinterpret_cast<lds_u32x4*>(row) = c0;
  *reinterpret_cast<lds_u32x4*>(row + 16) = c1;
  const f32x4 rf = __builtin_bit_cast(f32x4, rec);
  const float scale = rf.x;
  xs[blk * 8 + m] = scale;
  xss[blk * 8 + m] = rf.y;
  lds_i32* xi = reinterpret_cast<lds_i32*>(xf);
  xi[(2 * blk) * 8 + m] = static_cast<int32_t>(rec.z);
  xi[(2 * blk + 1) * 8 + m] = static_cast<int32_t>(rec.w);
}

// A lane's register image of one tile (16 rows x one superblock).
struct Q4Tile {
  u32x4 head, qa, qb;  // d, dmin, scales; qs[16kq..+16]; qs[64+16kq..+16]
};
struct Q6Tile {
  u32x4 la, lb, ha, hb, sc;  // ql[16kq..], ql[64+16kq..], qh[16(kq&1)..], qh[32+16(kq&1)..], scales
  uint32_t d;
};

template <int TYPE>
using BmvTile = typename std::conditional<TYPE == QK_TYPE_Q4_K, Q4Tile, Q6Tile>::type;

// Loads of a tile: sb = this lane's row's superblock (16-byte aligned for
// Q4_K, 2-byte for Q6_K); every byte read lies inside the superblock.
__device__ __forceinline__ void bmv_load(Q4Tile& t, const uint8_t* sb, int kq) {
  t.head = load16(sb);
  t.qa = load16(sb + 16 + 16 * kq);
  t.qb = load16(sb + 80 + 16 * kq);
}
__device__ __forceinline__ void bmv_load(Q6Tile& t, const uint8_t* sb, int kq) {
  t.la = load16_a2(sb + 16 * kq);
  t.lb = load16_a2(sb + 64 + 16 * kq);
  t.ha = load16_a2(sb + 128 + 16 * (kq & 1));
  t.hb = load16_a2(sb + 160 + 16 * (kq & 1));
  t.sc = load16_a2(sb + 192);
  t.d = load_u16(sb + 208);
}

__device__ __forceinline__ i32x4 mfma_i8(i32x4 a, u32x4 b, i32x4 c = i32x4{0, 0, 0, 0}) {
  return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, __builtin_bit_cast(i32x4, b), c, 0, 0, 0);
}

__device__ __forceinline__ i32x4 lds_read_i32x4(const lds_u8* base, uint32_t off) {
  return *reinterpret_cast<const lds_i32x4*>(base + off);
}
__device__ __forceinline__ f32x4 lds_read_f32x4(const lds_f32* p) {
  return *reinterpret_cast<const lds_f32x4*>(p);
}

// Per-lane constants of the tile computation.
struct BmvLane {
  int n, kq;
  uint32_t a4_base;   // Q4_K A: this lane's activation row and k-quarter, or the zero line
  bool a4_valid;
  uint32_t a6_base;   // Q6_K A at M <= 4
  bool a6_valid;
  uint32_t a6p_base;  // Q6_K A at M > 4: product p reads it in the lanes of odd (p) / even k-quarters
  bool a6p_valid[2];
  uint32_t zero;
};

__device__ __forceinline__ BmvLane bmv_lane(int lane, int stride) {
  BmvLane L;
  L.n = lane & 15;
  L.kq = lane >> 4;
  L.zero = static_cast<uint32_t>(8 * stride);
  L.a4_valid = (L.n < 8) == (L.kq < 2);
  L.a4_base = static_cast<uint32_t>((L.n & 7) * stride + 16 * (L.kq & 1));
  L.a6_valid = (L.n >> 2) == L.kq;
  L.a6_base = static_cast<uint32_t>((L.n & 3) * stride + 16 * L.kq);
  L.a6p_base = static_cast<uint32_t>((L.n & 7) * stride + 16 * L.kq);
  for (int p = 0; p < 2; ++p) L.a6p_valid[p] = (L.n >> 3) == (L.kq >> 1) && (L.kq & 1) == p;
  return L;
}

// Q4_K tile at superblock column s: acc[i] += row n's dot for activation row
// 4*(kq&1)+i over the sub-blocks of set kq>>1 (the other set sits in lane l^32).
__device__ __forceinline__ void bmv_tile(const Q4Tile& t, int s, const BmvLane& L, int stride,
                                         const lds_u8* codes, const lds_f32* xs, const lds_f32* xss,
                                         f32x4& acc) {
  const int khi = L.kq >> 1, klo = L.kq & 1;
  i32x4 c[4];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int nib = 0; nib < 2; ++nib) {
      const int j = 4 * h + nib + 2 * khi;  // this lane's sub-block (A side and C side)
      const uint32_t aoff = L.a4_valid ? L.a4_base + 256 * s + 32 * j : L.zero;
      const u32x4 q = h ? t.qb : t.qa;
      const u32x4 bq = nib ? ((q >> 4) & 0x0F0F0F0Fu) : (q & 0x0F0F0F0Fu);
      c[2 * h + nib] = mfma_i8(lds_read_i32x4(codes, aoff), bq);
    }
  }
  const uint32_t s0 = t.head.y, s1 = t.head.z, s2 = t.head.w;
  f32x4 mainv = {0.0f, 0.0f, 0.0f, 0.0f}, minv = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int nib = 0; nib < 2; ++nib) {
      const int j = 4 * h + nib + 2 * khi;
      // 6-bit (scale, min) of sub-block j (get_scale_min_k4, src/cuda/embedding.cu:20-23)
      const uint32_t o = 8u * static_cast<uint32_t>(nib + 2 * khi);
      uint32_t sc, mn;
      if (h == 0) {
        sc = ubfe(s0, o, 6);
        mn = ubfe(s1, o, 6);
      } else {
        sc = ubfe(s2, o, 4) | (ubfe(s0, o + 6, 2) << 4);
        mn = ubfe(s2, o + 4, 4) | (ubfe(s1, o + 6, 2) << 4);
      }
      const float scf = static_cast<float>(sc);
      const float mf = static_cast<float>(mn);
      const f32x4 x4 = lds_read_f32x4(xs + (8 * s + j) * 8 + 4 * klo);
      const f32x4 y4 = lds_read_f32x4(xss + (8 * s + j) * 8 + 4 * klo);
      const i32x4 ci = c[2 * h + nib];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        mainv[i] = __builtin_fmaf(static_cast<float>(ci[i]), x4[i] * scf, mainv[i]);
        minv[i] = __builtin_fmaf(mf, y4[i], minv[i]);
      }
    }
  }
  const float d = half_bits_to_float(t.head.x & 0xFFFFu);
  const float dmin = half_bits_to_float(t.head.x >> 16);
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i] = __builtin_fmaf(-dmin, minv[i], __builtin_fmaf(d, mainv[i], acc[i]));
}

// 16 codes of nibble nib of a Q6_K half's bytes (ql nibble | qh pair << 4,
// 0..63): src/cuda/matmul.cu:71-79. The qh bit pair of group 2 nib + khi moves
// to bits 4-5 of each byte.
__device__ __forceinline__ u32x4 bmv_codes6(u32x4 ql, u32x4 qh, int nib, int khi) {
  const uint32_t sh = (nib ? 0u : 28u) + 2u * static_cast<uint32_t>(khi);
  u32x4 b;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t lo = nib ? (ql[e] >> 4) & 0x0F0F0F0Fu : ql[e] & 0x0F0F0F0Fu;
    b[e] = bit_insert(0x30303030u, __builtin_amdgcn_alignbit(qh[e], qh[e], sh), lo);
  }
  return b;
}

// Half h of a Q6_K tile at superblock column s (sc[nib]: scales 8h+4nib..+3).
// The -32 offset of the codes enters as the MFMA's accumulator input
// -32 * sum(activation codes), so the integer dots are exact.
//  MH = 1 (M <= 4): acc[i] += row n's dot for activation row i over the
//    sub-blocks 8h+4nib+kq (the other kq in lanes l^16, l^32).
//  MH = 2 (M = 5..8): acc[i] += the dot for activation row 4*(kq&1)+i over the
//    Q8 blocks 4h+2nib+(kq>>1) (the others in lane l^32). A rows 4g..4g+3 hold
//    activation rows 4*(g&1).. against k-quarter 2*(g>>1)+p in product p, so a
//    lane's two products are the two sub-blocks of ONE Q8 block and the same
//    four activation rows: sc0*dot0 + sc1*dot1 is formed in integers (|dot| <=
//    16*127*32 < 2^17 and |sc| <= 128: exact in 32 bits) and takes one
//    conversion and one block scale, where a product of its own per half of
//    the activation rows took two of each (lm_head at M = 5 / 8: 79.2 / 80.2
//    -> 75.4 / 76.4 us).
template <int MH>
__device__ __forceinline__ void bmv_half6(u32x4 ql, u32x4 qh, uint32_t sc0, uint32_t sc1, int h, int s,
                                          const BmvLane& L, const lds_u8* codes, const lds_f32* xs,
                                          const lds_f32* xf, f32x4& acc) {
  const int khi = L.kq >> 1, klo = L.kq & 1;
#pragma unroll
  for (int nib = 0; nib < 2; ++nib) {
    const u32x4 b = bmv_codes6(ql, qh, nib, khi);
    const uint32_t scw = nib ? sc1 : sc0;
    const int blk = 4 * h + 2 * nib + khi;  // this lane's Q8 block
    const lds_u8* neg = reinterpret_cast<const lds_u8*>(xf);
    if constexpr (MH == 1) {
      const int sb16 = 8 * h + 4 * nib + L.kq;  // this lane's sub-block
      const float scf = static_cast<float>(static_cast<int8_t>((scw >> (8 * L.kq)) & 0xFFu));
      const uint32_t aoff = L.a6_valid ? L.a6_base + 256 * s + 128 * h + 64 * nib : L.zero;
      const i32x4 n4 = lds_read_i32x4(neg, 4u * ((16 * s + sb16) * 8));
      const i32x4 ci = mfma_i8(lds_read_i32x4(codes, aoff), b, n4);
      const f32x4 x4 = lds_read_f32x4(xs + (8 * s + blk) * 8);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = __builtin_fmaf(scf, x4[i] * static_cast<float>(ci[i]), acc[i]);
    } else {
      i32x4 dot[2];
      int sc[2];
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const uint32_t aoff = L.a6p_valid[p] ? L.a6p_base + 256 * s + 128 * h + 64 * nib : L.zero;
        const i32x4 n4 = lds_read_i32x4(neg, 4u * ((16 * s + 2 * blk + p) * 8 + 4 * klo));
        dot[p] = mfma_i8(lds_read_i32x4(codes, aoff), b, n4);
        sc[p] = __builtin_amdgcn_sbfe(static_cast<int>(scw), 16 * khi + 8 * p, 8);
      }
      const f32x4 x4 = lds_read_f32x4(xs + (8 * s + blk) * 8 + 4 * klo);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int sum = __mul24(dot[0][i], sc[0]) + __mul24(dot[1][i], sc[1]);
        acc[i] = __builtin_fmaf(x4[i], static_cast<float>(sum), acc[i]);
      }
    }
  }
}

// The tile of either type: MH = 1 for M <= 4, 2 for M = 5..8 (Q4_K: the same).
template <int MH>
__device__ __forceinline__ void bmv_tile_any(const Q4Tile& t, int s, const BmvLane& L, int stride, const lds_u8* codes,
                                             const lds_f32* xs, const lds_f32* xss, const lds_f32*, f32x4& acc) {
  bmv_tile(t, s, L, stride, codes, xs, xss, acc);
}
template <int MH>
__device__ __forceinline__ void bmv_tile_any(const Q6Tile& t, int s, const BmvLane& L, int, const lds_u8* codes,
                                             const lds_f32* xs, const lds_f32*, const lds_f32* xf, f32x4& acc) {
  f32x4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
  bmv_half6<MH>(t.la, t.ha, t.sc.x, t.sc.y, 0, s, L, codes, xs, xf, sum);
  bmv_half6<MH>(t.lb, t.hb, t.sc.z, t.sc.w, 1, s, L, codes, xs, xf, sum);
  const float d = half_bits_to_float(t.d);
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i] = __builtin_fmaf(d, sum[i], acc[i]);
}

// A unit's sums over its lanes: every lane of the result holds activation rows
// 4*(kq&1).. (Q4_K, and Q6_K at M > 4: the other sub-block set is in lane
// l^32) or rows 0..3 (Q6_K at M <= 4: one sub-block of four in each kq).
template <int TYPE, int MH>
__device__ __forceinline__ f32x4 bmv_lane_sums(const f32x4& acc) {
  f32x4 v;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[i] = swap32_sum(acc[i]);
    if constexpr (TYPE == QK_TYPE_Q6_K && MH == 1) v[i] = swap16_sum(v[i]);
  }
  return v;
}
// Lanes whose kq is below this hold distinct sums.
template <int TYPE, int MH>
constexpr int kBmvSumLanes = TYPE == QK_TYPE_Q6_K && MH == 1 ? 1 : 2;

// Position of a wave in its stream of tiles: unit (part, group g, run rr),
// superblock s of the run [s, s_end), tiles left including this one.
struct BmvCursor {
  int part, g, rr, s, s_end, left;
};

// The workgroup's share of one segment and the run split of superblocks.
struct BmvShare {
  const uint8_t* w[2];  // per part (mode 1: gate, up)
  int r0, nrows, groups, S, row_bytes, ranges, run_q, run_r;
  int per, rem;  // the segment's cut: per rows a workgroup, the first rem one more
  __device__ __forceinline__ int run_begin(int rr) const { return rr * run_q + min(rr, run_r); }
};

__device__ __forceinline__ void cursor_seek(BmvCursor& c, const BmvShare& sh, int u) {
  c.rr = u % sh.ranges;
  const int pg = u / sh.ranges;
  c.part = pg / sh.groups;
  c.g = pg - c.part * sh.groups;
  c.s = sh.run_begin(c.rr);
  c.s_end = sh.run_begin(c.rr + 1);
}

__device__ __forceinline__ void cursor_next(BmvCursor& c, const BmvShare& sh) {
  if (c.left > 1) {
    --c.left;
    if (++c.s == c.s_end) {
      if (++c.rr == sh.ranges) {
        c.rr = 0;
        if (++c.g == sh.groups) {
          c.g = 0;
          ++c.part;
        }
      }
      c.s = sh.run_begin(c.rr);
      c.s_end = sh.run_begin(c.rr + 1);
    }
  }
}

// This lane's superblock of the cursor's tile: row min(16g + n, nrows - 1)
// of the share (rows past the share re-read its last row; their results are
// not stored).
template <int B>
__device__ __forceinline__ const uint8_t* bmv_sb(const BmvShare& sh, const BmvCursor& c, int n) {
  const int row = min(16 * c.g + n, sh.nrows - 1);
  return (c.part ? sh.w[1] : sh.w[0]) + static_cast<int64_t>(sh.r0 + row) * sh.row_bytes + c.s * B;
}

// Unit sums into LDS: sums[((part*groups_max + g)*16 + n)*ranges + rr][m].
template <int TYPE, int MH>
__device__ __forceinline__ void bmv_flush(const f32x4& acc, const BmvCursor& c, const BmvLane& L,
                                          int groups_max, int ranges, lds_f32* sums) {
  const f32x4 v = bmv_lane_sums<TYPE, MH>(acc);
  if (L.kq < kBmvSumLanes<TYPE, MH>)
    *reinterpret_cast<lds_f32x4*>(sums + (((c.part * groups_max + c.g) * 16 + L.n) * ranges + c.rr) * 8 +
                                  4 * L.kq) = v;
}

// One type's share: the tile stream of this wave, then (after the caller's
// barrier) nothing; the caller forms the row totals.
template <int TYPE, int P, int MH>
__device__ __forceinline__ void bmv_stream(const BmvShare& sh, BmvCursor lc, const BmvLane& L, int stride,
                                           int groups_max, const lds_u8* codes, const lds_f32* xs,
                                           const lds_f32* xss, const lds_f32* xf, lds_f32* sums,
                                           BmvTile<TYPE> (&buf)[P], BmvCursor cc) {
  constexpr int B = TYPE == QK_TYPE_Q4_K ? kQ4KBytes : kQ6KBytes;
  f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  const int ntiles = cc.left;
  for (int base = 0; base < ntiles; base += P) {
#pragma unroll
    for (int j = 0; j < P; ++j) {
      if (base + j < ntiles) {
        bmv_tile_any<MH>(buf[j], cc.s, L, stride, codes, xs, xss, xf, acc);
        if (cc.s + 1 == cc.s_end) {  // last tile of the unit
          bmv_flush<TYPE, MH>(acc, cc, L, groups_max, sh.ranges, sums);
          acc = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
        cursor_next(cc, sh);
      }
      // refill the buffer P tiles ahead (past the end: the last tile again,
      // from cache), unconditionally so the waits count it
      bmv_load(buf[j], bmv_sb<B>(sh, lc, L.n), L.kq);
      cursor_next(lc, sh);
    }
  }
}

}  // namespace qk
