// Batched mat-vec kernel entry (bmv.hpp) and its host launcher: M = 2..8
// activation rows in fp32 or (one matrix) Q8 blocks, one matrix, several or
// gate and up, one workgroup per CU.
#include <algorithm>
#include <climits>

#include "bmv_ws.hpp"

namespace qk {

namespace {

// Workgroup owning row r of a segment cut as in bmv_kernel (per rows each,
// the first rem workgroups one more).
__device__ __forceinline__ int bmv_owner(int r, int per, int rem) {
  const int big = rem * (per + 1);
  return r < big ? r / (per + 1) : rem + (r - big) / per;
}

// Q8 of h (qk_ffn at M = 2..8) in the gate/up launch. Block b of h (values
// 32b..32b+31 of every activation row) spans the workgroups that own those
// rows. Each of them, once its h stores are performed at the memory side
// (agent-scope stores, then s_waitcnt vmcnt(0) and the workgroup barrier),
// adds 1 to the block's arrival counter (agent-scope atomic, performed at
// the memory side); the one whose add completes the owner count resets the
// counter for the next launch and quantises the block for every activation
// row, a quad per row, with the quantiser of quantize_q8_kernel (same codes
// and record bits). Its h loads are agent-scope loads issued after the
// atomic returned, so they read every owner's stores. No workgroup waits
// for another, so nothing assumes co-residency.
__device__ __forceinline__ void bmv_close_blocks(const BmvParams& p, const BmvShare& sh, int N,
                                                 unsigned char* lds_raw) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this thread's h stores are performed
  __syncthreads();                                   // ... and every thread's
  lds_u32* closes = (lds_u32*)(lds_raw);             // the activation codes are no longer read
  const int tid = static_cast<int>(threadIdx.x);
  const int b0 = sh.r0 >> 5, nb = ((sh.r0 + sh.nrows - 1) >> 5) - b0 + 1;
  const int per = sh.per, rem = sh.rem;
  if (tid < nb) {
    const int b = b0 + tid;
    const int owners = bmv_owner(min(32 * b + 31, N - 1), per, rem) - bmv_owner(32 * b, per, rem) + 1;
    const uint32_t seen =
        __hip_atomic_fetch_add(p.arrive + b, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u;
    const bool last = seen == static_cast<uint32_t>(owners);
    if (last) __hip_atomic_store(p.arrive + b, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    closes[tid] = last ? 1u : 0u;
  }
  __syncthreads();
  const int M = p.M, q = tid >> 2;  // quad q: block b0 + q / M, activation row q % M
  if (q >= nb * M) return;           // whole quads
  const int i = q / M, m = q - i * M;
  if (closes[i] == 0u) return;
  const int b = b0 + i;
  const float* src = p.h + static_cast<int64_t>(m) * N + 32 * b + 8 * (tid & 3);
  float v[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) v[k] = __hip_atomic_load(src + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  store_q8_quarter(p.hq + static_cast<int64_t>(m) * (N / 32) + b, static_cast<uint32_t>(tid & 3),
                   quantize_quarter(v));
}

// A workgroup's path: prefetch, activations into LDS, stream, totals.
template <int TYPE, int MODE, bool Q8IN>
__device__ __forceinline__ void bmv_body(const BmvParams& p, const BmvShare& sh, int rows_seg,
                                         float* yout, int groups_max, unsigned char* lds_raw) {
  constexpr int B = TYPE == QK_TYPE_Q4_K ? kQ4KBytes : kQ6KBytes;
  constexpr bool kSlots = TYPE == QK_TYPE_Q6_K && MODE == 0;
  constexpr int P = TYPE == QK_TYPE_Q4_K ? kBmvP4 : kSlots ? kBmvSlotP : kBmvP6;
  constexpr int kParts = MODE == 1 ? 2 : 1;
  constexpr int kThreads = 64 * kBmvWaves;
  const int K = p.K, M = p.M, stride = p.stride;
  const int tid = static_cast<int>(threadIdx.x);
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // activations: the first tasks (8 fp32 values) or Q8 blocks per lane load
  // ahead of the weights
  const int groups8 = K / 8, tasks = M * groups8;
  const int bpr = K / 32, nblocks = M * bpr;
  f32x4 xa[Q8IN ? 1 : kBmvXStaged], xb[Q8IN ? 1 : kBmvXStaged];
  u32x4 qa[Q8IN ? kBmvQ8Staged : 1], qb[Q8IN ? kBmvQ8Staged : 1], qr[Q8IN ? kBmvQ8Staged : 1];
  auto load_blocks = [&](int first) {
    const u32x4* src = reinterpret_cast<const u32x4*>(p.q8);
#pragma unroll
    for (int i = 0; i < kBmvQ8Staged; ++i) {
      const int b = min(first + kThreads * i, nblocks - 1);
      qa[i] = src[3 * b];
      qb[i] = src[3 * b + 1];
      qr[i] = src[3 * b + 2];
    }
  };
  auto load_tasks = [&](int first) {
#pragma unroll
    for (int i = 0; i < kBmvXStaged; ++i)
      load_x_group(p.x, M, K, min(first + kThreads * i, tasks - 1), xa[i], xb[i]);
  };
  if constexpr (Q8IN)
    load_blocks(tid);
  else
    load_tasks(tid);
  __builtin_amdgcn_sched_barrier(0);

  // this wave's units [u_lo, u_hi) and its tile count
  const int units = kParts * sh.groups * sh.ranges;
  const int u_lo = units * wave / kBmvWaves, u_hi = units * (wave + 1) / kBmvWaves;
  int ntiles = 0;
  for (int u = u_lo; u < u_hi; ++u) {
    const int rr = u % sh.ranges;
    ntiles += sh.run_begin(rr + 1) - sh.run_begin(rr);
  }
  BmvCursor start;
  cursor_seek(start, sh, u_lo < u_hi ? u_lo : 0);
  start.left = ntiles;

  const BmvLane L = bmv_lane(lane, stride);

  // the first P tiles
  BmvTile<TYPE> buf[kSlots ? 1 : P];
  u32x4 chunk[kSlots ? P : 1][kBmvSlotLoads];
  BmvCursor lc = start;
  // slots: this lane's chunks c = lane + 64 j (clamped to the share's last) of
  // a tile, chunk c % 14 of row c / 14; loads through a descriptor that ends
  // at the dword boundary at or above the matrix end (dwords past it are zero)
  uint32_t base[kBmvSlotLoads], q16[kBmvSlotLoads];
  const int nchunks = kBmvSlotChunks * sh.nrows;
  const uint32_t end4 = (static_cast<uint32_t>(rows_seg) * static_cast<uint32_t>(sh.row_bytes) + 3u) & ~3u;
  const __amdgpu_buffer_rsrc_t rsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(sh.w[0]), 0, static_cast<int>(end4), 0x00020000);
  auto issue = [&](u32x4 (&to)[kBmvSlotLoads], int s) {
#pragma unroll
    for (int j = 0; j < kBmvSlotLoads; ++j)
      to[j] = __builtin_amdgcn_raw_buffer_load_b128(
          rsrc, static_cast<int>(((base[j] + static_cast<uint32_t>(s * B)) & ~3u) + q16[j]), 0, 0);
  };
  if constexpr (kSlots) {
#pragma unroll
    for (int j = 0; j < kBmvSlotLoads; ++j) {
      const int c = min(lane + 64 * j, nchunks - 1), row = c / kBmvSlotChunks;
      base[j] = static_cast<uint32_t>(sh.r0 + row) * static_cast<uint32_t>(sh.row_bytes);
      q16[j] = 16u * static_cast<uint32_t>(c - kBmvSlotChunks * row);
    }
  }
#pragma unroll
  for (int j = 0; j < P; ++j) {
    if constexpr (kSlots)
      issue(chunk[j], lc.s);
    else
      bmv_load(buf[j], bmv_sb<B>(sh, lc, L.n), L.kq);
    cursor_next(lc, sh);
  }
  __builtin_amdgcn_sched_barrier(0);

  lds_u8* codes = (lds_u8*)(lds_raw);
  lds_f32* xs = (lds_f32*)(lds_raw + bmv_lds_z(stride));
  lds_f32* xss = xs + K / 4;
  lds_f32* xf = xs + K / 2;
  lds_f32* sums = xs + K;
  // the staged round, then (wide rows) one round after another
  if constexpr (Q8IN) {
    for (int b0 = tid; b0 < nblocks; b0 += kThreads * kBmvQ8Staged) {
      if (b0 != tid) load_blocks(b0);
#pragma unroll
      for (int i = 0; i < kBmvQ8Staged; ++i) {
        const int b = b0 + kThreads * i;
        if (b < nblocks) bmv_store_block(qa[i], qb[i], qr[i], b, bpr, stride, codes, xs, xss, xf);
      }
    }
  } else {
    for (int t0 = tid; t0 < tasks; t0 += kThreads * kBmvXStaged) {
      if (t0 != tid) load_tasks(t0);
#pragma unroll
      for (int i = 0; i < kBmvXStaged; ++i) {
        const int t = t0 + kThreads * i;
        if (t < tasks) bmv_quantize_task(xa[i], xb[i], t, groups8, stride, codes, xs, xss, xf);
      }
    }
  }
  if (tid == 0) *reinterpret_cast<lds_u32x4*>(codes + 8 * stride) = u32x4{0u, 0u, 0u, 0u};
  __syncthreads();

  auto stream = [&](auto mh) {
    constexpr int MH = decltype(mh)::value;
    if constexpr (kSlots) {
      lds_u8* slot = (lds_u8*)(sums) + groups_max * 16 * sh.ranges * 32 + wave * bmv_slot_bytes(p.rows_max);
      const int n = min(L.n, sh.nrows - 1);  // rows past the share redo its last one and are not stored
      const lds_u8* row = slot + bmv_slot_bytes(n);
      BmvCursor cc = start;
      f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
      const int ntiles = cc.left;
      for (int t0 = 0; t0 < ntiles; t0 += P) {
#pragma unroll
        for (int j = 0; j < P; ++j) {
          if (t0 + j < ntiles) {
#pragma unroll
            for (int i = 0; i < kBmvSlotLoads; ++i)
              *reinterpret_cast<lds_u32x4*>(slot + 16 * min(lane + 64 * i, nchunks - 1)) = chunk[j][i];
            asm volatile("" ::: "memory");  // (a wave's LDS accesses keep their order)
            const uint32_t first = static_cast<uint32_t>(sh.r0 + n) * static_cast<uint32_t>(sh.row_bytes);
            ws_tile6<MH>(row + ((first + static_cast<uint32_t>(cc.s * B)) & 3u), cc.s, L, codes, xs, xf, acc);
            asm volatile("" ::: "memory");  // the next tile's slot writes follow these reads
            if (cc.s + 1 == cc.s_end) {
              bmv_flush<TYPE, MH>(acc, cc, L, groups_max, sh.ranges, sums);
              acc = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            }
            cursor_next(cc, sh);
          }
          issue(chunk[j], lc.s);  // P tiles ahead (past the end: the last tile again)
          cursor_next(lc, sh);
        }
      }
    } else {
      bmv_stream<TYPE, P, MH>(sh, lc, L, stride, groups_max, codes, xs, xss, xf, sums, buf, start);
    }
  };
  if (TYPE == QK_TYPE_Q4_K || M <= 4)
    stream(std::integral_constant<int, 1>{});
  else
    stream(std::integral_constant<int, 2>{});
  __syncthreads();

  // row totals: runs added in order; one thread per (activation row, row)
  const int nrows = sh.nrows, R = sh.ranges;
  for (int idx = tid; idx < nrows * M; idx += kThreads) {
    const int m = idx / nrows, row = idx - m * nrows;
    const lds_f32* pa = sums + ((row >> 4) * 16 + (row & 15)) * R * 8 + m;
    float a = 0.0f;
    for (int rr = 0; rr < R; ++rr) a += pa[rr * 8];
    if constexpr (MODE == 0) {
      yout[static_cast<int64_t>(m) * rows_seg + sh.r0 + row] = a;
    } else {
      const lds_f32* pb = pa + groups_max * 16 * R * 8;
      float b = 0.0f;
      for (int rr = 0; rr < R; ++rr) b += pb[rr * 8];
      float* dst = p.h + static_cast<int64_t>(m) * rows_seg + sh.r0 + row;
      const float hv = (a / (1.0f + expf(-a))) * b;
      if (p.hq != nullptr)  // read back by the workgroup that completes the block
        __hip_atomic_store(dst, hv, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      else
        *dst = hv;
    }
  }
  if constexpr (MODE == 1) {
    if (p.hq != nullptr) bmv_close_blocks(p, sh, rows_seg, lds_raw);
  }
}

// TYPE: the type of the matrix (mode 1: of gate and up), or 0 for a launch of
// several matrices, where each workgroup takes its matrix's. (The other
// launches read their two segments' arguments only: with all four read in
// the prologue the FFN block at M = 8 took 0.8 us longer.)
template <int TYPE, int MODE, bool Q8IN>
__global__ __launch_bounds__(64 * kBmvWaves) void bmv_kernel(const BmvParams p) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
#pragma unroll
  for (int j = 0; j < (TYPE == 0 ? kMaxSegments : MODE + 1); ++j)
    asm volatile("" ::"s"(p.seg[j].w), "s"(p.seg[j].y), "s"(p.seg[j].rows), "s"(p.seg[j].type),
                 "s"(p.seg[j].wg_begin), "s"(p.seg[j].per), "s"(p.seg[j].rem), "s"(p.seg[j].pad));
  asm volatile("" ::"s"(p.x), "s"(p.q8), "s"(p.h), "s"(p.hq), "s"(p.arrive), "s"(p.M), "s"(p.K), "s"(p.S),
               "s"(p.stride), "s"(p.ranges), "s"(p.groups_max), "s"(p.rows_max), "s"(p.nseg));
  __builtin_amdgcn_sched_barrier(0);
  const int wg = static_cast<int>(blockIdx.x), nseg = TYPE == 0 ? p.nseg : 1;
  const int j = (nseg > 1 && wg >= p.seg[1].wg_begin) + (nseg > 2 && wg >= p.seg[2].wg_begin) +
                (nseg > 3 && wg >= p.seg[3].wg_begin);
  auto pick = [j](auto f0, auto f1, auto f2, auto f3) {
    if constexpr (TYPE != 0) return f0;
    return j == 0 ? f0 : j == 1 ? f1 : j == 2 ? f2 : f3;
  };
  const int g = wg - pick(p.seg[0].wg_begin, p.seg[1].wg_begin, p.seg[2].wg_begin, p.seg[3].wg_begin);
  const int per = pick(p.seg[0].per, p.seg[1].per, p.seg[2].per, p.seg[3].per);
  const int rem = pick(p.seg[0].rem, p.seg[1].rem, p.seg[2].rem, p.seg[3].rem);
  const int rows = pick(p.seg[0].rows, p.seg[1].rows, p.seg[2].rows, p.seg[3].rows);
  float* const yout = pick(p.seg[0].y, p.seg[1].y, p.seg[2].y, p.seg[3].y);
  BmvShare sh;
  sh.w[0] = pick(p.seg[0].w, p.seg[1].w, p.seg[2].w, p.seg[3].w);
  sh.w[1] = MODE == 1 ? p.seg[1].w : sh.w[0];
  sh.r0 = g * per + min(g, rem);
  sh.nrows = per + (g < rem ? 1 : 0);
  sh.per = per;
  sh.rem = rem;
  sh.groups = (sh.nrows + 15) >> 4;
  sh.S = p.S;
  sh.ranges = p.ranges;
  sh.run_q = p.S / p.ranges;
  sh.run_r = p.S - sh.run_q * p.ranges;
  if (TYPE == QK_TYPE_Q4_K ||
      (TYPE == 0 && pick(p.seg[0].type, p.seg[1].type, p.seg[2].type, p.seg[3].type) == QK_TYPE_Q4_K)) {
    if constexpr (TYPE != QK_TYPE_Q6_K) {
      sh.row_bytes = p.S * kQ4KBytes;
      bmv_body<QK_TYPE_Q4_K, MODE, Q8IN>(p, sh, rows, yout, p.groups_max, lds_raw);
    }
  } else if constexpr (TYPE != QK_TYPE_Q4_K) {
    sh.row_bytes = p.S * kQ6KBytes;
    bmv_body<QK_TYPE_Q6_K, MODE, Q8IN>(p, sh, rows, yout, p.groups_max, lds_raw);
  }
}

using BmvKernel = void (*)(BmvParams);

BmvKernel bmv_kernel_for(int type, int mode, bool q8) {
  if (type == 0) return q8 || mode == 1 ? nullptr : &bmv_kernel<0, 0, false>;
  if (mode == 1) return type == QK_TYPE_Q4_K ? &bmv_kernel<QK_TYPE_Q4_K, 1, false> : &bmv_kernel<QK_TYPE_Q6_K, 1, false>;
  if (type == QK_TYPE_Q4_K) return q8 ? &bmv_kernel<QK_TYPE_Q4_K, 0, true> : &bmv_kernel<QK_TYPE_Q4_K, 0, false>;
  return q8 ? &bmv_kernel<QK_TYPE_Q6_K, 0, true> : &bmv_kernel<QK_TYPE_Q6_K, 0, false>;
}

}  // namespace

// Tiles on the busiest wave when `rows` rows (parts of them each) are cut
// into groups of 16 and each group's S superblocks into `ranges` runs, and
// the units are dealt to kBmvWaves waves in contiguous blocks.
int64_t bmv_wave_tiles(int64_t rows, int parts, int S, int ranges) {
  if (rows <= 0) return 0;
  const int64_t groups = (rows + 15) / 16;
  const int64_t units = parts * groups * ranges;
  const int64_t per_wave = (units + kBmvWaves - 1) / kBmvWaves;
  return per_wave * ((S + ranges - 1) / ranges);
}

struct BmvPlan {
  int count[kMaxSegments] = {0};
  int ranges = 0, groups_max = 0, lds = 0;
  int rows_max = 0;       // of the largest share (with slots: of the largest that goes through them)
  int64_t tiles = 0;      // on the busiest wave
  int64_t all_tiles = 0;  // the same if LDS held the sums of any number of runs
};

// The workgroups of each matrix and the run split of a launch (the CPU index
// model of the tests restates these rules). One matrix, or gate and up, over
// every CU; several matrices: at most kBmvMaxGroups row groups of 16 a
// workgroup (Q6_K: one of at most kBmvSlotRows rows, through the slots), the
// fewest that fit the CUs, what is left in proportion to the bytes. Returns
// false when the shape does not fit.
bool bmv_plan(const MatvecParams& p, int mode, int cus, int max_lds, BmvPlan& plan) {
  int(&count)[kMaxSegments] = plan.count;
  const int parts = mode == 1 ? 2 : 1, nseg = mode == 1 ? 1 : p.nseg;
  bool slots = false;
  if (nseg == 1) {
    count[0] = std::clamp(cus, 1, p.seg[0].rows);
    slots = mode == 0 && p.seg[0].type == QK_TYPE_Q6_K;
  } else {
    int sum = cus + 1;
    for (int groups = 1; groups <= kBmvMaxGroups && sum > cus; ++groups) {
      sum = 0;
      for (int j = 0; j < nseg; ++j) {
        const int rows = p.seg[j].type == QK_TYPE_Q6_K ? kBmvSlotRows : 16 * groups;
        count[j] = p.seg[j].rows / rows + (p.seg[j].rows % rows != 0);
        sum += count[j];
      }
    }
    if (sum > cus) return false;
    double bytes[kMaxSegments] = {0.0}, total = 0.0;
    for (int j = 0; j < nseg; ++j) {
      slots = slots || p.seg[j].type == QK_TYPE_Q6_K;
      bytes[j] = static_cast<double>(p.seg[j].rows) * (p.seg[j].type == QK_TYPE_Q4_K ? kQ4KBytes : kQ6KBytes);
      total += bytes[j];
    }
    const int left = cus - sum;
    for (int j = 0; j < nseg; ++j)
      count[j] = std::min(p.seg[j].rows, count[j] + static_cast<int>(left * bytes[j] / total));
  }
  int rows_max = 0, slot_rows = 0;
  for (int j = 0; j < nseg; ++j) {
    const int rows = p.seg[j].rows / count[j] + (p.seg[j].rows % count[j] != 0);
    rows_max = std::max(rows_max, rows);
    if (mode == 0 && p.seg[j].type == QK_TYPE_Q6_K) {
      slot_rows = std::max(slot_rows, rows);
      if (rows > kBmvSlotRows || static_cast<int64_t>(p.seg[j].rows) * p.S * kQ6KBytes + 16 > INT32_MAX) return false;
    }
  }
  plan.groups_max = (rows_max + 15) / 16;
  plan.rows_max = slots ? slot_rows : rows_max;
  const int stride = p.K + 16, slot_bytes = slots ? kBmvWaves * bmv_slot_bytes(slot_rows) : 0;
  // runs per group: the fewest tiles on the busiest wave of any workgroup,
  // then the fewest units (each unit ends with a lane reduction)
  int64_t best = INT64_MAX;
  plan.all_tiles = INT64_MAX;
  for (int r = 1; r <= p.S; ++r) {
    const int lds = bmv_lds_bytes(p.K, stride, parts, plan.groups_max, r) + slot_bytes;
    const bool fits = lds <= max_lds;
    if (!fits && plan.ranges == 0) return false;
    int64_t tiles = 0, units = 0;
    for (int j = 0; j < nseg; ++j) {
      const int rows = p.seg[j].rows / count[j] + (p.seg[j].rows % count[j] != 0);
      tiles = std::max(tiles, bmv_wave_tiles(rows, parts, p.S, r));
      units = std::max<int64_t>(units, (parts * ((rows + 15) / 16) * r + kBmvWaves - 1) / kBmvWaves);
    }
    plan.all_tiles = std::min(plan.all_tiles, tiles);
    const int64_t cost = 8 * tiles + units;
    if (fits && cost < best) {
      best = cost;
      plan.ranges = r;
      plan.tiles = tiles;
      plan.lds = lds;
    }
  }
  return true;
}

// Where a launch of mode 0 pays: measured on MI355X against the streaming and
// per-row kernels, graphs over weights out of cache, 3,400 launches of M = 2..8,
// 256 to 16384 columns, 16 to 8192 rows, one to three matrices; none that is
// taken is more than 3% slower. us, the other kernel -> this one:
//  - one Q4_K matrix from M = 3 (9728 -> 2560 at M = 3 / 8 13.2 / 22.2 -> 9.5 /
//    14.6; at M = 2 9.2 -> 9.5), at M = 2 up to K = 8192 (the streaming kernel, which
//    the quantiser's registers slowed there: 7936 -> 2560 10.65 -> 7.7).
//  - one Q6_K matrix from M = 5 (9728 -> 2560 at M = 8 22.4 -> 17.9), at M = 8, and
//    at M = 7 up to K = 8192, above 3 rows a CU (5120 -> 256 10.5 -> 11.2). At M = 3 and 4 while K <=
//    8192, where the streaming kernel would run (6400 -> 256 9.7 -> 7.9), or
//    above 8 rows a CU (9728 -> 2560 at M = 3 13.1 -> 12.2): with fewer a tile is
//    mostly empty (9728 -> 256 9.6 -> 10.2).
//  - several matrices from 9 superblocks a row: below, the waves have a tile
//    each or none (2048 -> 4096 + 1024 + 1024 at M = 3 6.9 -> 8.0). From M = 5 all
//    of these (2560 -> 4096 + 1024 + 1024 at M = 8 11.8 -> 8.4). At M = 2..4 not
//    both types, nor over 20 rows a CU (24 at K = 4096), where 8 divides the
//    superblocks and the others idle no lanes (6144 -> 4096 + 4064 at M = 3 12.9
//    -> 14.3; 6400 0.88 times the time); all Q4_K from M = 3, at M = 2 up to K =
//    6400, 8192 with at most 16 rows a CU (8192 -> 4096 + 1024 + 1024 10.6 ->
//    13.1, 2048 + 512 + 512 10.6 -> 9.0); with Q6_K from M = 3 as one matrix of
//    it, with both types only above 8 rows a CU (4352 -> 4096 + 1024 + 1024 0.89
//    times the time, 1024 + 256 + 256 1.04), 16 below K = 3328 (2560 -> 2048 + 1024
//    + 1024 1.04).
bool bmv_pays(const MatvecParams& p, int cus) {
  int64_t rows = 0;
  bool q4 = false, q6 = false;
  for (int j = 0; j < p.nseg; ++j) {
    rows += p.seg[j].rows;
    (p.seg[j].type == QK_TYPE_Q4_K ? q4 : q6) = true;
  }
  const bool full = rows > 8 * cus;
  if (p.nseg == 1) {
    if (q4) return p.M >= 3 || p.K <= 8192;
    if (p.M < 3) return false;
    if (p.M <= 4) return p.K <= 8192 || full;
    return p.M <= 6 || rows > 3 * cus || (p.M == 7 && p.K > 8192);
  }
  if (p.S < 9 || p.M >= 5) return p.S >= 9;
  if (p.S % 8 == 0 && ((q4 && q6) || rows > (p.K <= 4096 ? 24 : 20) * cus)) return false;
  if (!q6) return p.M >= 3 || p.K <= (rows > 16 * cus ? 6400 : 8192);
  if (q4) return p.M >= 3 && rows > (p.K < 3328 ? 16 : 8) * cus;
  return p.M >= 3 && (full || p.K <= 8192);
}

hipError_t launch_bmv(const MatvecParams& p, int mode, hipStream_t stream, bool& launched) {
  launched = false;
  if (p.M < 2 || p.M > 8 || (mode != 0 && mode != 1)) return hipSuccess;
  if (mode == 1 ? p.x == nullptr || p.nseg != 2 : p.nseg > 1 && p.x == nullptr) return hipSuccess;
  if (p.K > INT32_MAX / 16) return hipSuccess;  // (the LDS plan counts in 32 bits)
  int cus = 0, max_lds = 0;
  hipError_t e = device_limits(cus, max_lds);
  if (e != hipSuccess) return e;
  if (mode == 0 && !bmv_pays(p, cus)) return hipSuccess;
  BmvPlan plan;
  if (!bmv_plan(p, mode, cus, max_lds, plan)) return hipSuccess;
  if (mode == 0 && p.nseg == 1 && plan.groups_max > 1) return hipSuccess;
  // Runs that LDS has no room for leave waves idle: at M <= 4 the other kernels
  // win as soon as the busiest wave has a tile more (Q6_K 10240 -> 2560, 5 tiles
  // for 3, M = 4 1.12 times the time), at M >= 5 past twice its tiles (5 for 3
  // 0.90 times at M = 8; 12288 -> 1024, 16 for 3, 20.7 -> 34.0 us).
  if (mode == 0 && plan.tiles > (p.M <= 4 ? 1 : 2) * plan.all_tiles) return hipSuccess;
  if (p.hq != nullptr) {  // Q8(h) in the launch: a quad per (block, activation row) of a share
    const int64_t rows_max = (p.seg[0].rows + plan.count[0] - 1) / plan.count[0];
    const int64_t blocks = (rows_max + 30) / 32 + 1;  // blocks a run of rows_max rows can touch
    if (p.seg[0].rows % 32 != 0 || blocks > kBmvMaxCloseBlocks || 4 * blocks * p.M > 64 * kBmvWaves ||
        p.arrive == nullptr)
      return hipSuccess;
  }

  BmvParams bp{};
  bp.x = p.x;
  bp.q8 = p.x == nullptr ? p.q8 : nullptr;
  bp.h = p.h;
  bp.hq = p.hq;
  bp.arrive = p.hq != nullptr ? p.arrive : nullptr;
  bp.M = p.M;
  bp.K = p.K;
  bp.S = p.S;
  bp.stride = p.K + 16;
  bp.ranges = plan.ranges;
  bp.groups_max = plan.groups_max;
  bp.rows_max = plan.rows_max;
  bp.nseg = p.nseg;
  int begin = 0;
  for (int j = 0; j < p.nseg; ++j) {
    const int c = mode == 1 ? plan.count[0] : plan.count[j];
    bp.seg[j] = {p.seg[j].w, p.seg[j].y, p.seg[j].rows, p.seg[j].type, begin, p.seg[j].rows / c, p.seg[j].rows % c, 0};
    if (mode == 0 || j == 0) begin += c;
  }
  const int type = mode == 0 && p.nseg > 1 ? 0 : p.seg[0].type;
  const BmvKernel fn = bmv_kernel_for(type, mode, p.x == nullptr);
  if (!fn) return hipSuccess;
  e = allow_lds(reinterpret_cast<const void*>(fn), plan.lds);
  if (e != hipSuccess) return e;
  note("bmv_kernel", begin, type, mode, plan.ranges, plan.groups_max, p.hq != nullptr);
  hipLaunchKernelGGL(fn, dim3(static_cast<uint32_t>(begin)), dim3(64 * kBmvWaves),
                     static_cast<size_t>(plan.lds), stream, bp);
  launched = true;
  return hipGetLastError();
}

}  // namespace qk
