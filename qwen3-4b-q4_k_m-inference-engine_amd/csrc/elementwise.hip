// out = gate/(1+exp(-gate)) * up (src/cuda/silu_multiply.cu:6-12), with the
// ROCm device library's expf; the row-wise RMSNorm (src/cuda/rms_norm.cu:6-24)
// with its rsqrtf; and state += branch (src/cuda/residual_add.cu:6-9).
#include "qk_device.hpp"
#include "qk_launch.hpp"

namespace qk {
namespace {

// 16-byte accesses (rows and tensors are only float-aligned: gfx950 takes
// dword-aligned 16-byte global accesses); the last count % 4 elements go one
// a lane.
__global__ __launch_bounds__(256) void silu_multiply_kernel(const float* __restrict__ gate,
                                                            const float* __restrict__ up,
                                                            float* __restrict__ out,
                                                            int64_t count) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * 256;
  const int64_t first = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int64_t quads = count / 4;
  auto one = [](float g, float u) { return (g / (1.0f + expf(-g))) * u; };
  for (int64_t i = first; i < quads; i += stride) {
    const f32x4 g = *reinterpret_cast<const f32x4_a4*>(gate + 4 * i);
    const f32x4 u = *reinterpret_cast<const f32x4_a4*>(up + 4 * i);
    *reinterpret_cast<f32x4_a4*>(out + 4 * i) = f32x4{one(g.x, u.x), one(g.y, u.y), one(g.z, u.z), one(g.w, u.w)};
  }
  if (first < count - 4 * quads) {
    const int64_t i = 4 * quads + first;
    out[i] = one(gate[i], up[i]);
  }
}

// The sum of the workgroup's four waves' `sum`, in every thread. Lane bits
// 5, 4, .. 0 in turn (row rotations stand for the exchanges of bits 3 to 0:
// lanes that differ only in bits already added hold the same sum).
__device__ __forceinline__ float workgroup_sum(float sum, float (&partial)[4]) {
  sum = swap16_sum(swap32_sum(sum));
  sum = add_dpp<0x121>(add_dpp<0x122>(add_dpp<0x124>(add_dpp<0x128>(sum))));
  if ((threadIdx.x & 63) == 0) partial[threadIdx.x >> 6] = sum;
  __syncthreads();
  return (partial[0] + partial[1]) + (partial[2] + partial[3]);
}

// out = x * rsqrt(mean(x^2) + eps) * scale for one row per workgroup (the
// mat-vec's RMSNorm fold does the same inside its prologue at M = 1). A few
// rows are bound by latency alone, so a row of at most 256 R values stays in
// registers: its loads and those of the scale are all issued at entry, and
// the row is read once: 8 / 2047 rows of 2560 in 2.30 / 6.64 us against 3.98 /
// 10.09 with the row read twice (a launch of 40 in a graph). Thread t adds
// values t, t + 256, .. in order, as the form below does: the sum's last bit
// reaches Q8 codes near a tie, so every width keeps one order of its sums
// (four neighbours a thread and load: 2.15 / 6.63 us, and other codes).
template <int R>
__global__ __launch_bounds__(256) void rms_norm_row_kernel(const float* __restrict__ x,
                                                           const float* __restrict__ scale,
                                                           float* __restrict__ out, int width,
                                                           float eps) {
  __shared__ float partial[4];
  const int64_t row = static_cast<int64_t>(blockIdx.x) * width;
  const int tid = static_cast<int>(threadIdx.x);
  float v[R], s[R];
#pragma unroll
  for (int i = 0; i < R; ++i) {  // loads past the row re-read its last value
    const int at = min(tid + 256 * i, width - 1);
    v[i] = x[row + at];
    s[i] = scale[at];
  }
  float sum = 0.0f;
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const float t = tid + 256 * i < width ? v[i] : 0.0f;
    sum = __builtin_fmaf(t, t, sum);
  }
  const float inv = rsqrtf(workgroup_sum(sum, partial) / static_cast<float>(width) + eps);
#pragma unroll
  for (int i = 0; i < R; ++i)
    if (tid + 256 * i < width) out[row + tid + 256 * i] = (v[i] * inv) * s[i];
}

// Wider rows: two passes over the row.
__global__ __launch_bounds__(256) void rms_norm_kernel(const float* __restrict__ x,
                                                       const float* __restrict__ scale,
                                                       float* __restrict__ out, int width,
                                                       float eps) {
  __shared__ float partial[4];
  const float* xr = x + static_cast<int64_t>(blockIdx.x) * width;
  float* o = out + static_cast<int64_t>(blockIdx.x) * width;
  const int tid = static_cast<int>(threadIdx.x);
  float sum = 0.0f;
  for (int i = tid; i < width; i += 256) sum = __builtin_fmaf(xr[i], xr[i], sum);
  const float inv = rsqrtf(workgroup_sum(sum, partial) / static_cast<float>(width) + eps);
  for (int i = tid; i < width; i += 256) o[i] = (xr[i] * inv) * scale[i];
}

__global__ __launch_bounds__(256) void residual_add_kernel(float* __restrict__ state,
                                                           const float* __restrict__ branch,
                                                           int64_t count) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * 256;
  const int64_t first = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int64_t quads = count / 4;
  for (int64_t i = first; i < quads; i += stride) {
    f32x4_a4* s = reinterpret_cast<f32x4_a4*>(state + 4 * i);
    *s = *s + *reinterpret_cast<const f32x4_a4*>(branch + 4 * i);
  }
  if (first < count - 4 * quads) state[4 * quads + first] += branch[4 * quads + first];
}

// Workgroups of an elementwise launch over `count` values, four a thread.
uint32_t elementwise_grid(int64_t count) {
  const int64_t blocks = (count + 1023) / 1024;
  return static_cast<uint32_t>(blocks < 16384 ? blocks : 16384);
}

}  // namespace

hipError_t launch_residual_add(float* state, const float* branch, int64_t count,
                               hipStream_t stream) {
  residual_add_kernel<<<elementwise_grid(count), 256, 0, stream>>>(state, branch, count);
  return hipGetLastError();
}

hipError_t launch_rms_norm(const float* x, const float* scale, float* out, int64_t rows,
                           int64_t width, float eps, hipStream_t stream) {
  const dim3 grid(static_cast<uint32_t>(rows));
  const int w = static_cast<int>(width);
  // Up to 8192 values the one-pass form, in the least of these rounds.
  if (w <= 1024)
    rms_norm_row_kernel<4><<<grid, 256, 0, stream>>>(x, scale, out, w, eps);
  else if (w <= 2048)
    rms_norm_row_kernel<8><<<grid, 256, 0, stream>>>(x, scale, out, w, eps);
  else if (w <= 2560)
    rms_norm_row_kernel<10><<<grid, 256, 0, stream>>>(x, scale, out, w, eps);
  else if (w <= 4096)
    rms_norm_row_kernel<16><<<grid, 256, 0, stream>>>(x, scale, out, w, eps);
  else if (w <= 8192)
    rms_norm_row_kernel<32><<<grid, 256, 0, stream>>>(x, scale, out, w, eps);
  else
    rms_norm_kernel<<<grid, 256, 0, stream>>>(x, scale, out, w, eps);
  return hipGetLastError();
}

hipError_t launch_silu_multiply(const float* gate, const float* up, float* out, int64_t count,
                                hipStream_t stream) {
  silu_multiply_kernel<<<elementwise_grid(count), 256, 0, stream>>>(gate, up, out, count);
  return hipGetLastError();
}

}  // namespace qk
