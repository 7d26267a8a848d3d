// Offline weight pack on the device: per-tensor absmean scale and the I2_S 2-bit layout.
//
// Follows pack_ternary_sglkernel (packages/inference/scripts/convert_to_sglkernel.py:51-123):
//   s = mean(|W|) (s < 1e-8 -> 1.0), q = clamp(round_half_even(W / s), -1, 1), code = q + 1,
//   byte j of 128-weight block b = code[128b+j]<<6 | code[128b+32+j]<<4 | code[128b+64+j]<<2 | code[128b+96+j].
#include "wfb_common.h"

namespace wfb {

namespace {

constexpr int kAbsBlocks = WFB_ABSMEAN_WS_DOUBLES;

// Stage 1: block b sums |w| over the grid-stride set {i : i % (blocks*256) in block b's range},
// in fp64, each thread sequentially, then a fixed tree.  Deterministic for a given numel.
// Bound by how many loads are in flight (one dependent fp64 add per element hides none): a thread requests
// kAbsBatch elements before it adds the first, in the same order as one at a time, so the sum keeps its bits.
// The last elements are taken kAbsTail at a time from clamped indices, those past the end adding +0.0 (which
// leaves a non-negative sum as it is): a guard around each load would wait for each.  SMALL, up to
// two elements per thread: one at a time, clamped loads only add to them (64 x 4096 fp32, both stages, 5.6 -> 5.4 us).
// 14336 x 4096 fp32: 103 -> 42 us (5.6 TB/s), 6912 x 2560 bf16 21.9 -> 8.6 us (traced).
constexpr int kAbsBatch = 16, kAbsTail = 4;
constexpr int64_t kStride = (int64_t)kAbsBlocks * 256;

template <int DT, bool SMALL>
__global__ __launch_bounds__(256) void absmean_partial_kernel(const void* __restrict__ w, int64_t numel,
                                                              double* __restrict__ partial) {
  __shared__ double red[256];
  double acc = 0.0;
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if constexpr (SMALL) {
    for (; i < numel; i += kStride) acc += (double)fabsf(load_elem<DT>(w, i));
  } else {
    for (; i + (kAbsBatch - 1) * kStride < numel; i += kAbsBatch * kStride) {
      float v[kAbsBatch];
#pragma unroll
      for (int u = 0; u < kAbsBatch; ++u) v[u] = load_elem<DT>(w, i + u * kStride);
#pragma unroll
      for (int u = 0; u < kAbsBatch; ++u) acc += (double)fabsf(v[u]);
    }
    for (; i < numel; i += kAbsTail * kStride) {
      float v[kAbsTail];
#pragma unroll
      for (int u = 0; u < kAbsTail; ++u) {
        const int64_t j = i + u * kStride;
        v[u] = load_elem<DT>(w, j < numel ? j : numel - 1);
      }
#pragma unroll
      for (int u = 0; u < kAbsTail; ++u) acc += i + u * kStride < numel ? (double)fabsf(v[u]) : 0.0;
    }
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int o = 128; o >= 1; o >>= 1) {
    if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

__global__ __launch_bounds__(256) void absmean_final_kernel(const double* __restrict__ partial, int64_t numel,
                                                            float* __restrict__ scale) {
  __shared__ double red[256];
  double acc = 0.0;
  for (int i = threadIdx.x; i < kAbsBlocks; i += 256) acc += partial[i];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int o = 128; o >= 1; o >>= 1) {
    if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    float s = numel > 0 ? (float)(red[0] / (double)numel) : 0.0f;
    if ((double)s < 1e-8) s = 1.0f;
    scale[0] = s;
  }
}

// clamp(rint(w / s), -1, 1) + 1 of the correctly rounded quotient; NaN gives 0.
__device__ __forceinline__ uint32_t ternary_code(float w, float s) {
  float q = __builtin_rintf(__fdiv_rn(w, s));
  q = fminf(fmaxf(q, -1.0f), 1.0f);
  return (uint32_t)((int)q + 1);
}

// The same code for h = s / 2 of a finite s >= 2^-125 (h is exact then): rint gives 1 where the quotient rounds to more
// than 1/2, which is where w / s > 1/2 + 2^-25 (a tie goes to the even 1/2), that is w > h + h 2^-24 -- a bound within
// [h + ulp(h) / 2, h + ulp(h)), which the floats above h, and only they, exceed.  NaN fails both comparisons.
__device__ __forceinline__ uint32_t ternary_code_half(float w, float h) { return w > h ? 2u : w >= -h ? 1u : 0u; }

// One thread per output dword: bytes j..j+3 (j = 4*(p % 8)) of block b = p / 8 of row `row`.  A pass over the weights:
// with a division per weight and 64-bit index divisions per thread, 16-bit weights were bound by those (6912 x 2560
// bf16 13.0 us); with the comparisons and one uniform 64-bit division per workgroup 8.9.  fp32 weights are bound by the
// reads before and after (14336 x 4096 36.5 us, 6.4 TB/s).
template <int DT>
__global__ __launch_bounds__(256) void pack_i2s_kernel(const void* __restrict__ w, int64_t n, int64_t k,
                                                       int64_t ldw, const float* __restrict__ scale,
                                                       uint32_t* __restrict__ qw) {
  const int64_t dw_per_row = k / 16;
  const int64_t first = (int64_t)blockIdx.x * 256, row0 = first / dw_per_row;
  int64_t row = row0, p = first - row0 * dw_per_row + threadIdx.x;
  if (dw_per_row < 256) {  // rows end within the workgroup, more than once for the shortest
    row += (uint32_t)p / (uint32_t)dw_per_row;
    p = (uint32_t)p % (uint32_t)dw_per_row;
  } else if (p >= dw_per_row) {
    row += 1;
    p -= dw_per_row;
  }
  if (row >= n) return;
  const int64_t b = p >> 3;
  const int j = (int)(p & 7) * 4;
  const float s = scale[0];
  const bool plain = s >= 0x1p-125f && s <= 0x1.fffffep127f;
  const float h = 0.5f * s;
  const int64_t base = row * ldw + 128 * b + j;
  float v[4][4];
#pragma unroll
  for (int f = 0; f < 4; ++f)
#pragma unroll
    for (int t = 0; t < 4; ++t) v[f][t] = load_elem<DT>(w, base + 32 * f + t);
  uint32_t out = 0;
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int f = 0; f < 4; ++f)
      out |= (plain ? ternary_code_half(v[f][t], h) : ternary_code(v[f][t], s)) << (8 * t + 6 - 2 * f);
  qw[first + threadIdx.x] = out;
}

__global__ __launch_bounds__(256) void unpack_i2s_kernel(const uint8_t* __restrict__ qw, int64_t n, int64_t k,
                                                         int8_t* __restrict__ out) {
  const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;  // one packed byte
  const int64_t kb = k / 4;
  if (gid >= n * kb) return;
  const int64_t row = gid / kb, p = gid % kb;
  const int64_t b = p / 32;
  const int j = (int)(p % 32);
  const uint32_t byte = qw[gid];
  int8_t* o = out + row * k + 128 * b + j;
#pragma unroll
  for (int f = 0; f < 4; ++f) o[32 * f] = (int8_t)((int)((byte >> (6 - 2 * f)) & 3u) - 1);
}

template <int DT>
hipError_t absmean_t(const void* w, int64_t numel, float* scale, double* ws, hipStream_t s) {
  if (numel <= 2 * kStride)
    hipLaunchKernelGGL((absmean_partial_kernel<DT, true>), dim3(kAbsBlocks), dim3(256), 0, s, w, numel, ws);
  else
    hipLaunchKernelGGL((absmean_partial_kernel<DT, false>), dim3(kAbsBlocks), dim3(256), 0, s, w, numel, ws);
  hipLaunchKernelGGL(absmean_final_kernel, dim3(1), dim3(256), 0, s, ws, numel, scale);
  return hipGetLastError();
}

template <int DT>
hipError_t pack_t(const void* w, int64_t n, int64_t k, int64_t ldw, const float* scale, uint8_t* qw,
                  hipStream_t s) {
  const int64_t total = n * (k / 16);
  if (total == 0) return hipSuccess;
  hipLaunchKernelGGL((pack_i2s_kernel<DT>), dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, w, n, k, ldw,
                     scale, reinterpret_cast<uint32_t*>(qw));
  return hipGetLastError();
}

}  // namespace

hipError_t launch_weight_absmean(const void* w, int dt, int64_t numel, float* scale, double* ws, hipStream_t s) {
  if (dt == WFB_F32) return absmean_t<WFB_F32>(w, numel, scale, ws, s);
  if (dt == WFB_BF16) return absmean_t<WFB_BF16>(w, numel, scale, ws, s);
  return absmean_t<WFB_F16>(w, numel, scale, ws, s);
}

hipError_t launch_pack_i2s(const void* w, int dt, int64_t n, int64_t k, int64_t ldw, const float* scale,
                           uint8_t* qw, hipStream_t s) {
  if (dt == WFB_F32) return pack_t<WFB_F32>(w, n, k, ldw, scale, qw, s);
  if (dt == WFB_BF16) return pack_t<WFB_BF16>(w, n, k, ldw, scale, qw, s);
  return pack_t<WFB_F16>(w, n, k, ldw, scale, qw, s);
}

hipError_t launch_unpack_i2s(const uint8_t* qw, int64_t n, int64_t k, int8_t* out, hipStream_t s) {
  const int64_t total = n * (k / 4);
  if (total == 0) return hipSuccess;
  hipLaunchKernelGGL(unpack_i2s_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, qw, n, k, out);
  return hipGetLastError();
}

}  // namespace wfb
