// Backward of the RMSNorm / SubLN in front of a quantised linear (WF/models/subln.py:42-59), fp32 arithmetic:
//   y = x r w,  r = (mean(x^2) + eps)^(-1/2)
//   grad_x = r (g w) - x r^3 mean(g w x)
//   grad_w[h] = sum_m g[m, h] x[m, h] r[m]
// One pass over x and g (torch's composition of the same takes fifteen, each a launch).  A workgroup takes rows
// blockIdx.x, + gridDim.x, ...; a thread keeps its columns' part of grad_w in registers over all of them, and the
// row's elements between the two sums and the output, so every element is read once.  Bound by the two block
// reductions of a row at small M and by memory at large M: the next row's loads are requested before this row's
// reductions.  Against the torch composition, with the column sums: 501 x 1536 fp32 185 -> 11 us, 2048 x 2560 bf16 194
// -> 19 us, 8192 x 6912 bf16 1335 -> 139 us (3.3 TB/s).  Rows above 8192 hold 422 registers a thread, one workgroup per
// CU: 8192 x 14336 bf16 384 us (2.5 TB/s), fp32 289 (4.9), 501 x 14336 bf16 41.
#include "wfb_common.h"

namespace wfb {

namespace {

constexpr int kThreads = 256;

template <int DT>
__device__ __forceinline__ void load8_any(const void* p, int64_t i, bool vec, float (&v)[8]) {
  if (vec) {
    load8<DT>(p, i, v);
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = load_elem<DT>(p, i + e);
  }
}

// Sums of a and b over the workgroup, in every thread; `red` holds 2 x 4 floats and alternates between rows.
__device__ __forceinline__ void block_sum2(float& a, float& b, float (*red)[4]) {
  a = group_sum_f32<64>(a);
  b = group_sum_f32<64>(b);
  if ((threadIdx.x & 63) == 0) {
    red[0][threadIdx.x >> 6] = a;
    red[1][threadIdx.x >> 6] = b;
  }
  __syncthreads();
  a = (red[0][0] + red[0][1]) + (red[0][2] + red[0][3]);
  b = (red[1][0] + red[1][1]) + (red[1][2] + red[1][3]);
}

// VPT 8-element vectors per thread: vector t + 256 j, j < VPT (H <= 2048 VPT, a multiple of 8).
template <int DT, int VPT>
__global__ __launch_bounds__(kThreads) void norm_grad_kernel(const void* __restrict__ x, const void* __restrict__ w,
                                                             int wdt, const float* __restrict__ g, float eps, int M, int H,
                                                             bool vec, void* __restrict__ gx,
                                                             float* __restrict__ part) {
  __shared__ float red[2][2][4];
  const int t = threadIdx.x, nv = H / 8;
  float wv[VPT][8], gw[VPT][8], xv[VPT][8], gv[VPT][8];
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    const int v = t + kThreads * j;
#pragma unroll
    for (int e = 0; e < 8; ++e) gw[j][e] = 0.0f;
    if (v >= nv) continue;
    if (wdt == WFB_F32) load8_any<WFB_F32>(w, 8 * (int64_t)v, false, wv[j]);
    else if (wdt == WFB_BF16) load8_any<WFB_BF16>(w, 8 * (int64_t)v, false, wv[j]);
    else load8_any<WFB_F16>(w, 8 * (int64_t)v, false, wv[j]);
  }
  auto load_row = [&](int m) {
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
      const int v = t + kThreads * j;
      if (v < nv) {
        load8_any<DT>(x, (int64_t)m * H + 8 * v, vec, xv[j]);
        load8<WFB_F32>(g, (int64_t)m * H + 8 * v, gv[j]);
      }
    }
  };
  int buf = 0;
  if ((int)blockIdx.x < M) load_row(blockIdx.x);
  for (int m = blockIdx.x; m < M; m += gridDim.x, buf ^= 1) {
    float ss = 0.0f, sd = 0.0f;
    float xr[VPT][8], gr[VPT][8];
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
      if (t + kThreads * j >= nv) continue;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        xr[j][e] = xv[j][e];
        gr[j][e] = gv[j][e];
        ss += xr[j][e] * xr[j][e];
        sd += gr[j][e] * wv[j][e] * xr[j][e];
      }
    }
    if (m + (int)gridDim.x < M) load_row(m + gridDim.x);
    block_sum2(ss, sd, red[buf]);
    const float r = 1.0f / sqrtf(ss / (float)H + eps);
    const float c = r * r * r * (sd / (float)H);
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
      const int v = t + kThreads * j;
      if (v >= nv) continue;
      float y[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        y[e] = r * (gr[j][e] * wv[j][e]) - xr[j][e] * c;
        gw[j][e] += gr[j][e] * (xr[j][e] * r);
      }
      if (!gx) continue;
      const int64_t off = (int64_t)m * H + 8 * v;  // gx is 16-byte aligned (host-checked)
      if constexpr (DT == WFB_F32) {
        float4* o = reinterpret_cast<float4*>(reinterpret_cast<float*>(gx) + off);
        o[0] = make_float4(y[0], y[1], y[2], y[3]);
        o[1] = make_float4(y[4], y[5], y[6], y[7]);
      } else {
        union { uint16_t h[8]; uint4 q; } o;
#pragma unroll
        for (int e = 0; e < 8; ++e)
          o.h[e] = DT == WFB_BF16 ? f32_to_bf16_rne(y[e]) : __builtin_bit_cast(uint16_t, (_Float16)y[e]);
        *reinterpret_cast<uint4*>(reinterpret_cast<uint16_t*>(gx) + off) = o.q;
      }
    }
  }
  if (!part) return;
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    const int v = t + kThreads * j;
    if (v >= nv) continue;
    float4* o = reinterpret_cast<float4*>(part + (int64_t)blockIdx.x * H + 8 * v);
    o[0] = make_float4(gw[j][0], gw[j][1], gw[j][2], gw[j][3]);
    o[1] = make_float4(gw[j][4], gw[j][5], gw[j][6], gw[j][7]);
  }
}

template <int DT>
hipError_t launch_t(const void* x, const void* w, int wdt, const float* g, float eps, int m, int h, void* gx,
                    float* part, int grid, hipStream_t s) {
  const bool vec = (uintptr_t)x % 16 == 0;
#define WFB_NG(V)                                                                                                \
  hipLaunchKernelGGL((norm_grad_kernel<DT, V>), dim3(grid), dim3(kThreads), 0, s, x, w, wdt, g, eps, m, h, vec, gx, \
                     part)
  if (h <= 2048) WFB_NG(1);
  else if (h <= 4096) WFB_NG(2);
  else if (h <= 8192) WFB_NG(4);
  else WFB_NG(8);
#undef WFB_NG
  return hipGetLastError();
}

// out[c] = sum over the rows of part[rows][cols], in a fixed order: 16 rows of threads each take every 16th row,
// 8 loads in flight, then a tree.  16 x 16 threads: 16 columns per workgroup.
__global__ __launch_bounds__(256) void column_sum_kernel(const float* __restrict__ part, int rows, int64_t cols,
                                                         void* __restrict__ out, int out_dtype) {
  __shared__ float red[16][17];
  const int c = threadIdx.x & 15, r = threadIdx.x >> 4;
  const int64_t col = (int64_t)blockIdx.x * 16 + c, cc = col < cols ? col : cols - 1;
  float acc = 0.0f;
  for (int i = r; i < rows; i += 16 * 8) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int j = i + 16 * u;
      v[u] = part[(int64_t)(j < rows ? j : rows - 1) * cols + cc];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) acc += i + 16 * u < rows ? v[u] : 0.0f;
  }
  red[r][c] = acc;
  __syncthreads();
#pragma unroll
  for (int o = 8; o >= 1; o >>= 1) {
    if (r < o) red[r][c] += red[r + o][c];
    __syncthreads();
  }
  if (r != 0 || col >= cols) return;
  const float y = red[0][c];
  if (out_dtype == WFB_F32) reinterpret_cast<float*>(out)[col] = y;
  else if (out_dtype == WFB_BF16) reinterpret_cast<uint16_t*>(out)[col] = f32_to_bf16_rne(y);
  else reinterpret_cast<uint16_t*>(out)[col] = __builtin_bit_cast(uint16_t, (_Float16)y);
}

}  // namespace

hipError_t launch_column_sum(const float* part, int rows, int64_t cols, void* out, int out_dtype, hipStream_t s) {
  hipLaunchKernelGGL(column_sum_kernel, dim3((unsigned)((cols + 15) / 16)), dim3(256), 0, s, part, rows, cols, out,
                     out_dtype);
  return hipGetLastError();
}

// 512 workgroups walk the rows, two per CU (one after the other where a row is longer than 8192); each leaves one row of
// partial sums.
int norm_grad_parts(int64_t m) { return (int)(m < 512 ? m : 512); }

hipError_t launch_norm_grad(const void* x, int dt, const void* w, int wdt, const float* g, float eps, int64_t m,
                            int64_t h, void* gx, void* gw, int gw_dtype, float* part, hipStream_t s) {
  const int grid = norm_grad_parts(m);
  float* pp = gw ? part : nullptr;
  hipError_t e;
  if (dt == WFB_F32) e = launch_t<WFB_F32>(x, w, wdt, g, eps, (int)m, (int)h, gx, pp, grid, s);
  else if (dt == WFB_BF16) e = launch_t<WFB_BF16>(x, w, wdt, g, eps, (int)m, (int)h, gx, pp, grid, s);
  else e = launch_t<WFB_F16>(x, w, wdt, g, eps, (int)m, (int)h, gx, pp, grid, s);
  if (e != hipSuccess || !gw) return e;
  return launch_column_sum(part, grid, h, gw, gw_dtype, s);
}

}  // namespace wfb
