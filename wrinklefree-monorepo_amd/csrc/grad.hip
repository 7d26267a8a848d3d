// Gradients of the ternary linear under the straight-through estimator, on the bf16 matrix cores.
//
// The reference trains F.linear(x + (q(x) - x).detach(), w + (q(w) - w).detach())
// (packages/training/src/wrinklefree/models/bitlinear.py:86-113), whose gradients are plain products with one
// exactly representable operand:
//   grad_x[m, k] = w_scale * sum_n g[m, n] * t[n, k]               t in {-1, 0, 1}
//   grad_w[n, k] = sum_m (g[m, n] * a_scale[m]) * q[m, k]          q an int8 code
// Both run as C[i, j] = alpha * sum_p sum_c A_p[i, c] * B[j, c] with bf16 operands and fp32 accumulators.  t and
// q are exact in bf16.  An fp32 factor enters as three bf16 planes cut off its bits (8 + 8 + 8 significant bits:
// the planes sum to the value exactly, see split3 for where), so every product is exact in fp32 and the only roundings
// are those of the fp32 sums and of g * a_scale (an fp32 product would round q * a_scale instead: where g * a_scale
// leaves fp32's range, a code of 0 gives NaN).  A bf16 gradient is its own single plane in grad_x.
//
// Bound by the matrix cores: one pass over grad_x and three over grad_w instead of fp32 products, which run at a
// sixteenth of the bf16 rate.  2048 tokens, 2560 -> 6912, bf16 (traced): grad_x 549 -> 87 us + 12 for its three
// partial sums, grad_w 549 -> 180 + 7 us, the layout kernels 40 us in place of 160 us of conversions and transposes;
// the whole step 1364 -> 397 us.
//
// Two steps.  Layout kernels write the operands with the summed index contiguous (the ternary codes and the int8
// codes transposed to bf16; g * a_scale transposed and split), zero-padded to whole stages; then the tile kernel.

#include <algorithm>

#include "wfb_common.h"

namespace wfb {

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

// v = p[0] + p[1] + p[2] exactly for |v| above 2^-110 (below, bits under 2^-133, the smallest bf16, are cut off): each
// plane is the top 16 bits of what is left, by truncation, so none overflows and each remainder is exact.  An
// infinite v has the planes v, 0, 0 and a NaN NaN, 0, 0: they reach the product as they are.
__device__ __forceinline__ void split3(float v, uint16_t (&p)[3]) {
  const uint32_t u = __float_as_uint(v);
  const bool finite = (u & 0x7f800000u) != 0x7f800000u;
  const float h = __uint_as_float(u & 0xffff0000u);
  const float r1 = finite ? __fsub_rn(v, h) : 0.0f;
  const uint32_t u1 = __float_as_uint(r1);
  const float r2 = __fsub_rn(r1, __uint_as_float(u1 & 0xffff0000u));
  p[0] = (uint16_t)(u >> 16) | (uint16_t)(!finite && (u & 0x007fffffu) ? 0x40u : 0u);
  p[1] = (uint16_t)(u1 >> 16);
  p[2] = (uint16_t)(__float_as_uint(r2) >> 16);
}

// ---- operand layouts ---------------------------------------------------------------------------

// Planes of v[n][m] = g[m][n] * a_scale[m], dst[p][n][m] with rows of mp elements (m >= M: zeros).  One 64 x 64
// tile per workgroup through LDS: whole 128-byte lines in and out; the padded rows keep both sides of the
// transpose free of bank conflicts.  With colsum, also the tile's column sums of g, colsum[m0 / 64][n].
template <int DT>
__global__ __launch_bounds__(256) void grad_scaled_t_kernel(const void* __restrict__ g, int64_t ldg,
                                                            const float* __restrict__ a_scale, int64_t M, int64_t N,
                                                            int64_t mp, uint16_t* __restrict__ dst,
                                                            float* __restrict__ colsum) {
  __shared__ float tile[64][65];
  __shared__ float sums[4][64];
  const int64_t m0 = (int64_t)blockIdx.x * 64, n0 = (int64_t)blockIdx.y * 64;
  const int c = threadIdx.x & 63, r0 = threadIdx.x >> 6;
  float v[16], sum = 0.0f;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const int64_t m = m0 + r0 + 4 * j, n = n0 + c;
    const int64_t mc = m < M ? m : M - 1, nc = n < N ? n : N - 1;
    const float x = load_elem<DT>(g, mc * ldg + nc), s = a_scale[mc];
    v[j] = m < M ? __fmul_rn(x, s) : 0.0f;
    sum += m < M ? x : 0.0f;
  }
  sums[r0][c] = sum;
#pragma unroll
  for (int j = 0; j < 16; ++j) tile[r0 + 4 * j][c] = v[j];
  __syncthreads();
  if (colsum && r0 == 0 && n0 + c < N)
    colsum[(int64_t)blockIdx.x * N + n0 + c] = (sums[0][c] + sums[1][c]) + (sums[2][c] + sums[3][c]);
  const int64_t plane = N * mp;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int idx = threadIdx.x + 256 * j, ch = idx & 7, nl = idx >> 3;
    const int64_t n = n0 + nl, m = m0 + 8 * ch;
    if (n >= N || m >= mp) continue;
    union { uint16_t h[8]; uint4 q; } o[3];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      uint16_t p[3];
      split3(tile[8 * ch + e][nl], p);
#pragma unroll
      for (int k = 0; k < 3; ++k) o[k].h[e] = p[k];
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) *reinterpret_cast<uint4*>(dst + k * plane + n * mp + m) = o[k].q;
  }
}

// Planes of g itself, dst[p][m][n] with rows of np elements (n >= N: zeros): three planes of an fp32 or fp16
// gradient, or one (a copy with padded rows) of a bf16 gradient whose rows do not start 16-byte aligned.
template <int DT, int P>
__global__ __launch_bounds__(256) void grad_planes_kernel(const void* __restrict__ g, int64_t ldg, int64_t M,
                                                          int64_t N, int64_t np, uint16_t* __restrict__ dst) {
  const int64_t per = np / 8, idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= M * per) return;
  const int64_t m = idx / per, n = 8 * (idx % per);
  union { uint16_t h[8]; uint4 q; } o[P];
  float v[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int64_t nc = n + e < N ? n + e : N - 1;
    v[e] = load_elem<DT>(g, m * ldg + nc);
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    uint16_t p[3];
    split3(n + e < N ? v[e] : 0.0f, p);
#pragma unroll
    for (int k = 0; k < P; ++k) o[k].h[e] = p[k];
  }
#pragma unroll
  for (int k = 0; k < P; ++k) *reinterpret_cast<uint4*>(dst + k * M * np + m * np + n) = o[k].q;
}

// int8 codes q[m][k] as bf16 dst[k][m], rows of mp elements (m >= M: zeros).  VEC: 16 codes per load (rows 16-byte
// aligned); a row's last codes, fewer than 16, one at a time: nothing has to lie behind the last row's.
template <bool VEC>
__global__ __launch_bounds__(256) void codes_t_kernel(const int8_t* __restrict__ q, int64_t ldq, int64_t M, int64_t K,
                                                      int64_t mp, uint16_t* __restrict__ dst) {
  __shared__ __attribute__((aligned(4))) int8_t tile[64][68];
  const int64_t m0 = (int64_t)blockIdx.x * 64, k0 = (int64_t)blockIdx.y * 64;
  const int r = threadIdx.x >> 2, c = 16 * (threadIdx.x & 3);  // 16 codes of row r
  const int64_t m = m0 + r, row = (m < M ? m : M - 1) * ldq;
  uint32_t v[4] = {0, 0, 0, 0};
  if (VEC && k0 + c + 16 <= K) {
    if (m < M) {
      const uint4 x = *reinterpret_cast<const uint4*>(q + row + k0 + c);
      v[0] = x.x, v[1] = x.y, v[2] = x.z, v[3] = x.w;
    }
  } else if (k0 + c < K) {
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int64_t k = k0 + c + e;
      const uint32_t b = (uint8_t)q[row + (k < K ? k : K - 1)];
      v[e / 4] |= (m < M ? b : 0u) << (8 * (e % 4));
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) *reinterpret_cast<uint32_t*>(&tile[r][c + 4 * e]) = v[e];
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int idx = threadIdx.x + 256 * j, ch = idx & 7, kl = idx >> 3;
    const int64_t k = k0 + kl, mo = m0 + 8 * ch;
    if (k >= K || mo >= mp) continue;
    union { uint16_t h[8]; uint4 q4; } o;
#pragma unroll
    for (int e = 0; e < 8; ++e) o.h[e] = (uint16_t)(__float_as_uint((float)tile[8 * ch + e][kl]) >> 16);
    *reinterpret_cast<uint4*>(dst + k * mp + mo) = o.q4;
  }
}

// The weight scale's power of two, 2^-126 at least; 1 for a scale that is not finite.  The weight codes
// carry it (exact in bf16), so the sums of a gradient run at the size of its result, and the epilogue's factor is what
// is left of the scale: the same bits, without overflow where only the unscaled sum leaves fp32's range.
__device__ __forceinline__ float scale_unit(float s) {
  const uint32_t e = __float_as_uint(s) & 0x7f800000u;
  return e == 0x7f800000u ? 1.0f : __uint_as_float(e ? e : 0x00800000u);
}

// I2_S codes of W[n][k] as bf16 {-u, 0, u}, u = scale_unit(scale), dst[k][n], rows of np elements (n >= N: zeros).
// One 128-weight block of 64 rows per workgroup.
__global__ __launch_bounds__(256) void weight_codes_t_kernel(const uint8_t* __restrict__ qw, int64_t row_bytes,
                                                             int64_t N, int64_t K, int64_t np,
                                                             const float* __restrict__ scale,
                                                             uint16_t* __restrict__ dst) {
  __shared__ __attribute__((aligned(4))) uint8_t tile[64][36];
  const int64_t n0 = (int64_t)blockIdx.x * 64, b = blockIdx.y;
  {
    const int r = threadIdx.x >> 2, c8 = threadIdx.x & 3;  // 8 bytes of one row per thread
    const int64_t n = n0 + r;
    const uint2 w = *reinterpret_cast<const uint2*>(qw + (n < N ? n : N - 1) * row_bytes + 32 * b + 8 * c8);
    uint32_t* t = reinterpret_cast<uint32_t*>(&tile[r][8 * c8]);  // (code 1 = weight 0)
    t[0] = n < N ? w.x : 0x55555555u;
    t[1] = n < N ? w.y : 0x55555555u;
  }
  const float unit = scale_unit(scale[0]);
  __syncthreads();
#pragma unroll
  for (int it = 0; it < 4; ++it) {
    const int idx = threadIdx.x + 256 * it, ch = idx & 7, kl = idx >> 3;  // 8 rows n of column kl
    const int64_t k = 128 * b + kl, n = n0 + 8 * ch;
    if (k >= K || n >= np) continue;
    const int j = kl & 31, sh = 6 - 2 * (kl >> 5);
    union { uint16_t h[8]; uint4 q4; } o;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int code = (tile[8 * ch + e][j] >> sh) & 3;
      o.h[e] = (uint16_t)(__float_as_uint((float)(code - 1) * unit) >> 16);
    }
    *reinterpret_cast<uint4*>(dst + k * np + n) = o.q4;
  }
}

// ---- tile kernel -------------------------------------------------------------------------------

typedef __attribute__((address_space(3))) void lds_void;
__device__ __forceinline__ void lds_load16(buf_t r, void* lds_base, uint32_t voff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)lds_base, 16, voff, 0, 0, 0);
}

struct GradGemm {
  const uint16_t* a;   // [P][I][lda]
  int64_t lda, a_plane;
  const uint16_t* b;   // [J][ldb]
  int64_t ldb;
  int I, J;
  int c_a;             // elements of an A row (offsets past it read zeros)
  int stages;          // of BK elements, all splits together
  int full;            // the first `full` tiles are summed by one workgroup each,
  int nsplit;          // the others by nsplit: split s takes stages [s * per, ...), per = ceil(stages / nsplit)
  const float* alpha;  // device scalar, of which the B rows carry scale_unit, or null (1)
  float* parts;        // fp32 partial tiles [tiles past full][nsplit][BI][BJ]
  void* out;           // [I][ldo] in out_dtype
  int out_dtype;
  int64_t ldo;
  bool vec;            // rows of out 16-byte aligned
};

__device__ __forceinline__ float alpha_of(const GradGemm& p) {
  if (!p.alpha) return 1.0f;
  const float s = p.alpha[0];
  return __fdiv_rn(s, scale_unit(s));  // (exact)
}

__device__ __forceinline__ void store1(const GradGemm& p, int64_t off, float y) {
  if (p.out_dtype == WFB_F32) reinterpret_cast<float*>(p.out)[off] = y;
  else if (p.out_dtype == WFB_BF16) reinterpret_cast<uint16_t*>(p.out)[off] = f32_to_bf16_rne(y);
  else reinterpret_cast<uint16_t*>(p.out)[off] = __builtin_bit_cast(uint16_t, (_Float16)y);
}

// 8 consecutive outputs at element offset off, column col
__device__ __forceinline__ void store8(const GradGemm& p, int64_t off, int col, float4 ya, float4 yb) {
  const float y[8] = {ya.x, ya.y, ya.z, ya.w, yb.x, yb.y, yb.z, yb.w};
  if (!p.vec || col + 8 > p.J) {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (col + e < p.J) store1(p, off + e, y[e]);
    return;
  }
  if (p.out_dtype == WFB_F32) {
    float* o = reinterpret_cast<float*>(p.out) + off;
    *reinterpret_cast<float4*>(o) = ya;
    *reinterpret_cast<float4*>(o + 4) = yb;
    return;
  }
  union { uint16_t h[8]; uint4 q; } o;
#pragma unroll
  for (int e = 0; e < 8; ++e)
    o.h[e] = p.out_dtype == WFB_BF16 ? f32_to_bf16_rne(y[e]) : __builtin_bit_cast(uint16_t, (_Float16)y[e]);
  *reinterpret_cast<uint4*>(reinterpret_cast<uint16_t*>(p.out) + off) = o.q;
}

// C tile of (32 TI WI) x (32 TJ WJ), WI x WJ waves of (32 TI) x (32 TJ), v_mfma_f32_32x32x16_bf16 with B rows as
// src0 and A rows as src1 (lane (i, g), register r: row i of A, row 8 (r / 4) + 4 g + r % 4 of B).  The summed
// index advances in stages of BK: the P planes' rows and the B rows of a stage go from global memory straight
// into one of two LDS buffers (whole 64- or 128-byte row pieces, 16-byte chunks XOR-swizzled by row so that 16
// rows at one chunk meet 16 distinct bank groups), the next stage's loads in flight while a stage is multiplied.
template <int P, int TI, int TJ, int WI, int WJ, int BK, int WPE>
__global__ __launch_bounds__(64 * WI * WJ) __attribute__((amdgpu_waves_per_eu(WPE, WPE))) void grad_tile_kernel(
    GradGemm p, int tiles_i, int tiles_j) {
  constexpr int W = WI * WJ, BI = 32 * TI * WI, BJ = 32 * TJ * WJ;
  constexpr int ROW = 2 * BK, CH = ROW / 16, RPI = 64 / CH;  // bytes and chunks of a row, rows per load
  constexpr int ASZ = P * BI * ROW, BSZ = BJ * ROW, SZ = ASZ + BSZ;
  constexpr int AI = ASZ / 1024 / W, NB = BSZ / 1024 / W;
  constexpr int KS = BK / 16;
  static_assert(AI * 1024 * W == ASZ && NB * 1024 * W == BSZ && (BK == 32 || BK == 64), "tile shape");
  static_assert((P * BI / RPI / W) * W * RPI == P * BI && BI % RPI == 0, "a load stays in one plane");
  __shared__ __attribute__((aligned(16))) uint8_t lds0[SZ];
  __shared__ __attribute__((aligned(16))) uint8_t lds1[SZ];
  const int tid = threadIdx.x, l = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wi = w / WJ, wj = w % WJ, i = l & 31, g = l >> 5;

  // whole tiles first, each XCD a contiguous range of them; then the split ones
  const int per8 = (p.full + 7) / 8, bid = blockIdx.x, u = bid - 8 * per8;
  const bool whole = u < 0;
  const int tt = whole ? (bid % 8) * per8 + bid / 8 : p.full + u / p.nsplit;
  if (whole && tt >= p.full) return;
  const int split = whole ? 0 : u % p.nsplit;
  constexpr int kGroup = 8;
  const int gsz = kGroup * tiles_j, grp = tt / gsz, rr = tt - grp * gsz;
  const int gm = min(kGroup, tiles_i - grp * kGroup);
  const int i0 = (grp * kGroup + rr % gm) * BI, j0 = (rr / gm) * BJ;
  const int per = whole ? p.stages : (p.stages + p.nsplit - 1) / p.nsplit;
  const int s0 = split * per, s1 = min(s0 + per, p.stages);

  const int irows = min(BI, p.I - i0), jrows = min(BJ, p.J - j0);
  const uint32_t a_row = 2u * (uint32_t)p.lda, b_row = 2u * (uint32_t)p.ldb;
  const uint32_t a_end = (uint32_t)irows * a_row, b_end = (uint32_t)jrows * b_row;
  buf_t ab[AI];  // of the plane that load jj of this wave lies in
#pragma unroll
  for (int jj = 0; jj < AI; ++jj)
    ab[jj] = make_buf(p.a + (RPI * (AI * w + jj) / BI) * p.a_plane + (int64_t)i0 * p.lda, a_end);
  const buf_t bb = make_buf(p.b + (int64_t)j0 * p.ldb, b_end);
  const uint32_t a_cols = 2u * (uint32_t)p.c_a;

  auto swz = [](int r) { return BK == 64 ? ((r >> 1) & 7) : ((r >> 2) & 3); };
  // rows past the operand lie past the buffer's end and read zeros
  uint32_t arow[AI], acol[AI], boff[NB];
#pragma unroll
  for (int jj = 0; jj < AI; ++jj) {
    const int R = RPI * (AI * w + jj) + l / CH, r = R % BI;
    arow[jj] = (uint32_t)r * a_row;
    acol[jj] = 16u * ((l % CH) ^ swz(r));
  }
#pragma unroll
  for (int jj = 0; jj < NB; ++jj) {
    const int r = RPI * (NB * w + jj) + l / CH;
    boff[jj] = (uint32_t)r * b_row + 16u * ((l % CH) ^ swz(r));
  }
  auto issue = [&](int s, uint8_t* lds) {
#pragma unroll
    for (int jj = 0; jj < AI; ++jj) {
      const uint32_t col = (uint32_t)ROW * s + acol[jj];
      lds_load16(ab[jj], lds + (AI * w + jj) * 1024, col < a_cols ? arow[jj] + col : a_end);
    }
#pragma unroll
    for (int jj = 0; jj < NB; ++jj) lds_load16(bb, lds + ASZ + (NB * w + jj) * 1024, boff[jj] + (uint32_t)ROW * s);
  };

  f32x16_t acc[TJ][TI];
#pragma unroll
  for (int tj = 0; tj < TJ; ++tj)
#pragma unroll
    for (int ti = 0; ti < TI; ++ti)
#pragma unroll
      for (int q = 0; q < 16; ++q) acc[tj][ti][q] = 0.0f;

  const uint32_t afr = (uint32_t)(wi * TI * 32 + i) * ROW, bfr = ASZ + (uint32_t)(wj * TJ * 32 + i) * ROW;
  // fragments of one 16-element step, two sets: a step's MFMAs run while the next step's are read
  bf16x8_t af[2][P][TI], bf[2][TJ];
  auto read = [&](const uint8_t* lds, int x) {
    const uint32_t c = (uint32_t)(((2 * x + g) ^ swz(i)) * 16);
#pragma unroll
    for (int tj = 0; tj < TJ; ++tj) bf[x & 1][tj] = *reinterpret_cast<const bf16x8_t*>(lds + bfr + tj * 32 * ROW + c);
#pragma unroll
    for (int q = 0; q < P; ++q)
#pragma unroll
      for (int ti = 0; ti < TI; ++ti)
        af[x & 1][q][ti] = *reinterpret_cast<const bf16x8_t*>(lds + afr + (q * BI + ti * 32) * ROW + c);
  };
  auto multiply = [&](int x, bool reads) {
#pragma unroll
    for (int q = 0; q < P; ++q)
#pragma unroll
      for (int ti = 0; ti < TI; ++ti)
#pragma unroll
        for (int tj = 0; tj < TJ; ++tj)
          acc[tj][ti] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bf[x & 1][tj], af[x & 1][q][ti], acc[tj][ti], 0, 0, 0);
    // the reads spread over the MFMAs (left alone, the compiler reads each fragment right before its first use
    // and waits for it)
#pragma unroll
    for (int k = 0; k < P * TI * TJ; ++k) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      if (reads && k < TJ + P * TI) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // stage s from cur; its last step's MFMAs run behind the barrier that hands cur over to stage s + 2's loads and
  // behind the first reads of stage s + 1 from nxt
  auto stage = [&](int s, uint8_t* cur, uint8_t* nxt) {
#pragma unroll
    for (int x = 0; x + 1 < KS; ++x) {
      read(cur, x + 1);
      multiply(x, true);
    }
    if (s + 1 < s1) {
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's loads of stage s + 1 are in LDS
      __syncthreads();                      // everyone's, and everyone has read the last of stage s
      if (s + 2 < s1) issue(s + 2, cur);
      read(nxt, 0);
    }
    multiply(KS - 1, true);
  };
  static_assert(KS % 2 == 0, "a stage starts with fragment set 0");
  if (s0 < s1) {
    issue(s0, lds0);
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();
    if (s0 + 1 < s1) issue(s0 + 1, lds1);
    read(lds0, 0);
    __builtin_amdgcn_sched_barrier(0);
    for (int s = s0; s < s1; s += 2) {
      stage(s, lds0, lds1);
      if (s + 1 < s1) stage(s + 1, lds1, lds0);
    }
  }
  __syncthreads();  // the operand buffers are free

  // per 32-row MFMA tile: 32 rows x 32 TS fp32 (TS of the TJ tiles at a time, as the operand buffers hold it for
  // every wave) through this wave's LDS, 16-byte chunks XOR-swizzled by row; then 8 consecutive outputs of a row
  // per lane, whole lines per instruction
  constexpr int TS = 2 * (SZ / (4096 * TJ)) >= W ? TJ : TJ / 2;
  constexpr int CPR = 8 * TS, ST = 32 * CPR * 16;  // chunks of a staged row, bytes a wave stages
  constexpr int WPB = SZ / ST;                     // waves whose staging fits one buffer
  static_assert(TJ % TS == 0 && WPB >= 1 && 2 * WPB >= W, "staging fits the two operand buffers");
  uint8_t* st = w < WPB ? lds0 + w * ST : lds1 + (w - WPB) * ST;
  const float alpha = whole ? alpha_of(p) : 1.0f;
  constexpr int LPR = CPR / 2, RP = 64 / LPR;
  float* const part = whole ? nullptr : p.parts + (int64_t)u * (BI * BJ);
  auto wave_sync = [] {  // orders the wave's LDS accesses for the compiler (the LDS keeps a wave's order by itself)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
#pragma unroll
  for (int ti = 0; ti < TI; ++ti)
#pragma unroll
    for (int ts = 0; ts < TJ; ts += TS) {
#pragma unroll
      for (int tj = 0; tj < TS; ++tj)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f32x16_t& v = acc[ts + tj][ti];
          const int c = tj * 8 + 2 * q + g;
          *reinterpret_cast<float4*>(st + (i * CPR + (c ^ (i & (CPR - 1)))) * 16) =
              make_float4(v[4 * q] * alpha, v[4 * q + 1] * alpha, v[4 * q + 2] * alpha, v[4 * q + 3] * alpha);
        }
      wave_sync();
#pragma unroll
      for (int jj = 0; jj < 32 / RP; ++jj) {
        const int r = RP * jj + l / LPR, c8 = l % LPR;
        const float4 ya = *reinterpret_cast<const float4*>(st + (r * CPR + ((2 * c8) ^ (r & (CPR - 1)))) * 16);
        const float4 yb = *reinterpret_cast<const float4*>(st + (r * CPR + ((2 * c8 + 1) ^ (r & (CPR - 1)))) * 16);
        const int row = wi * 32 * TI + ti * 32 + r, col = (wj * TJ + ts) * 32 + 8 * c8;  // within the tile
        if (!whole) {
          float4* o = reinterpret_cast<float4*>(part + row * BJ + col);
          o[0] = ya;
          o[1] = yb;
        } else if (i0 + row < p.I && j0 + col < p.J) {
          store8(p, (int64_t)(i0 + row) * p.ldo + j0 + col, j0 + col, ya, yb);
        }
      }
      wave_sync();
    }
}

// The tiles past p.full: out = alpha * the sum of a tile's parts, in order.  A workgroup sums 2048 outputs.
__global__ __launch_bounds__(256) void grad_reduce_kernel(GradGemm p, int bi, int bj, int tiles_i, int tiles_j) {
  const int per = bi * bj / 2048, tile = blockIdx.x / per, e = 2048 * (blockIdx.x % per) + 8 * threadIdx.x;
  const int tt = p.full + tile, gsz = 8 * tiles_j, grp = tt / gsz, rr = tt - grp * gsz;  // the tile kernel's order
  const int gm = min(8, tiles_i - grp * 8);
  const int row = (grp * 8 + rr % gm) * bi + e / bj, col = (rr / gm) * bj + e % bj;
  if (row >= p.I || col >= p.J) return;
  const float* src = p.parts + (int64_t)tile * p.nsplit * (bi * bj) + e;
  float4 a = *reinterpret_cast<const float4*>(src), b = *reinterpret_cast<const float4*>(src + 4);
  for (int s = 1; s < p.nsplit; ++s) {
    src += bi * bj;
    const float4 c = *reinterpret_cast<const float4*>(src), d = *reinterpret_cast<const float4*>(src + 4);
    a.x += c.x, a.y += c.y, a.z += c.z, a.w += c.w;
    b.x += d.x, b.y += d.y, b.z += d.z, b.w += d.w;
  }
  const float alpha = alpha_of(p);
  store8(p, (int64_t)row * p.ldo + col, col, make_float4(a.x * alpha, a.y * alpha, a.z * alpha, a.w * alpha),
         make_float4(b.x * alpha, b.y * alpha, b.z * alpha, b.w * alpha));
}

constexpr int64_t kPad = 64;  // operand rows are whole stages of every variant
constexpr int64_t pad_to(int64_t v, int64_t a) { return (v + a - 1) / a * a; }

// Tile variants: workgroups a CU holds, the rate (PFLOP/s) with all of them busy and the microseconds a round of
// workgroups takes beside its products (first loads, epilogue), measured on MI355X.  Three planes run slower than
// one against ternary rows: the same kernel on constant data reaches 1.5 PFLOP/s, on random planes 1.15 -- the
// power that toggling operands draw lowers the clock.
struct Variant {
  int planes, bi, bj, bk, per_cu;
  double rate, round_us;
};
constexpr Variant kVariants[] = {{1, 256, 256, 64, 1, 1.20, 8}, {1, 128, 128, 64, 2, 1.05, 5},
                                 {1, 64, 128, 64, 3, 0.80, 3}, {3, 128, 256, 32, 2, 1.15, 8},
                                 {3, 64, 128, 32, 4, 0.85, 2.5}};
constexpr int kNumVariants = sizeof(kVariants) / sizeof(kVariants[0]);

// The first `full` tiles whole, the others in nsplit parts of the summed index, each a workgroup of its own.
struct Plan {
  int variant;
  int64_t tiles, full;
  int nsplit;
};

// The least estimated time of every variant, of its tiles all split (or none) or only those past the last full round
// of workgroups, and of the number of parts: rounds of workgroups (a last round that leaves CUs with one workgroup
// runs it in less than the time of a full one) and the partial sums written and read back.  Swept on MI355X over
// every (variant, split of all tiles) of 18 shapes from 1 x 576 x 576 to 4096^3, both products: the estimate's pick
// is within 8% of the fastest on all but four, within 15% there.  Splitting only the tiles past the last full round
// (28 of 540 at 2048 x 6912 x 2560) took grad_w there from 200 us and 26 for all tiles' sums to 180-189 and 7.
Plan plan(int planes, int64_t I, int64_t J, int64_t C) {
  Plan best{-1, 0, 0, 1};
  double best_us = 0;
  for (int v = 0; v < kNumVariants; ++v) {
    const Variant& t = kVariants[v];
    if (t.planes != planes) continue;
    const int64_t tiles = ((I + t.bi - 1) / t.bi) * ((J + t.bj - 1) / t.bj), slots = 256 * t.per_cu;
    const int64_t stages = pad_to(C, kPad) / t.bk;
    const double rate = t.rate * 1e9 / slots;  // operations per us of one workgroup's slot
    auto rounds_us = [&](int64_t wgs, int64_t n) {  // wgs workgroups of n stages each
      const int64_t full = wgs / slots;
      const double r = (double)(wgs % slots) / slots;
      const double last = r == 0 ? 0 : t.per_cu == 1 ? 0.85 : r * t.per_cu <= 1 ? 0.6 : 0.6 + 0.4 * r;
      return (full + last) * 2.0 * planes * t.bi * t.bj * n * t.bk / rate + t.round_us * (full + (r > 0));
    };
    auto consider = [&](int64_t full, int64_t ns, double us) {
      if (best.variant < 0 || us < best_us) best = {v, tiles, full, (int)ns}, best_us = us;
    };
    consider(tiles, 1, rounds_us(tiles, stages));
    for (int64_t want = 2; want <= 32 && stages / want >= 4; ++want) {
      const int64_t per = (stages + want - 1) / want, ns = (stages + per - 1) / per;  // no empty split
      if (ns != want) continue;
      for (const int64_t full : {(int64_t)0, tiles / slots * slots}) {
        const int64_t rest = tiles - full;
        if (rest == 0 || rest * ns > 4 * slots) continue;  // (no rest, or enough workgroups without so many parts)
        const double sums = 4.0 + 8.0 * ns * rest * t.bi * t.bj / 8e6;
        consider(full, ns, (full ? rounds_us(full, stages) : 0) + rounds_us(rest * ns, per) + sums);
      }
    }
  }
  return best;
}

template <int P, int TI, int TJ, int WI, int WJ, int BK, int WPE>
hipError_t launch_tiles(const GradGemm& p, const Plan& pl, hipStream_t s) {
  constexpr int BI = 32 * TI * WI, BJ = 32 * TJ * WJ;
  const int ti = (p.I + BI - 1) / BI, tj = (p.J + BJ - 1) / BJ;
  const int64_t rest = pl.tiles - pl.full, grid = pad_to(pl.full, 8) + rest * pl.nsplit;
  if (grid > INT32_MAX) return hipErrorInvalidValue;
  hipLaunchKernelGGL((grad_tile_kernel<P, TI, TJ, WI, WJ, BK, WPE>), dim3((unsigned)grid), dim3(64 * WI * WJ), 0, s, p,
                     ti, tj);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || rest == 0) return e;
  hipLaunchKernelGGL(grad_reduce_kernel, dim3((unsigned)(rest * (BI * BJ / 2048))), dim3(256), 0, s, p, BI, BJ, ti, tj);
  return hipGetLastError();
}

hipError_t run_gemm(GradGemm p, const Plan& pl, int64_t C, float* parts, hipStream_t s) {
  p.stages = (int)(pad_to(C, kPad) / kVariants[pl.variant].bk);
  p.full = (int)pl.full;
  p.nsplit = pl.nsplit;
  p.parts = parts;
  const int osz = p.out_dtype == WFB_F32 ? 4 : 2;
  p.vec = (uintptr_t)p.out % 16 == 0 && (p.ldo * osz) % 16 == 0;
  switch (pl.variant) {  // kVariants
    case 0: return launch_tiles<1, 4, 2, 2, 4, 64, 2>(p, pl, s);
    case 1: return launch_tiles<1, 2, 2, 2, 2, 64, 2>(p, pl, s);
    case 2: return launch_tiles<1, 1, 2, 2, 2, 64, 3>(p, pl, s);
    case 3: return launch_tiles<3, 2, 4, 2, 2, 32, 2>(p, pl, s);
    default: return launch_tiles<3, 1, 2, 2, 2, 32, 4>(p, pl, s);
  }
}

constexpr int64_t align256(int64_t b) { return pad_to(b, 256); }
int64_t part_bytes(const Plan& pl) {
  return 4 * (pl.tiles - pl.full) * pl.nsplit * kVariants[pl.variant].bi * kVariants[pl.variant].bj;
}

int grad_x_planes(int gdt) { return gdt == WFB_BF16 ? 1 : 3; }

}  // namespace

// grad_x operands in the workspace: [K][Np] weight codes, then the planes of g (always reserved, so that the size
// does not depend on the alignment of g), then the partial sums.
int64_t grad_x_workspace(int64_t m, int64_t n, int64_t k, int gdt) {
  const int64_t np = pad_to(n, kPad);
  const int P = grad_x_planes(gdt);
  return align256(2 * k * np) + align256(2 * P * m * np) + part_bytes(plan(P, m, k, n));
}

int64_t grad_w_workspace(int64_t m, int64_t n, int64_t k) {
  const int64_t mp = pad_to(m, kPad);
  return align256(2 * 3 * n * mp) + align256(2 * k * mp) + align256(4 * (mp / 64) * n) +
         part_bytes(plan(3, n, k, m));
}

void grad_plan(bool of_x, int64_t m, int64_t n, int64_t k, int gdt, int64_t (&out)[5]) {
  const Plan pl = of_x ? plan(grad_x_planes(gdt), m, k, n) : plan(3, n, k, m);
  const Variant& v = kVariants[pl.variant];
  const int64_t o[5] = {v.bi, v.bj, pl.tiles, pl.full, pl.nsplit};
  std::copy(o, o + 5, out);
}

hipError_t launch_grad_x(const void* g, int gdt, int64_t ldg, int64_t m, int64_t n, const uint8_t* qw, int64_t k,
                         int64_t k_pad, const float* w_scale, void* out, int odt, int64_t ldo, void* work,
                         hipStream_t s) {
  const int64_t np = pad_to(n, kPad);
  const int P = grad_x_planes(gdt);
  char* ws = static_cast<char*>(work);
  uint16_t* wt = reinterpret_cast<uint16_t*>(ws);
  uint16_t* gp = reinterpret_cast<uint16_t*>(ws + align256(2 * k * np));
  float* parts = reinterpret_cast<float*>(ws + align256(2 * k * np) + align256(2 * P * m * np));
  hipLaunchKernelGGL(weight_codes_t_kernel, dim3((unsigned)(np / 64), (unsigned)((k + 127) / 128)), dim3(256), 0, s, qw,
                     k_pad / 4, n, k, np, w_scale, wt);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  GradGemm p{};
  p.b = wt;
  p.ldb = np;
  p.I = (int)m;
  p.J = (int)k;
  p.alpha = w_scale;
  p.out = out;
  p.out_dtype = odt;
  p.ldo = ldo;
  if (gdt == WFB_BF16 && (uintptr_t)g % 16 == 0 && ldg % 8 == 0 && n % 8 == 0) {
    p.a = static_cast<const uint16_t*>(g);
    p.lda = ldg;
    p.c_a = (int)n;
  } else {
    const unsigned grid = (unsigned)((m * (np / 8) + 255) / 256);
    if (gdt == WFB_BF16)
      hipLaunchKernelGGL((grad_planes_kernel<WFB_BF16, 1>), dim3(grid), dim3(256), 0, s, g, ldg, m, n, np, gp);
    else if (gdt == WFB_F32)
      hipLaunchKernelGGL((grad_planes_kernel<WFB_F32, 3>), dim3(grid), dim3(256), 0, s, g, ldg, m, n, np, gp);
    else
      hipLaunchKernelGGL((grad_planes_kernel<WFB_F16, 3>), dim3(grid), dim3(256), 0, s, g, ldg, m, n, np, gp);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    p.a = gp;
    p.lda = np;
    p.a_plane = m * np;
    p.c_a = (int)np;
  }
  return run_gemm(p, plan(P, m, k, n), n, parts, s);
}

hipError_t launch_grad_w(const void* g, int gdt, int64_t ldg, int64_t m, int64_t n, const int8_t* q, int64_t ldq,
                         const float* a_scale, int64_t k, void* out, int odt, int64_t ldo, void* bias_out, int bdt,
                         void* work, hipStream_t s) {
  const int64_t mp = pad_to(m, kPad);
  char* ws = static_cast<char*>(work);
  uint16_t* gt = reinterpret_cast<uint16_t*>(ws);
  uint16_t* qt = reinterpret_cast<uint16_t*>(ws + align256(2 * 3 * n * mp));
  float* sums = reinterpret_cast<float*>(ws + align256(2 * 3 * n * mp) + align256(2 * k * mp));
  float* parts = reinterpret_cast<float*>(reinterpret_cast<char*>(sums) + align256(4 * (mp / 64) * n));
  float* cs = bias_out ? sums : nullptr;
  const dim3 gg((unsigned)(mp / 64), (unsigned)((n + 63) / 64));
  if (gdt == WFB_F32)
    hipLaunchKernelGGL((grad_scaled_t_kernel<WFB_F32>), gg, dim3(256), 0, s, g, ldg, a_scale, m, n, mp, gt, cs);
  else if (gdt == WFB_BF16)
    hipLaunchKernelGGL((grad_scaled_t_kernel<WFB_BF16>), gg, dim3(256), 0, s, g, ldg, a_scale, m, n, mp, gt, cs);
  else
    hipLaunchKernelGGL((grad_scaled_t_kernel<WFB_F16>), gg, dim3(256), 0, s, g, ldg, a_scale, m, n, mp, gt, cs);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (bias_out && (e = launch_column_sum(sums, (int)(mp / 64), n, bias_out, bdt, s)) != hipSuccess) return e;
  const dim3 gq((unsigned)(mp / 64), (unsigned)((k + 63) / 64));
  if ((uintptr_t)q % 16 == 0 && ldq % 16 == 0)
    hipLaunchKernelGGL((codes_t_kernel<true>), gq, dim3(256), 0, s, q, ldq, m, k, mp, qt);
  else
    hipLaunchKernelGGL((codes_t_kernel<false>), gq, dim3(256), 0, s, q, ldq, m, k, mp, qt);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  GradGemm p{};
  p.a = gt;
  p.lda = mp;
  p.a_plane = n * mp;
  p.b = qt;
  p.ldb = mp;
  p.I = (int)n;
  p.J = (int)k;
  p.c_a = (int)mp;
  p.out = out;
  p.out_dtype = odt;
  p.ldo = ldo;
  return run_gemm(p, plan(3, n, k, m), m, parts, s);
}

}  // namespace wfb
