// Causal GQA attention for a prefill chunk of T tokens per sequence (bf16 caches), with the rotary
// embedding of the new queries/keys and the cache append.
//
// Same contract as the decode kernel (attention_forward, SGB/sgl-kernel/csrc/inference/bitnet_engine.cpp:381-441,
// and kv_cache_update_key / _value, SGB/sgl-kernel/csrc/inference/kv_cache.h:81-101) for every query of the
// chunk: token i of sequence b sits at position start + i and attends over keys 0..start+i (causal), the
// rotary embedding in the HF rotate-half form of the stage-1 model
// (packages/training/src/wrinklefree/training/stage1.py:169-214), applied with the same fp32 operations as
// the torch formula and rounded to bf16.
//
// Two launches.  gqa_append_kernel ropes the T new keys and writes them and the values into the cache
// (bit-identical to the torch cache writes).  gqa_prefill_kernel then runs flash attention on the matrix cores: one
// workgroup per (32 query tokens, kv head, sequence), one wave per query head of the group (more tokens where a group
// has one or two heads), so each 64-key block of K and V is staged in LDS once for all heads of the group.  Per key
// block a wave
//   S^T[key, q] = K Q^T        v_mfma_f32_32x32x16_bf16, K rows from LDS (A), roped Q in registers (B)
//   online softmax per query   the 32 queries sit in lanes l % 32; a query's 64 keys in lanes l and l ^ 32
//   O^T[d, q] += V^T P^T       V rows from LDS through the transposing read (A); P from the S^T registers of the same
//                              lane (B), split P = hi + lo (two bf16 products, ~16 mantissa bits)
// The reduction index k of an MFMA is a free labelling as long as A and B agree: S^T takes k = head
// dimension (16ks + 8(l/32) + j, 16 contiguous bytes of a row of K and of Q); O^T takes k = key, mapped to
// the keys the lane already holds from S^T (16c + 4(l/32) + j and 16c + 8 + 4(l/32) + j - 4).
// Scores and softmax are fp32; products of bf16 operands are exact in fp32 and summed in fp32.
//
// What bounds it: vector issue.  A wave's 64 keys take 48 MFMAs (1536 matrix cycles, 768 of issue) and some 1300 cycles
// of softmax and conversion, 512 of them the 32 exponentials; counters at 4096 tokens, 32/8 heads of 128: MFMA busy
// 55%, VALU 49% of the cycles of busy CUs.  32 queries per wave halve the LDS reads and the issue slots per product of
// the 16-query form, which was LDS-bound; fragments are read 4 ahead of their products; the exponentials of a step run
// under the products of the step before.  Whole calls in a graph, buffers in turn, against the 16-token form: 4096
// tokens, 32/8 heads of 128 357 -> 217 us (211 in a stream of calls: 650 TFLOP/s); 8 x 2048 637 -> 436; 8 x 256 29.4 ->
// 23.3; 2048 tokens of 40/8 heads 204 -> 93; 4096 of 9/3 heads of 64 147 -> 79.
// Measured without gain: K and V^T staged through registers as in the 16-token form (260 against 253 us of the kernel
// as it was then; the transposing reads make it no slower and free 32 registers), 32-key blocks at 3 waves per SIMD (25
// spills, 307 us).
#include "wfb_common.h"

namespace wfb {

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

union Frag8 {
  bf16x8_t v;
  uint16_t h[8];
  uint32_t u[4];
  v4i q;
};

typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4_t lds_s16x4;
typedef __attribute__((address_space(3))) void lds_void;
__device__ __forceinline__ void lds_load16(buf_t r, void* lds_base, uint32_t voff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)lds_base, 16, voff, 0, 0, 0);
}
// slots j < 4 from the first transposing read, j >= 4 from the second
__device__ __forceinline__ bf16x8_t vfrag(const s16x4_t (&v)[2]) {
  return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(v[0], v[1], 0, 1, 2, 3, 4, 5, 6, 7));
}

__device__ __forceinline__ float bf16f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// y1 = x1 c + (-x2) s, y2 = x2 c + x1 s, each product and sum rounded to fp32, then to bf16
__device__ __forceinline__ void rope_pair(float x1, float x2, float c, float s, uint16_t& y1, uint16_t& y2) {
  y1 = f32_to_bf16_rne(__fadd_rn(__fmul_rn(x1, c), __fmul_rn(-x2, s)));
  y2 = f32_to_bf16_rne(__fadd_rn(__fmul_rn(x2, c), __fmul_rn(x1, s)));
}

// One workgroup per (token i, sequence b): rotary of the token's kv heads' keys, cache writes of key
// and value at position start + i.
template <int D>
__global__ __launch_bounds__(256) void gqa_append_kernel(const uint16_t* __restrict__ kn, int64_t ldk,
                                                         const uint16_t* __restrict__ vn, int64_t ldv,
                                                         const float* __restrict__ rope_cos,
                                                         const float* __restrict__ rope_sin, uint16_t* __restrict__ kc,
                                                         uint16_t* __restrict__ vc, int64_t max_len, int hkv, int T,
                                                         int64_t start, bool vec) {
  constexpr int HD = D / 2;
  const int i = blockIdx.x, b = blockIdx.y;
  const int64_t pos = start + i;
  const int64_t row = (int64_t)b * T + i;
  if (vec) {  // 16-byte pieces: 8 rotary pairs of a key, or 8 value elements, per thread
    constexpr int KI = HD / 8, VI = D / 8;
    for (int e = threadIdx.x; e < hkv * (KI + VI); e += blockDim.x) {
      if (e < hkv * KI) {
        const int g = e / KI, j0 = 8 * (e % KI);
        const uint16_t* kr = kn + row * ldk + (int64_t)g * D;
        uint16_t* dst = kc + (((int64_t)b * hkv + g) * max_len + pos) * D;
        Frag8 x1, x2;
        x1.q = *reinterpret_cast<const v4i*>(kr + j0);
        x2.q = *reinterpret_cast<const v4i*>(kr + j0 + HD);
        if (rope_cos) {
          const float4* cp = reinterpret_cast<const float4*>(rope_cos + pos * HD + j0);
          const float4* sp = reinterpret_cast<const float4*>(rope_sin + pos * HD + j0);
          const float4 c0 = cp[0], c1 = cp[1], s0 = sp[0], s1 = sp[1];
          const float cs[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
          const float sn[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
          float y1[8], y2[8];
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float a = bf16f(x1.h[j]), c = bf16f(x2.h[j]);
            y1[j] = __fadd_rn(__fmul_rn(a, cs[j]), __fmul_rn(-c, sn[j]));
            y2[j] = __fadd_rn(__fmul_rn(c, cs[j]), __fmul_rn(a, sn[j]));
          }
#pragma unroll
          for (int j = 0; j < 8; j += 2) {  // bf16, round to nearest even (v_cvt_pk_bf16_f32)
            x1.u[j / 2] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t){y1[j], y1[j + 1]}, bf16x2_t));
            x2.u[j / 2] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t){y2[j], y2[j + 1]}, bf16x2_t));
          }
        }
        *reinterpret_cast<v4i*>(dst + j0) = x1.q;
        *reinterpret_cast<v4i*>(dst + j0 + HD) = x2.q;
      } else {
        const int e2 = e - hkv * KI, g = e2 / VI, j0 = 8 * (e2 % VI);
        *reinterpret_cast<v4i*>(vc + (((int64_t)b * hkv + g) * max_len + pos) * D + j0) =
            *reinterpret_cast<const v4i*>(vn + row * ldv + (int64_t)g * D + j0);
      }
    }
    return;
  }
  for (int e = threadIdx.x; e < hkv * HD; e += blockDim.x) {
    const int g = e / HD, j = e % HD;
    const uint16_t* kr = kn + row * ldk + (int64_t)g * D;
    uint16_t* dst = kc + (((int64_t)b * hkv + g) * max_len + pos) * D;
    if (rope_cos) {
      uint16_t y1, y2;
      rope_pair(bf16f(kr[j]), bf16f(kr[j + HD]), rope_cos[pos * HD + j], rope_sin[pos * HD + j], y1, y2);
      dst[j] = y1;
      dst[j + HD] = y2;
    } else {
      dst[j] = kr[j];
      dst[j + HD] = kr[j + HD];
    }
  }
  for (int e = threadIdx.x; e < hkv * D; e += blockDim.x) {
    const int g = e / D, j = e % D;
    vc[(((int64_t)b * hkv + g) * max_len + pos) * D + j] = vn[row * ldv + (int64_t)g * D + j];
  }
}

// Flash attention, QW blocks of 32 query tokens x G query heads of one kv head per workgroup, a wave each.
template <int D, int G, int QW>
__global__ __launch_bounds__(64 * G * QW) __attribute__((amdgpu_waves_per_eu(2))) void gqa_prefill_kernel(
    const uint16_t* __restrict__ q, int64_t ldq, const float* __restrict__ rope_cos, const float* __restrict__ rope_sin,
    const uint16_t* __restrict__ kc, const uint16_t* __restrict__ vc, int64_t max_len, int hkv, int T, int64_t start,
    float scale, uint16_t* __restrict__ out, int64_t ldo, int nhb, int nqb) {
  constexpr int KS = D / 16;       // MFMA k-steps over the head dimension
  constexpr int DT = D / 32;       // 32-row tiles of O^T
  constexpr int KB = 64;           // keys per block
  constexpr int kRing = 4;         // K / V fragments read ahead of their MFMAs
  constexpr int CH = D / 8;        // 16-byte chunks of a key or value row
  constexpr int W = G * QW;
  __shared__ __attribute__((aligned(16))) uint16_t k0_[KB * D], k1_[KB * D], v0_[KB * D], v1_[KB * D];

  // workgroups of one (kv head, sequence) are nhb apart, so with 8 or more of them an XCD's L2 holds few heads; the
  // longest rows (the last query blocks) come first
  const int hb = blockIdx.x % nhb, i0 = (nqb - 1 - blockIdx.x / nhb) * 32 * QW, g = hb % hkv, b = hb / hkv;
  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int h = g * G + w % G;
  const int grp = lane >> 5;
  const int iw = i0 + 32 * (w / G);            // the wave's first query token
  const int qi = iw + (lane & 31);             // this lane's query token (S^T / O^T column)
  const bool qvalid = qi < T;
  const int64_t qpos = start + qi;
  const int qpos32 = (int)qpos;                // positions < max_len < 2^23 (host-checked)
  const int qpos_first = (int)(start + iw);    // the wave's first query position
  // exp(s scale - m) as one fma and one exp2: scores in units of scale * log2(e), a negative scale moved into the
  // signs of Q (exact); the floor, the smallest normal float, keeps a masked score's -inf * c2 from being NaN at scale 0
  const float c2 = fmaxf(fabsf(scale) * 1.4426950408889634f, 0x1p-126f);
  const uint32_t flip = scale < 0.0f ? 0x80008000u : 0u;

  // roped query fragments: lane holds Q[qi][16ks + 8grp .. +7] for each ks
  Frag8 qf[KS];
  {
    const uint16_t* qr = q + ((int64_t)b * T + (qvalid ? qi : 0)) * ldq + (int64_t)h * D;
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[s].q = *reinterpret_cast<const v4i*>(qr + 16 * s + 8 * grp);
    if (!qvalid) {
#pragma unroll
      for (int s = 0; s < KS; ++s) qf[s].q = v4i{0, 0, 0, 0};
    } else if (rope_cos) {
      constexpr int HD = D / 2;
#pragma unroll
      for (int s = 0; s < KS / 2; ++s) {
        // elements d = 16s + 8grp + j (< D/2) and their partners d + D/2 (fragment s + KS/2, slot j);
        // the 8 table entries of d are contiguous (16-byte aligned tables, host-checked)
        const float4* cp = reinterpret_cast<const float4*>(rope_cos + qpos * HD + 16 * s + 8 * grp);
        const float4* sp = reinterpret_cast<const float4*>(rope_sin + qpos * HD + 16 * s + 8 * grp);
        const float4 c0 = cp[0], c1 = cp[1], s0 = sp[0], s1 = sp[1];
        const float cs[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
        const float sn[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
        float y1[8], y2[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float x1 = bf16f(qf[s].h[j]), x2 = bf16f(qf[s + KS / 2].h[j]);
          y1[j] = __fadd_rn(__fmul_rn(x1, cs[j]), __fmul_rn(-x2, sn[j]));
          y2[j] = __fadd_rn(__fmul_rn(x2, cs[j]), __fmul_rn(x1, sn[j]));
        }
#pragma unroll
        for (int j = 0; j < 8; j += 2) {  // round to bf16, nearest even (v_cvt_pk_bf16_f32)
          qf[s].u[j / 2] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t){y1[j], y1[j + 1]}, bf16x2_t));
          qf[s + KS / 2].u[j / 2] =
              __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t){y2[j], y2[j + 1]}, bf16x2_t));
        }
      }
    }
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int j = 0; j < 4; ++j) qf[s].u[j] ^= flip;
  }

  // keys needed by the workgroup's last valid query; loads past them read zeros (no stale cache rows enter
  // the P V product, where a masked p = 0 would still meet them)
  const int64_t kend = start + (i0 + 32 * QW < T ? i0 + 32 * QW : T);
  const int nkb = (int)((kend + KB - 1) / KB);
  const int64_t slice = ((int64_t)b * hkv + g) * max_len * D;  // element offset of the (b, g) cache slice
  const buf_t kb_ = make_buf(kc + slice, (uint32_t)(kend * D * 2));
  const buf_t vb_ = make_buf(vc + slice, (uint32_t)(kend * D * 2));

  f32x16_t o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[dt][r] = 0.0f;
  float m_ref = -__builtin_inff(), l_run = 0.0f;

  // K and V rows go from global memory straight into LDS, row-major, block kb + 1's while block kb is computed (two
  // buffers).  Position p of row r holds chunk p ^ f(r): for K so that one chunk of 16 consecutive rows (an MFMA
  // operand read) lies on 16 distinct 16-byte bank groups, for V so that 32 bytes of 4 consecutive rows (a
  // transposing read) lie on distinct banks.
  auto kswz = [](int r) { return D == 128 ? r & 15 : (r >> 1) & 7; };
  auto vswz = [](int r) { return D == 128 ? 4 * (r & 3) : 4 * ((r >> 1) & 1); };
  constexpr int RPI = 64 / CH, NI = KB / RPI;  // rows per 1 KB load instruction, instructions per tile
  auto issue = [&](int key0, uint16_t* kd, uint16_t* vd) {
#pragma unroll
    for (int it = 0; it < (2 * NI + W - 1) / W; ++it) {
      const int i = w + it * W;  // uniform
      if (2 * NI % W != 0 && i >= 2 * NI) break;
      const int r = RPI * (i < NI ? i : i - NI) + lane / CH, c = (lane % CH) ^ (i < NI ? kswz(r) : vswz(r));
      const uint32_t off = (uint32_t)(((key0 + r) * D + 8 * c) * 2);
      if (i < NI) lds_load16(kb_, kd + i * 512, off);
      else lds_load16(vb_, vd + (i - NI) * 512, off);
    }
  };

  const int ka = (lane & 31) * D, kx = kswz(lane & 31);
  const int vrow = 4 * grp + ((lane >> 2) & 3), vcol = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  const int vx = vswz(vrow);
  auto block = [&](int kb, uint16_t* ks, uint16_t* vs, uint16_t* kn, uint16_t* vn) {
    const int key0 = kb * KB;
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's loads of block kb are in LDS
    __syncthreads();                      // everyone's, and everyone is done with block kb - 1
    if (kb + 1 < nkb) issue(key0 + KB, kn, vn);

    // S^T = K Q^T for the 2 sub-blocks of 32 keys: register r holds key 32 nb + 8 (r / 4) + 4 grp + r % 4
    // (the fragments kRing steps ahead of their MFMAs: read right before its use, each costs an LDS round trip)
    f32x16_t s[2];
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
      for (int r = 0; r < 16; ++r) s[nb][r] = 0.0f;
    {
      v4i a[kRing];
      auto read_k = [&](int i) {
        a[i % kRing] = *reinterpret_cast<const v4i*>(ks + 32 * D * (i & 1) + ka + 8 * ((2 * (i >> 1) + grp) ^ kx));
      };
#pragma unroll
      for (int i = 0; i < kRing; ++i) read_k(i);
#pragma unroll
      for (int i = 0; i < 2 * KS; ++i) {
        s[i & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a[i % kRing]), qf[i >> 1].v,
                                                           s[i & 1], 0, 0, 0);
        if (i + kRing < 2 * KS) read_k(i + kRing);
      }
      __builtin_amdgcn_sched_group_barrier(0x100, kRing, 0);
#pragma unroll
      for (int i = 0; i < 2 * KS; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if (i + kRing < 2 * KS) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (key0 + KB - 1 > qpos_first) {  // causal mask: only blocks reaching past the wave's first query (uniform)
#pragma unroll
      for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (key0 + 32 * nb + 8 * (r / 4) + 4 * grp + r % 4 > qpos32) s[nb][r] = -__builtin_inff();
    }
    float bmax = s[0][0];
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
      for (int r = 0; r < 16; ++r) bmax = fmaxf(bmax, s[nb][r]);
    bmax = fmaxf(bmax, xor_lanes_f32<32>(bmax)) * c2;
    // the reference exponent follows the running maximum only when a query's grows by more than 2^8 (always in the
    // first block, which holds key 0 <= qpos): p stays below 2^8, and o and l need no rescale in most blocks
    if (__any(bmax > m_ref + 8.0f)) {
      const float m_new = fmaxf(m_ref, bmax), alpha = __builtin_amdgcn_exp2f(m_ref - m_new);
      m_ref = m_new;
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) o[dt] *= alpha;
    }
    // O^T += V^T P^T over 4 steps of 16 keys (slots j < 4: keys 16t + 4grp + j, j >= 4: 16t + 8 + 4grp + j - 4); a
    // step's exponentials and conversions run under the MFMAs of the step before
    float psum = 0.0f;
    // p - hi, exactly, as a two-element dot product with (-1, 0) or (0, -1), which picks its half of the packed pair
    // (kept in registers: as a literal, (0, -1) has the bits of the float -1, which the instruction takes for a
    // 16-bit constant in the low half)
    uint32_t neg_lo = 0x0000BF80u, neg_hi = 0xBF800000u;
    asm("" : "+s"(neg_lo), "+s"(neg_hi));
    Frag8 phi[2], plo[2];  // hi = bf16(p), lo = bf16(p - hi), both round-to-nearest-even (v_cvt_pk_bf16_f32)
    auto probs = [&](int c) {
#pragma unroll
      for (int j = 0; j < 8; j += 2) {
        const int r = 8 * (c & 1) + j;
        const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[c / 2][r], c2, -m_ref));
        const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[c / 2][r + 1], c2, -m_ref));
        psum += p0;
        psum += p1;
        const uint32_t hi = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t){p0, p1}, bf16x2_t));
        const bf16x2_t h2 = __builtin_bit_cast(bf16x2_t, hi);
        const float r0 = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, neg_lo), h2, p0, false);
        const float r1 = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, neg_hi), h2, p1, false);
        phi[c & 1].u[j / 2] = hi;
        plo[c & 1].u[j / 2] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t){r0, r1}, bf16x2_t));
      }
    };
    s16x4_t vf[kRing][2];
    auto read_v = [&](int i) {  // fragment of step i / DT, row tile i % DT: 4 keys of this lane's column, and 4 more
      const int col = 32 * (i % DT) + vcol, row = 16 * (i / DT) + vrow;
      uint16_t* vr = vs + row * D + (((col >> 3) ^ vx) << 3) + (col & 7);
      vf[i % kRing][0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)vr);
      vf[i % kRing][1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(vr + 8 * D));
    };
#pragma unroll
    for (int i = 0; i < kRing; ++i) read_v(i);
    probs(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if (c + 1 < 4) probs(c + 1);
      // two row tiles at a time, so that no product waits for the one before it
#pragma unroll
      for (int d2 = 0; d2 < DT; d2 += 2) {
        const int i = c * DT + d2;
        const bf16x8_t a0 = vfrag(vf[i % kRing]), a1 = vfrag(vf[(i + 1) % kRing]);
        o[d2] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, phi[c & 1].v, o[d2], 0, 0, 0);
        o[d2 + 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, phi[c & 1].v, o[d2 + 1], 0, 0, 0);
        o[d2] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, plo[c & 1].v, o[d2], 0, 0, 0);
        o[d2 + 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, plo[c & 1].v, o[d2 + 1], 0, 0, 0);
        if (i + kRing < 4 * DT) read_v(i + kRing);
        if (i + 1 + kRing < 4 * DT) read_v(i + 1 + kRing);
      }
#pragma unroll
      for (int k = 0; k < 2 * DT; ++k) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if (c + 1 < 4) __builtin_amdgcn_sched_group_barrier(0x002, 40 / (2 * DT), 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    l_run += psum;  // (this lane's keys; the other half of a query's keys is in lane ^ 32, added at the end)
  };
  issue(0, k0_, v0_);
  for (int kb = 0; kb < nkb; kb += 2) {
    block(kb, k0_, v0_, k1_, v1_);
    if (kb + 1 < nkb) block(kb + 1, k1_, v1_, k0_, v0_);
  }

  l_run += xor_lanes_f32<32>(l_run);
  if (!qvalid) return;
  // lane holds O^T[32dt + 8(r / 4) + 4grp + r % 4][qi]: four consecutive elements of the output row per quarter
  uint16_t* orow = out + ((int64_t)b * T + qi) * ldo + (int64_t)h * D;
  const float inv_l = 1.0f / l_run;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; r += 4) {
      uint2 v;
      v.x = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t){o[dt][r] * inv_l, o[dt][r + 1] * inv_l}, bf16x2_t));
      v.y = __builtin_bit_cast(uint32_t,
                               __builtin_convertvector((f32x2_t){o[dt][r + 2] * inv_l, o[dt][r + 3] * inv_l}, bf16x2_t));
      *reinterpret_cast<uint2*>(orow + 32 * dt + 2 * r + 4 * grp) = v;
    }
}

// 16 query tokens per workgroup, for prompts whose workgroups leave CUs idle (launch_prefill_g): one wave per query head of
// the group, v_mfma_f32_16x16x32_bf16, both K and V^T staged through registers.  Half the products per wave and key
// block of the kernel above, so the serial chain of a lone workgroup is shorter.  S^T takes k = head dimension (32ks +
// 8(l/16) + j); O^T takes k = key, mapped to the keys the lane already holds from S^T (32c + 4(l/16) + j and 32c + 16 +
// 4(l/16) + j - 4).
// At D = 128 with 4 query heads per kv head (Llama-3-8B) the kernel is held to 3 waves per SIMD
// (158 registers, no spills; 29.1 -> 26.3 us at the Llama-3-8B prompt shape, where the compiler's own
// choice was 176 registers and 2 waves); the other shapes keep the compiler's choice.
template <int D, int G>
__global__ __launch_bounds__(64 * G) __attribute__((amdgpu_waves_per_eu(D == 128 && G == 4 ? 3 : 1))) void gqa_prefill16_kernel(const uint16_t* __restrict__ q, int64_t ldq,
                                                             const float* __restrict__ rope_cos,
                                                             const float* __restrict__ rope_sin,
                                                             const uint16_t* __restrict__ kc,
                                                             const uint16_t* __restrict__ vc, int64_t max_len, int hkv,
                                                             int T, int64_t start, float scale,
                                                             uint16_t* __restrict__ out, int64_t ldo) {
  constexpr int KS = D / 32;       // MFMA k-steps over the head dimension
  constexpr int DB = D / 16;       // 16-row blocks of O^T
  constexpr int KB = 64;           // keys per block
  constexpr int KROW = D + 8;      // K tile row stride (elements): 16-byte aligned, rows 4 banks apart
  constexpr int VROW = KB + 4;     // V^T tile row stride (elements): rows 2 banks apart (+ 8-byte reads)
  constexpr int NT = 64 * G;
  __shared__ __attribute__((aligned(16))) uint16_t ks_[KB * KROW];
  __shared__ __attribute__((aligned(16))) uint16_t vs_[D * VROW];

  const int i0 = blockIdx.x * 16, g = blockIdx.y, b = blockIdx.z;
  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int h = g * G + w;
  const int grp = lane >> 4;
  const int qi = i0 + (lane & 15);  // this lane's query token (S^T / O^T column)
  const bool qvalid = qi < T;
  const int64_t qpos = start + qi;
  const int qpos32 = (int)qpos;                // positions < max_len < 2^23 (host-checked)
  const int qpos_first = (int)(start + i0);    // the workgroup's first query position

  // roped query fragments: lane holds Q[qi][32ks + 8grp .. +7] for each ks
  Frag8 qf[KS];
  {
    const uint16_t* qr = q + ((int64_t)b * T + (qvalid ? qi : 0)) * ldq + (int64_t)h * D;
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[s].q = *reinterpret_cast<const v4i*>(qr + 32 * s + 8 * grp);
    if (!qvalid) {
#pragma unroll
      for (int s = 0; s < KS; ++s) qf[s].q = v4i{0, 0, 0, 0};
    } else if (rope_cos) {
      constexpr int HD = D / 2;
#pragma unroll
      for (int s = 0; s < KS / 2; ++s) {
        // elements d = 32s + 8grp + j (< D/2) and their partners d + D/2 (fragment s + KS/2, slot j);
        // the 8 table entries of d are contiguous (16-byte aligned tables, host-checked)
        const float4* cp = reinterpret_cast<const float4*>(rope_cos + qpos * HD + 32 * s + 8 * grp);
        const float4* sp = reinterpret_cast<const float4*>(rope_sin + qpos * HD + 32 * s + 8 * grp);
        const float4 c0 = cp[0], c1 = cp[1], s0 = sp[0], s1 = sp[1];
        const float cs[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
        const float sn[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
        float y1[8], y2[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float x1 = bf16f(qf[s].h[j]), x2 = bf16f(qf[s + KS / 2].h[j]);
          y1[j] = __fadd_rn(__fmul_rn(x1, cs[j]), __fmul_rn(-x2, sn[j]));
          y2[j] = __fadd_rn(__fmul_rn(x2, cs[j]), __fmul_rn(x1, sn[j]));
        }
#pragma unroll
        for (int j = 0; j < 8; j += 2) {  // round to bf16, nearest even (v_cvt_pk_bf16_f32)
          qf[s].u[j / 2] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t){y1[j], y1[j + 1]}, bf16x2_t));
          qf[s + KS / 2].u[j / 2] =
              __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t){y2[j], y2[j + 1]}, bf16x2_t));
        }
      }
    }
  }

  // keys needed by the block's last valid query; loads past them read zeros (no stale cache rows enter
  // the P V product, where a masked p = 0 would still meet them)
  const int64_t kend = start + (i0 + 16 < T ? i0 + 16 : T);
  const int nkb = (int)((kend + KB - 1) / KB);
  const int64_t slice = ((int64_t)b * hkv + g) * max_len * D;  // element offset of the (b, g) cache slice
  const buf_t kb_ = make_buf(kc + slice, (uint32_t)(kend * D * 2));
  const buf_t vb_ = make_buf(vc + slice, (uint32_t)(kend * D * 2));

  f32x4_t o[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) o[db] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  float m_run = -__builtin_inff(), l_run = 0.0f;

  // Tile staging, software-pipelined: the global loads of block kb + 1 are issued right after block kb
  // is written to LDS, so they are in flight while block kb is computed.  Trip counts are compile-time
  // constants, so every load of a tile is issued before the first LDS write waits for one.
  constexpr int KP = KB * (D / 8);        // 16-byte pieces of the K tile
  constexpr int KIT = (KP + NT - 1) / NT;
  constexpr int VP = (KB / 2) * (D / 8);  // (key pair, 8-element chunk) items of the V tile
  constexpr int VIT = (VP + NT - 1) / NT;
  v4i kreg[KIT];
  Frag8 va[VIT], vb2[VIT];
  auto load_tile = [&](int key0) {
#pragma unroll
    for (int it = 0; it < KIT; ++it) {
      const int p = t + it * NT;
      if (KP % NT == 0 || p < KP) {
        const int r = p / (D / 8), c = p % (D / 8);
        kreg[it] = buf_load16(kb_, (uint32_t)(((key0 + r) * D + 8 * c) * 2));
      }
    }
    // V: 16 consecutive lanes take 16 consecutive key pairs of one 8-element chunk, the next 16 lanes
    // the next chunk, so the transposed row stores below spread over all banks (rows 8c + j of chunks
    // c and c + 1 sit 16 banks apart) while each key row is still read as 64-byte pieces
#pragma unroll
    for (int it = 0; it < VIT; ++it) {
      const int p = t + it * NT;
      if (VP % NT == 0 || p < VP) {
        const int rest = p / 16, c = rest % (D / 8);
        const int r = 2 * ((p % 16) + 16 * (rest / (D / 8)));
        va[it].q = buf_load16(vb_, (uint32_t)(((key0 + r) * D + 8 * c) * 2));
        vb2[it].q = buf_load16(vb_, (uint32_t)(((key0 + r + 1) * D + 8 * c) * 2));
      }
    }
  };
  auto store_tile = [&]() {
#pragma unroll
    for (int it = 0; it < KIT; ++it) {
      const int p = t + it * NT;
      if (KP % NT == 0 || p < KP) {
        const int r = p / (D / 8), c = p % (D / 8);
        *reinterpret_cast<v4i*>(&ks_[r * KROW + 8 * c]) = kreg[it];
      }
    }
#pragma unroll
    for (int it = 0; it < VIT; ++it) {
      const int p = t + it * NT;
      if (VP % NT == 0 || p < VP) {
        const int rest = p / 16, c = rest % (D / 8);
        const int r = 2 * ((p % 16) + 16 * (rest / (D / 8)));
#pragma unroll
        for (int jj = 0; jj < 8; ++jj)
          *reinterpret_cast<uint32_t*>(&vs_[(8 * c + jj) * VROW + r]) =
              (uint32_t)va[it].h[jj] | ((uint32_t)vb2[it].h[jj] << 16);
      }
    }
  };

  load_tile(0);
  for (int kb = 0; kb < nkb; ++kb) {
    const int key0 = kb * KB;
    __syncthreads();  // the previous block's tiles are no longer read
    store_tile();
    __syncthreads();
    if (kb + 1 < nkb) load_tile(key0 + KB);

    // S^T = K Q^T for the 4 sub-blocks of 16 keys
    f32x4_t s[4];
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) {
      s[nb] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        Frag8 a;
        a.q = *reinterpret_cast<const v4i*>(&ks_[(16 * nb + (lane & 15)) * KROW + 32 * k + 8 * grp]);
        s[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, qf[k].v, s[nb], 0, 0, 0);
      }
    }
    // scale, causal mask (only blocks reaching past the workgroup's first query), block max
    float bmax = -__builtin_inff();
    const bool masked = key0 + KB - 1 > qpos_first;  // uniform
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = key0 + 16 * nb + 4 * grp + i;
        const float v = !masked || key <= qpos32 ? s[nb][i] * scale : -__builtin_inff();
        s[nb][i] = v;
        bmax = fmaxf(bmax, v);
      }
    bmax = fmaxf(bmax, xor_lanes_f32<16>(bmax));
    bmax = fmaxf(bmax, xor_lanes_f32<32>(bmax));
    const float m_new = fmaxf(m_run, bmax);  // finite: key 0 <= qpos is in block 0
    const float alpha = __expf(m_run - m_new);
    float psum = 0.0f;
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float p = __expf(s[nb][i] - m_new);
        s[nb][i] = p;
        psum += p;
      }
    psum += __shfl_xor(psum, 16, 64);
    psum += __shfl_xor(psum, 32, 64);
    l_run = l_run * alpha + psum;
    m_run = m_new;
#pragma unroll
    for (int db = 0; db < DB; ++db) o[db] *= alpha;

    // O^T += V^T P^T over two chunks of 32 keys (slots j < 4: sub-block 2c, j >= 4: sub-block 2c + 1)
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      Frag8 phi, plo;  // hi = bf16(p), lo = bf16(p - hi), both round-to-nearest-even (v_cvt_pk_bf16_f32)
#pragma unroll
      for (int j = 0; j < 8; j += 2) {
        const float p0 = s[2 * c + (j >> 2)][j & 3], p1 = s[2 * c + (j >> 2)][(j & 3) + 1];
        const uint32_t hi = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t){p0, p1}, bf16x2_t));
        const float r0 = p0 - __uint_as_float(hi << 16), r1 = p1 - __uint_as_float(hi & 0xffff0000u);
        phi.u[j / 2] = hi;
        plo.u[j / 2] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t){r0, r1}, bf16x2_t));
      }
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        const uint16_t* vr = &vs_[(16 * db + (lane & 15)) * VROW + 32 * c + 4 * grp];
        Frag8 a;
        const uint2 lo4 = *reinterpret_cast<const uint2*>(vr);
        const uint2 hi4 = *reinterpret_cast<const uint2*>(vr + 16);
        a.u[0] = lo4.x;
        a.u[1] = lo4.y;
        a.u[2] = hi4.x;
        a.u[3] = hi4.y;
        o[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, phi.v, o[db], 0, 0, 0);
        o[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, plo.v, o[db], 0, 0, 0);
      }
    }
  }

  if (!qvalid) return;
  // lane holds O^T[16db + 4grp + i][qi]: four consecutive elements of the output row per db
  uint16_t* orow = out + ((int64_t)b * T + qi) * ldo + (int64_t)h * D;
  const float inv_l = 1.0f / l_run;
#pragma unroll
  for (int db = 0; db < DB; ++db) {
    uint2 v;
    v.x = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t){o[db][0] * inv_l, o[db][1] * inv_l}, bf16x2_t));
    v.y = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t){o[db][2] * inv_l, o[db][3] * inv_l}, bf16x2_t));
    *reinterpret_cast<uint2*>(orow + 16 * db + 4 * grp) = v;
  }
}

template <int D, int G>
hipError_t launch_prefill_g(const uint16_t* q, int64_t ldq, const float* rc, const float* rs, const uint16_t* kc,
                            const uint16_t* vc, int64_t max_len, int b, int hkv, int t, int64_t start, float scale,
                            uint16_t* out, int64_t ldo, hipStream_t s) {
  // Few workgroups (up to one of 16 tokens per CU): the 16-token form up to so many keys that a workgroup's own chain
  // is what the call takes.  Swept on MI355X, both forms, over D 64 / 128, G 1 .. 8, (kv heads, batch) 1 x 1 .. 8 x 1,
  // 1 x 8 and 3 x 4, 20 (tokens, start) of 16 .. 6033 keys.  The line lies where the 32-token form gets ahead and keeps
  // every point below 4096 keys within 6% of the better form (16- against 32-token form, one kv head, us):
  //   G = 1: 128 + 0 tokens 8.5 against 9.1 at D = 64, 10.7 against 11.7 at D = 128; 160 + 0 the other way by 7-12%, as
  //     is a chunk of fewer tokens behind older keys;
  //   D = 64: G = 3 loses from 160 keys (8-11%, 17-32% at 256 .. 600); chunks of up to 512 tokens of G = 5 .. 7 win up to
  //     4096 (64 + 2000 tokens 53.6 against 57.2 at G = 5; 1024 + 0 33.0 against 31.5, and at 6033 keys and 24
  //     workgroups or more they lose 6-12%); the others lose from 512;
  //   D = 128: G = 4, 5 and 8 win throughout (33 + 6000 tokens 3, 11 and 0%), G = 6 and 7 up to 1024, G = 2 and 3 up to
  //     512 (one CU round more, 8 x 4 heads, 1000 tokens, 39.1 against 49.8 the other way).
  const int64_t keys16 = D == 64 ? (G == 3 ? 128 : G >= 5 && G <= 7 && t <= 512 ? 4096 : 512)
                                 : (G == 4 || G == 5 || G == 8 ? INT64_MAX : G >= 6 ? 1024 : 512);
  const int64_t wg16 = (int64_t)((t + 15) / 16) * hkv * b;
  if (wg16 <= 256 && (G == 1 ? t > 64 && start + t <= 128 : start + t <= keys16)) {
    hipLaunchKernelGGL((gqa_prefill16_kernel<D, G>), dim3((t + 15) / 16, hkv, b), dim3(64 * G), 0, s, q, ldq, rc, rs,
                       kc, vc, max_len, hkv, t, start, scale, out, ldo);
    return hipGetLastError();
  }
  constexpr int QW = G == 1 ? 4 : G == 2 ? 2 : 1;  // three waves or more share each staged K and V tile
  const int64_t nqb = (t + 32 * QW - 1) / (32 * QW), nhb = (int64_t)hkv * b;
  if (nqb * nhb > INT32_MAX) return hipErrorInvalidValue;
  hipLaunchKernelGGL((gqa_prefill_kernel<D, G, QW>), dim3((unsigned)(nqb * nhb)), dim3(64 * G * QW), 0, s, q, ldq, rc, rs, kc, vc,
                     max_len, hkv, t, start, scale, out, ldo, (int)nhb, (int)nqb);
  return hipGetLastError();
}

template <int D>
hipError_t launch_prefill_d(int g, const uint16_t* q, int64_t ldq, const uint16_t* kn, int64_t ldk, const uint16_t* vn,
                            int64_t ldv, const float* rc, const float* rs, uint16_t* kc, uint16_t* vc, int64_t max_len,
                            int b, int hkv, int t, int64_t start, float scale, uint16_t* out, int64_t ldo,
                            hipStream_t s) {
  // 16-byte path when the key / value rows allow it (q|k|v column slices of one projection output do)
  const bool vec = (uintptr_t)kn % 16 == 0 && (uintptr_t)vn % 16 == 0 && ldk % 8 == 0 && ldv % 8 == 0;
  hipLaunchKernelGGL((gqa_append_kernel<D>), dim3(t, b), dim3(256), 0, s, kn, ldk, vn, ldv, rc, rs, kc, vc, max_len,
                     hkv, t, start, vec);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
#define WFB_PF_G(GG) \
  case GG: return launch_prefill_g<D, GG>(q, ldq, rc, rs, kc, vc, max_len, b, hkv, t, start, scale, out, ldo, s)
  switch (g) {
    WFB_PF_G(1);
    WFB_PF_G(2);
    WFB_PF_G(3);
    WFB_PF_G(4);
    WFB_PF_G(5);
    WFB_PF_G(6);
    WFB_PF_G(7);
    WFB_PF_G(8);
    default: return hipErrorInvalidValue;
  }
#undef WFB_PF_G
}

}  // namespace

hipError_t launch_gqa_prefill(int d, int g, const void* q, int64_t ldq, const void* kn, int64_t ldk, const void* vn,
                              int64_t ldv, const float* rc, const float* rs, void* kc, void* vc, int64_t max_len, int b,
                              int hkv, int t, int64_t start, float scale, void* out, int64_t ldo, hipStream_t s) {
  auto u16 = [](const void* p) { return reinterpret_cast<const uint16_t*>(p); };
  auto w16 = [](void* p) { return reinterpret_cast<uint16_t*>(p); };
  if (d == 64)
    return launch_prefill_d<64>(g, u16(q), ldq, u16(kn), ldk, u16(vn), ldv, rc, rs, w16(kc), w16(vc), max_len, b, hkv,
                                t, start, scale, w16(out), ldo, s);
  if (d == 128)
    return launch_prefill_d<128>(g, u16(q), ldq, u16(kn), ldk, u16(vn), ldv, rc, rs, w16(kc), w16(vc), max_len, b, hkv,
                                 t, start, scale, w16(out), ldo, s);
  return hipErrorInvalidValue;
}

}  // namespace wfb
