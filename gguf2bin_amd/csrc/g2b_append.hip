// g2b_append.hip - RoPE + KV append for gfx950.
//
// Replaces /root/reference/src/l5_model.c:505-516: QK-RMSNorm when the layer
// has norm weights (l3_math.c:107-114), apply_rope on q and on the new k
// (l5_model.c:448-452, l3_math.c:64-102), then kv_store
// (l5_model.c:235-247) which memcpy's F32 rows or quantises Q8_0 rows
// (l5_model.c:49-59).  The cos/sin table comes from the host C library (the
// same powf/cosf/sinf the reference calls), so rotated values and therefore
// the stored bytes are bit-exact; the quantiser follows the reference
// operation by operation (IEEE division, round half away from zero,
// truncating fp16 scale).  k_append_batch is two rows per (sequence, layer),
// and k_append_rows takes the shapes and alignments that k_append_run does
// not: both favour plain code over speed, one workgroup per row pair.
#include "g2b_internal.h"

namespace g2b {

// LDS: kr[nkv], then inv[n_heads]
__global__ __launch_bounds__(kThreads) void k_append_batch(AppendParams p) {
  extern __shared__ float kr[];
  const int seq = blockIdx.x, li = blockIdx.y;
  const SeqDev sd = p.seqs ? p.seqs[seq] : p.one;
  const size_t slot = (size_t)li * (size_t)p.n_seq + (size_t)seq;
  const size_t nq = (size_t)p.sh.n_heads * p.sh.head_dim;
  const size_t nkv = (size_t)p.sh.n_kv_heads * p.sh.head_dim;
  append_row(p.sh, sd, p.layer0 + li, sd.pos, p.k_in + slot * nkv, p.v_in + slot * nkv,
             p.q_in + slot * nq, p.q_rot + slot * nq, p.rope, p.norm, kr, kr + nkv);
}

__global__ __launch_bounds__(kThreads) void k_append_rows(AppendParams p, int layer) {
  extern __shared__ float kr[];
  const int r = blockIdx.x;
  const size_t nkv = (size_t)p.sh.n_kv_heads * p.sh.head_dim;
  append_row(p.sh, p.one, layer, p.pos0 + r, p.k_in + (size_t)r * nkv,
             p.v_in + (size_t)r * nkv, nullptr, nullptr, p.rope, p.norm, kr, kr + nkv);
}

// The prompt's rows, head_dim 64, 128 or 256 and 16-byte aligned operands.
// Bound by HBM once the rows are many (8 bytes of k and v in per element, 2.1
// (Q8_0) or 8 (F32) out); k_append_rows above, a row per workgroup with one
// thread per block and 2-byte stores, ran 2039 rows of 1024 elements into
// Q8_0 (21 MB) in 24.2 us, this one in 7.4 us (8.3 us with a division per
// element).
//
// A thread holds elements [8i, 8i + 8) and [hd/2 + 8i, hd/2 + 8i + 8) of one
// head of one row of k or v: both members of every RoPE pair, NEOX or LLaMA,
// and a quarter of two Q8_0 blocks, whose other quarters sit in the
// neighbouring lanes.  A workgroup takes rows_wg consecutive rows - one
// contiguous run of each cache - and Q8_0 blocks go to LDS first, so that the
// run leaves in 16-byte pieces (4-byte ones where rows are not whole pieces).
// The arithmetic is append_row's, element by element; QK-RMSNorm's sum of
// squares runs left to right over a head's lanes, each lane's eight products
// added in turn to the sum the lane before it hands on.
__device__ __forceinline__ float quad_max(float x) {  // '>' skips NaN, as q8_quant_block does
  float o = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0xB1, 0xF, 0xF, true));
  if (o > x) x = o;
  o = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x4E, 0xF, 0xF, true));
  return o > x ? o : x;
}

// Eight of a block's elements (part: which), the block's other 24 in the
// other lanes of the quad, into the 34-byte block at dst (LDS, 2-byte
// aligned).  Every byte is q8_quant_block's: |x / d| is at most 190 (d >= the
// smallest subnormal, x <= amax), or NaN, which it stores as 0.
//
// The workgroups of a launch all quantise at the same time, so the 16
// divisions of a thread are time that nothing hides.  They share the
// correctly rounded y = 1 / d: x * y, then two corrections by its remainder
// (an FMA each for remainder and correction), give the correctly rounded
// quotient (Markstein, Computation of elementary functions on the IBM RISC
// System/6000, 1990: with y correctly rounded and the quotient before it
// within an ulp, the last step rounds correctly) as long as no remainder is
// subnormal; other d take the division.  Half away from zero: the
// truncation of the quotient plus the largest float below a half with its
// sign (exact for |x| below 2^22, also just below 0.5).
__device__ __forceinline__ void quant_quarter(const float (&x)[8], int part, uint8_t *dst) {
  float amax = 0.f;
#pragma unroll
  for (int j = 0; j < 8; j++) {
    const float a = fabsf(x[j]);
    if (a > amax) amax = a;
  }
  amax = quad_max(amax);
  float d = __fdiv_rn(amax, 127.f);
  if (!(d > 0.f)) d = 1e-10f;
  uint16_t *o = reinterpret_cast<uint16_t *>(dst);
  if (part == 0) o[0] = (uint16_t)f32_to_half_trunc(d);
  float r[8];
  if (d >= 0x1p-90f && d <= 0x1p100f) {
    const float y = __fdiv_rn(1.f, d);
#pragma unroll
    for (int j = 0; j < 8; j++) {
      float q = x[j] * y;
      q = fmaf(fmaf(-q, d, x[j]), y, q);
      r[j] = fmaf(fmaf(-q, d, x[j]), y, q);
    }
  } else {
#pragma unroll
    for (int j = 0; j < 8; j++) r[j] = __fdiv_rn(x[j], d);
  }
#pragma unroll
  for (int j = 0; j < 8; j += 2) {
    int q[2];
#pragma unroll
    for (int k = 0; k < 2; k++) {
      const float t = r[j + k] + copysignf(0x1.fffffep-2f, r[j + k]);
      const int n = t == t ? (int)t : 0;
      q[k] = n > 127 ? 127 : (n < -127 ? -127 : n);
    }
    o[1 + 4 * part + j / 2] = (uint16_t)((uint32_t)(q[0] & 0xff) | ((uint32_t)(q[1] & 0xff) << 8));
  }
}

template <int FMT, int HD>
__global__ __launch_bounds__(kThreads) void k_append_run(AppendParams p, int layer, int n_rows,
                                                         int rows_wg) {
  constexpr int NT = HD / 16, half = HD / 2;  // NT: lanes per head
  extern __shared__ __align__(16) uint8_t run[];  // Q8_0: the K rows, then the V rows
  const int r0 = blockIdx.x * rows_wg, nr = min(rows_wg, n_rows - r0);
  const int nkvh = p.sh.n_kv_heads, per_row = nkvh * NT;
  const size_t nkv = (size_t)nkvh * HD;
  const uint32_t row = p.sh.row_bytes;
  const size_t off = ((size_t)layer * (size_t)p.one.ctx_cap + (size_t)(p.pos0 + r0)) * row;
  const float *wk = norm_weights(p.norm, layer, 1, HD);
  const bool llama = p.sh.arch_llama != 0;
  // (a head's NT lanes are consecutive and always active together)
  for (int it = threadIdx.x; it < 2 * nr * per_row; it += kThreads) {
    const bool is_v = it >= nr * per_row;
    const int e = is_v ? it - nr * per_row : it;
    const int r = e / per_row, h = (e - r * per_row) / NT, i = e & (NT - 1);
    const float *src = (is_v ? p.v_in : p.k_in) + (size_t)(r0 + r) * nkv + (size_t)h * HD + 8 * i;
    float a[8], b[8];
#pragma unroll
    for (int j = 0; j < 8; j += 4) {
      *reinterpret_cast<float4 *>(a + j) = *reinterpret_cast<const float4 *>(src + j);
      *reinterpret_cast<float4 *>(b + j) = *reinterpret_cast<const float4 *>(src + half + j);
    }
    if (!is_v) {
      const float *cs = p.rope ? p.rope + (size_t)(p.pos0 + r0 + r) * HD : nullptr;
      float c[16];  // LLaMA: the a pairs' cos and sin, then the b pairs'
      if (cs) {
        const float *ca = cs + (llama ? 8 * i : 16 * i), *cb = llama ? cs + half + 8 * i : ca + 8;
#pragma unroll
        for (int j = 0; j < 8; j += 4) {
          *reinterpret_cast<float4 *>(c + j) = *reinterpret_cast<const float4 *>(ca + j);
          *reinterpret_cast<float4 *>(c + 8 + j) = *reinterpret_cast<const float4 *>(cb + j);
        }
      }
      if (wk) {
        const int lane0 = (int)(threadIdx.x & 63) & ~(NT - 1);
        float ss = 0.f;
#pragma unroll
        for (int hf = 0; hf < 2; hf++) {
          float sq[8];
#pragma unroll
          for (int j = 0; j < 8; j++) sq[j] = hf ? b[j] * b[j] : a[j] * a[j];
#pragma unroll
          for (int t = 0; t < NT; t++) {
            float s = ss;
#pragma unroll
            for (int j = 0; j < 8; j++) s = s + sq[j];
            ss = __shfl(s, lane0 + t);
          }
        }
        const float inv = __fdiv_rn(1.f, sqrtf(__fdiv_rn(ss, (float)HD) + p.norm.eps));
#pragma unroll
        for (int j = 0; j < 8; j++) {
          const float wa = wk[8 * i + j] * a[j], wb = wk[half + 8 * i + j] * b[j];
          a[j] = wa * inv;
          b[j] = wb * inv;
        }
      }
      if (cs) {
        if (llama) {
#pragma unroll
          for (int j = 0; j < 8; j += 2) {
            rope_pair(a[j], a[j + 1], c[j], c[j + 1]);
            rope_pair(b[j], b[j + 1], c[8 + j], c[9 + j]);
          }
        } else {
#pragma unroll
          for (int j = 0; j < 8; j++) rope_pair(a[j], b[j], c[2 * j], c[2 * j + 1]);
        }
      }
    }
    if constexpr (FMT == 1) {
      uint8_t *blk = run + (size_t)(is_v ? nr + r : r) * row + (size_t)h * (HD / 32 * 34);
      quant_quarter(a, i & 3, blk + 34 * (i >> 2));
      quant_quarter(b, i & 3, blk + 34 * (half / 32 + (i >> 2)));
    } else {
      float *dst = reinterpret_cast<float *>((is_v ? p.one.v : p.one.k) + off + (size_t)r * row) +
                   h * HD + 8 * i;
#pragma unroll
      for (int j = 0; j < 8; j += 4) {
        *reinterpret_cast<float4 *>(dst + j) = *reinterpret_cast<const float4 *>(a + j);
        *reinterpret_cast<float4 *>(dst + half + j) = *reinterpret_cast<const float4 *>(b + j);
      }
    }
  }
  if constexpr (FMT == 1) {
    __syncthreads();
    const uint32_t bytes = (uint32_t)nr * row;
    if ((row & 15u) == 0) {
      for (uint32_t o = 16u * threadIdx.x; o < 2u * bytes; o += 16u * kThreads)
        *reinterpret_cast<uint4 *>(o < bytes ? p.one.k + off + o : p.one.v + off + (o - bytes)) =
            *reinterpret_cast<const uint4 *>(run + o);
    } else {
      for (uint32_t o = 4u * threadIdx.x; o < 2u * bytes; o += 4u * kThreads)
        *reinterpret_cast<uint32_t *>(o < bytes ? p.one.k + off + o : p.one.v + off + (o - bytes)) =
            *reinterpret_cast<const uint32_t *>(run + o);
    }
  }
}

template <int FMT, int HD>
static hipError_t launch_append_run(const AppendParams &p, int layer, int n_rows, hipStream_t s) {
  // about 256 lanes of work per workgroup
  const int nkv = p.sh.n_kv_heads * HD, rows_wg = nkv >= 2048 ? 1 : 2048 / nkv;
  const size_t lds = FMT ? (size_t)2 * rows_wg * p.sh.row_bytes : 0;
  hipLaunchKernelGGL((k_append_run<FMT, HD>), dim3((n_rows + rows_wg - 1) / rows_wg),
                     dim3(kThreads), lds, s, p, layer, n_rows, rows_wg);
  return hipGetLastError();
}

static size_t append_lds_bytes(const ShapeDev &sh) {
  return ((size_t)sh.n_kv_heads * sh.head_dim + (size_t)sh.n_heads) * sizeof(float);
}

hipError_t launch_append_batch(const AppendParams &p, int n_layers, hipStream_t s) {
  const size_t lds = append_lds_bytes(p.sh);
  hipLaunchKernelGGL(k_append_batch, dim3(p.n_seq, n_layers), dim3(kThreads), lds, s, p);
  return hipGetLastError();
}

hipError_t launch_append_rows(const AppendParams &p, int layer, int n_rows, hipStream_t s) {
  const uintptr_t at = (uintptr_t)p.k_in | (uintptr_t)p.v_in | (uintptr_t)p.one.k |
                       (uintptr_t)p.one.v;
  if ((at & 15u) == 0) {
    switch (p.sh.head_dim) {
      case 64:
        return p.sh.kv_q8 ? launch_append_run<1, 64>(p, layer, n_rows, s)
                          : launch_append_run<0, 64>(p, layer, n_rows, s);
      case 128:
        return p.sh.kv_q8 ? launch_append_run<1, 128>(p, layer, n_rows, s)
                          : launch_append_run<0, 128>(p, layer, n_rows, s);
      case 256:
        return p.sh.kv_q8 ? launch_append_run<1, 256>(p, layer, n_rows, s)
                          : launch_append_run<0, 256>(p, layer, n_rows, s);
    }
  }
  const size_t lds = append_lds_bytes(p.sh);
  hipLaunchKernelGGL(k_append_rows, dim3(n_rows), dim3(kThreads), lds, s, p, layer);
  return hipGetLastError();
}

}  // namespace g2b
