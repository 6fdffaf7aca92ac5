// g2b_wide.h - k_wide, the decode kernel with one KV head per workgroup and
// both products on the matrix cores.  Included only by g2b_wide_inst.hip (one
// KV format and head_dim at a time).
//
// Replaces the RoPE / append / score / softmax / V loops of l5_model.c:505-577
// in one launch.  It serves the shapes that k_layer and k_tiles do not take -
// wide GQA groups (up to 16 q heads per KV head), more KV heads than a wave's
// lanes hold, rows of any length, head_dim 64, 128 or 256 - and the calls that
// are bound by latency (one layer of few positions: g2b_api.hip has the rule).
//
// Workgroup (split, KV head, sequence and layer): four waves, each streaming
// every fourth 16-position tile of the split; no barrier falls inside the
// stream, and a wave has two tiles of registers, one being consumed while the
// next comes.
//
// Latency.  One launch is a chain of dependent steps, and every memory round
// trip in it that does not overlap another shows (~1 us each): so the launch's
// parameters are read in one batch, the descriptor and the layer's norm flag
// as scalars, and then everything the setup needs - q, cos/sin, norm weights,
// the new k and v - is requested before the first two tiles, in that order,
// because waits count in issue order: the setup runs while the tiles come.
// The setup is spread over the waves (q from wave 0 on, v on wave 2, k on wave
// 3) and needs one barrier.  One KV head's share of q (1 KB for two heads of
// 128) keeps it short; k_layer's covers all heads in every workgroup.
//
// With G q heads to a KV head the arithmetic is G x 4 flop per K or V element
// - 15 per byte of Q8_0 at G = 8, above what the VALU has per HBM byte:
//   scores, Q8_0: v_mfma_i32_16x16x32_i8 per (block, four heads): A row
//     4h + p = digit plane p of head h, B = the block's quants of 16
//     positions, exact int32 sums combined in float64 (as k_tiles);
//   scores, F32:  v_mfma_f32_16x16x4_f32: A row 4h + i = head 4i + h (16
//     heads), B = 16 positions; step 4j + i takes dims 16j + 4*quarter + i,
//     so that a lane's loads are 16-byte pieces and a position's four lanes
//     read 64 consecutive bytes;
//   V: v_mfma_f32_4x4x1_16b_f32, lane = (slot of positions, four dims), as
//     k_tiles: p (x the V block's scale) of four heads against the lane's own
//     V values, the positions dealt to 64 / (head_dim / 4) slots.
// Either way lane (quarter, col) of a score holds head 4*set + quarter at
// position col of the tile, and p reaches the V lanes through LDS.
//
// Q8_0 rows are read in dword windows straight from HBM (rows are whole
// dwords: head_dim is a multiple of 64): a lane's quants of a block are three
// dwords that start two bytes (even blocks) or four (odd blocks) before them,
// so that no window leaves the row.  Neighbouring windows share lines, which
// the vector cache serves (default policy), and so do neighbouring KV heads of
// a row (136 bytes each): the grid puts the KV heads of a split on one XCD
// (launch_wide_sets), whose L2 then fetches each line once.
//
// What bounds it: HBM in large batches, else that chain.  Measured per layer
// against the three-pass kernel that wide groups took before (one thread per
// position, every element converted on its own for every q head): 16 / 2
// heads of 128, Q8_0, 8 sequences of 1000-4000 positions (11 MB), append +
// decode + combine 786 us; with several KV heads per workgroup and the setup
// ahead of the tiles 20.0; now 16.6.
#pragma once
#include "g2b_layer.h"

namespace g2b {

constexpr int kWideTile = 16;  // positions per tile (the MFMA's columns)

// Floats between two heads' and two blocks' p in a wave's exchange (16 + 4
// and + 4: the V lanes' reads of four heads and of several blocks spread over
// the LDS banks).
constexpr int kWidePxHead = kWideTile + 4;
__host__ __device__ constexpr int wide_px_block(int sets) { return 4 * sets * kWidePxHead + 4; }
// Blocks of p per tile: F32 has one (no scales), Q8_0 one per 32 dims.
__host__ __device__ constexpr int wide_px_blocks(int fmt, int hd) { return fmt ? hd / 32 : 1; }
// A wave's exchange, and the rescale factors behind it.
__host__ __device__ constexpr int wide_px_floats(int fmt, int hd, int sets) {
  return wide_px_blocks(fmt, hd) * wide_px_block(sets) + 4 * sets;
}

// Sets of four q heads (template instances): 1, 2 or 4.
__host__ __device__ inline int wide_sets(int group) { return group <= 4 ? 1 : group <= 8 ? 2 : 4; }

// LDS: the waves' exchanges, the digit planes of the group's q and their units
// (Q8_0) or the rotated, scaled q (F32), the new K and V rows of the head.  The
// merge of the waves reuses it all.
struct WideLds {
  uint32_t q, rows, row_pad, total;
};
template <int FMT, int HD, int SETS>
__host__ __device__ constexpr WideLds wide_lds() {
  WideLds l{};
  l.q = ((uint32_t)(kWavesPerSplit * wide_px_floats(FMT, HD, SETS)) * 4u + 15u) & ~15u;
  const uint32_t qb = 4u * SETS * (FMT ? (uint32_t)dig_dwords<32>(HD / 32) : (uint32_t)HD) * 4u;
  l.rows = (l.q + qb + 15u) & ~15u;
  l.row_pad = ((FMT ? HD / 32 * 34u : HD * 4u) + 15u) & ~15u;
  const uint32_t end = l.rows + 2u * l.row_pad;
  const uint32_t merge = (uint32_t)(kWavesPerSplit * 4 * SETS * (kPartHead + HD)) * 4u;
  l.total = end > merge ? end : merge;
  return l;
}

// One tile of a wave's KV head in registers.
template <int FMT, int HD>
struct WideRaw;
template <int HD>
struct WideRaw<1, HD> {
  static constexpr int NB = HD / 32, NS = (NB + 3) / 4, VP = HD / 16;
  uint32_t k[NB][3];          // quants 8*quarter .. of each block, at position col
  uint32_t ks[NS], vs[NS];    // the dwords with the scales of block 4u + quarter, position col
  uint32_t v[VP][2];          // the lane's four dims at its slot's positions
};
template <int HD>
struct WideRaw<0, HD> {
  static constexpr int VP = HD / 16;
  f32x4 k[HD / 16], v[VP];
};

// (dword-aligned pair of dwords; a vector of three would be loaded as four)
typedef uint32_t u32x2a __attribute__((ext_vector_type(2), aligned(4)));

// The largest of N consecutive lanes' x, NaN skipped ('>', as q8_quant_block).
template <int N>
__device__ __forceinline__ float lanes_max_gt(float x) {
  float o = dpp_f<0xB1>(x);
  x = o > x ? o : x;
  o = dpp_f<0x4E>(x);
  x = o > x ? o : x;
  if constexpr (N == 8) {
    o = dpp_f<0x141>(x);
    x = o > x ? o : x;
  }
  return x;
}

// Four elements of a Q8_0 block whose largest |x| is amax, at element e of it,
// into the block at dst (LDS, 2-byte aligned); the scale with element 0.  The
// bytes of q8_quant_block.
__device__ __forceinline__ void wide_quant4(const float (&x)[4], float amax, int e, uint8_t *dst) {
  float d = __fdiv_rn(amax, 127.f);
  if (!(d > 0.f)) d = 1e-10f;
  uint16_t *o = reinterpret_cast<uint16_t *>(dst);
  if (e == 0) o[0] = (uint16_t)f32_to_half_trunc(d);
#pragma unroll
  for (int j = 0; j < 4; j += 2) {
    int q[2];
#pragma unroll
    for (int k = 0; k < 2; k++) {
      const int n = lround_i32_like_host(__fdiv_rn(x[j + k], d));
      q[k] = n > 127 ? 127 : (n < -127 ? -127 : n);
    }
    o[1 + (e + j) / 2] = (uint16_t)((uint32_t)(q[0] & 0xff) | ((uint32_t)(q[1] & 0xff) << 8));
  }
}

template <int FMT, int HD, int SETS>
__global__ __launch_bounds__(kThreads) void k_wide(DecodeParams P, int z0) {
  constexpr int NB = HD / 32, VP = HD / 16, DL = HD / 4;  // DL: V lanes per slot
  constexpr int GPH = HD / 8;                             // setup lanes per head
  constexpr int QG = (4 * SETS * GPH + kThreads - 1) / kThreads;  // q groups per thread
  constexpr int NBX = wide_px_blocks(FMT, HD), PXB = wide_px_block(SETS);
  constexpr uint32_t HB = FMT ? HD / 32 * 34 : HD * 4;    // a KV head's bytes of a row
  constexpr int pstr = kPartHead + HD;
  constexpr int half = HD / 2;
  constexpr WideLds ll = wide_lds<FMT, HD, SETS>();
  extern __shared__ __align__(16) uint8_t lds[];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, col = lane & 15, quarter = lane >> 4;

  // the launch's parameters, in one batch of scalar loads
  const int nkvh = P.sh.n_kv_heads, n_heads = P.sh.n_heads, n_seq = P.n_seq;
  const uint32_t row = P.sh.row_bytes;
  const int split_len = P.split_len, max_splits = P.max_splits, layer0 = P.layer0;
  const float *q_in = P.q_in, *k_in = P.k_in, *v_in = P.v_in, *rope = P.rope, *norm_w = P.norm.w;
  const int32_t *norm_on = P.norm.on;
  const SeqDev *seqs = P.seqs;
  const float qscale = P.qscale, eps = P.norm.eps;
  float *const att = P.att;
  const int llama = P.sh.arch_llama, rope_on = P.sh.rope_on, n_layers_call = P.n_layers_call;
  SeqDev sd = P.one;
  asm volatile("" ::"s"(nkvh), "s"(n_heads), "s"(n_seq), "s"(row), "s"(split_len), "s"(max_splits),
               "s"(layer0), "s"(q_in), "s"(k_in), "s"(v_in), "s"(rope), "s"(norm_w), "s"(norm_on),
               "s"(seqs), "s"(qscale), "s"(eps), "s"(sd.pos), "s"(sd.ctx_cap), "s"(sd.k), "s"(sd.v),
               "s"(att), "s"(llama), "s"(rope_on), "s"(n_layers_call));
  const int u = z0 + (int)blockIdx.z;  // li * n_seq + seq
  const int li = n_layers_call > 1 ? u / n_seq : 0, seq = u - li * n_seq;
  const int kvh = blockIdx.y, layer = layer0 + li;
  int on = 0;
  if (norm_w) on = ((const __attribute__((address_space(4))) int32_t *)norm_on)[layer];
  if (seqs) {
    typedef uint32_t u32x8 __attribute__((ext_vector_type(8)));
    const u32x8 d = *(const __attribute__((address_space(4))) u32x8 *)(seqs + seq);
    sd.pos = (int32_t)d[0];
    sd.ctx_cap = (int32_t)d[1];
    sd.k = (uint8_t *)((uint64_t)d[4] | ((uint64_t)d[5] << 32));
    sd.v = (uint8_t *)((uint64_t)d[6] | ((uint64_t)d[7] << 32));
  }
  const int G = n_heads / nkvh;
  // (rotated by the sequence: with a multiple of eight splits, the sequences'
  // first splits would all be on one XCD)
  int split = (int)blockIdx.x + (gridDim.x >= 8 ? (u & 7) : 0);
  if (split >= (int)gridDim.x) split -= (int)gridDim.x;
  const int npos = sd.pos + 1, t0 = split * split_len;
  if (t0 >= npos) return;
  int tend = min(npos, t0 + split_len);
  const bool owns_new = tend == npos;
  if (owns_new) tend--;  // pos itself comes from LDS
  const size_t nq = (size_t)n_heads * HD, nkv = (size_t)nkvh * HD;
  const size_t lbase = (size_t)layer * (size_t)sd.ctx_cap * row + (size_t)kvh * HB;
  const uint8_t *kb = sd.k + lbase, *vb = sd.v + lbase;

  // ---- requests: the setup's inputs, then the first two tiles ----
  const int i4 = tid % GPH;  // four pairs of a head: two float4s, at oa and ob
  const int oa = llama ? 8 * i4 : 4 * i4, ob = llama ? 8 * i4 + 4 : half + 4 * i4;
  const int ngq = G * GPH;
  const uint8_t *qh = (const uint8_t *)(q_in + (size_t)u * nq + (size_t)kvh * G * HD);
  f32x4 xa[QG], xb[QG], c0, c1, qwa, qwb, ka, kb4, kwa, kwb, v4;
#pragma unroll
  for (int g = 0; g < QG; g++) {  // (lanes past the group's heads read its last group)
    const int h = min(tid + kThreads * g, ngq - 1) / GPH;
    xa[g] = gload<f32x4>(qh + 4 * (h * HD + oa));
    xb[g] = gload<f32x4>(qh + 4 * (h * HD + ob));
  }
  const bool rot = rope_on && rope;
  if (rot) {
    const uint8_t *cs = (const uint8_t *)(rope + (size_t)sd.pos * HD);
    c0 = gload<f32x4>(cs + 32 * i4);
    c1 = gload<f32x4>(cs + 32 * i4 + 16);
  }
  const uint8_t *nw = (const uint8_t *)(norm_w + (size_t)layer * 2 * HD);
  if (on & 1) {
    qwa = gload<f32x4>(nw + 4 * oa);
    qwb = gload<f32x4>(nw + 4 * ob);
  }
  if (owns_new && wave == 3) {
    const uint8_t *ki = (const uint8_t *)(k_in + (size_t)u * nkv + (size_t)kvh * HD);
    ka = gload<f32x4>(ki + 4 * oa);
    kb4 = gload<f32x4>(ki + 4 * ob);
    if (on & 2) {
      kwa = gload<f32x4>(nw + 4 * (HD + oa));
      kwb = gload<f32x4>(nw + 4 * (HD + ob));
    }
  }
  if (owns_new && wave == 2)
    v4 = gload<f32x4>((const uint8_t *)(v_in + (size_t)u * nkv + (size_t)kvh * HD) +
                      16 * (lane % DL));

  // V lane: slot of VP positions, dims 4*vd .. 4*vd + 3 (block vd / 8)
  const int slot = lane / DL, vd = lane - slot * DL;
  const uint32_t vblk = (uint32_t)vd >> 3;
  // its quants' window: two bytes before them (even blocks) or four (odd)
  const uint32_t voff =
      FMT ? 34u * vblk + 2u + 4u * (uint32_t)(vd & 7) - ((vblk & 1u) ? 4u : 2u) : 16u * (uint32_t)vd;
  const uint32_t vsel = (vblk & 1u) ? 0x07060504u : 0x05040302u;
  // the scale a lane loads: block quarter (+ 4u), in the dword at its start
  const uint32_t sblk = NB >= 4 ? (uint32_t)quarter : (uint32_t)(quarter & (NB - 1));
  const uint32_t soff = (34u * sblk) & ~3u, sshift = (sblk & 1u) * 16u;

  // the wave's tiles: 16-position tiles wave, wave + 4, ... of the split, then
  // (one wave) the new row
  const int ntile = tend > t0 ? (tend - t0 + kWideTile - 1) / kWideTile : 0;
  const int mine = ntile > wave ? (ntile - wave + kWavesPerSplit - 1) / kWavesPerSplit : 0;
  const int total = mine + (owns_new && wave == (ntile & (kWavesPerSplit - 1)) ? 1 : 0);
  auto tile_at = [&](int i) { return t0 + kWideTile * (wave + kWavesPerSplit * i); };
  // Tile i (positions past its end read its last one and count for nothing).
  auto load = [&](WideRaw<FMT, HD> &r, int i) {
    const int ts = tile_at(i), n = min(kWideTile, tend - ts);
    const uint8_t *kt = kb + (size_t)ts * row, *vt = vb + (size_t)ts * row;
    const uint32_t ko = (uint32_t)min(col, n - 1) * row;
    if constexpr (FMT == 1) {
#pragma unroll
      for (int b = 0; b < NB; b++) {
        const uint8_t *a = kt + (ko + 34u * b + 2u + 8u * quarter - ((b & 1) ? 4u : 2u));
        const u32x2a w = gload<u32x2a>(a);
        r.k[b][0] = w.x;
        r.k[b][1] = w.y;
        r.k[b][2] = gload<uint32_t>(a + 8);
      }
#pragma unroll
      for (int x = 0; x < WideRaw<1, HD>::NS; x++) {
        r.ks[x] = gload<uint32_t>(kt + (ko + soff + 136u * x));
        r.vs[x] = gload<uint32_t>(vt + (ko + soff + 136u * x));
      }
#pragma unroll
      for (int x = 0; x < VP; x++) {
        const u32x2a w = gload<u32x2a>(vt + ((uint32_t)min(VP * slot + x, n - 1) * row + voff));
        r.v[x][0] = w.x;
        r.v[x][1] = w.y;
      }
    } else {
#pragma unroll
      for (int j = 0; j < HD / 16; j++) r.k[j] = gload<f32x4>(kt + (ko + 64u * j + 16u * quarter));
#pragma unroll
      for (int x = 0; x < VP; x++)
        r.v[x] = gload<f32x4>(vt + ((uint32_t)min(VP * slot + x, n - 1) * row + voff));
    }
  };
  WideRaw<FMT, HD> ra, rb;
  if (mine > 0) load(ra, 0);
  if (mine > 1) load(rb, 1);

  // ---- setup: [QK-RMSNorm,] RoPE, digit planes, the owner's new row ----
  uint32_t *const digs = reinterpret_cast<uint32_t *>(lds + ll.q);
  float *const qs = reinterpret_cast<float *>(lds + ll.q);
  uint8_t *const rowk = lds + ll.rows, *const rowv = rowk + ll.row_pad;
  constexpr int DS = dig_stride<32>(), NCH = 4 * SETS * NB;  // (digits of 4 * SETS heads)
  // the pairs of (a, b): four values of x in element order each
  auto rotate = [&](f32x4 &a, f32x4 &b) {
    if (!rot) return;
    float x[4] = {a[0], a[1], a[2], a[3]}, y[4] = {b[0], b[1], b[2], b[3]};
    if (llama) {
      rope_pair(x[0], x[1], c0[0], c0[1]);
      rope_pair(x[2], x[3], c0[2], c0[3]);
      rope_pair(y[0], y[1], c1[0], c1[1]);
      rope_pair(y[2], y[3], c1[2], c1[3]);
    } else {
      rope_pair(x[0], y[0], c0[0], c0[1]);
      rope_pair(x[1], y[1], c0[2], c0[3]);
      rope_pair(x[2], y[2], c1[0], c1[1]);
      rope_pair(x[3], y[3], c1[2], c1[3]);
    }
    a = f32x4{x[0], x[1], x[2], x[3]};
    b = f32x4{y[0], y[1], y[2], y[3]};
  };
#pragma unroll
  for (int g = 0; g < QG; g++) {
    const int gi = tid + kThreads * g, h = gi / GPH;
    f32x4 a = xa[g], b = xb[g];
    if (on & 1) {
      float ss = 0.f;
#pragma unroll
      for (int j = 0; j < 4; j++) ss = fmaf(a[j], a[j], ss);
#pragma unroll
      for (int j = 0; j < 4; j++) ss = fmaf(b[j], b[j], ss);
      ss = group_sum<(GPH < 16 ? GPH : 16)>(ss);
      if constexpr (GPH == 32) ss += lanes_xor<16>(ss);
      const float inv = __fdiv_rn(1.f, sqrtf(__fdiv_rn(ss, (float)HD) + eps));
#pragma unroll
      for (int j = 0; j < 4; j++) {
        a[j] = (qwa[j] * a[j]) * inv;
        b[j] = (qwb[j] * b[j]) * inv;
      }
    }
    rotate(a, b);
#pragma unroll
    for (int j = 0; j < 4; j++) {
      a[j] *= qscale;
      b[j] *= qscale;
    }
    if constexpr (FMT == 0) {
      if (gi < ngq) {
        *reinterpret_cast<f32x4 *>(qs + h * HD + oa) = a;
        *reinterpret_cast<f32x4 *>(qs + h * HD + ob) = b;
      }
    } else {
      // make_digits' digits: a block's largest |q| over its lanes (eight of
      // a, eight of b; LLaMA: four of both)
      float ma = 0.f, mb = 0.f;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        ma = max_abs(ma, a[j]);
        mb = max_abs(mb, b[j]);
      }
      if (llama) ma = mb = max_abs(ma, mb);
      ma = max_abs(ma, dpp_f<0xB1>(ma));
      mb = max_abs(mb, dpp_f<0xB1>(mb));
      ma = max_abs(ma, dpp_f<0x4E>(ma));
      mb = max_abs(mb, dpp_f<0x4E>(mb));
      if (!llama) {
        ma = max_abs(ma, dpp_f<0x141>(ma));
        mb = max_abs(mb, dpp_f<0x141>(mb));
      }
      auto put = [&](const f32x4 &x, float mx, int e) {
        const DigitScale ds = digit_scale(mx);
        uint32_t d[kQPlanes] = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int j = 0; j < 4; j++) {
          int dj[kQPlanes];
          split_digits((int)rintf(x[j] * ds.up), dj);
#pragma unroll
          for (int p = 0; p < kQPlanes; p++) d[p] |= ((uint32_t)dj[p] & 0xffu) << (8 * j);
        }
        const int ch = h * NB + (e >> 5);
        uint32_t *o = digs + ch * DS + ((e & 31) >> 2);
        if (gi < ngq) {
#pragma unroll
          for (int p = 0; p < kQPlanes; p++) o[p * 8] = d[p];
          if ((e & 31) == 0)
            digs[dig_unit_at<32>(NCH, ch)] = __float_as_uint(ds.unit);
        }
      };
      put(a, ma, oa);
      put(b, mb, ob);
    }
  }
  if (owns_new && wave == 3) {  // (lanes past the head's repeat its groups)
    f32x4 a = ka, b = kb4;
    if (on & 2) {
      // the reference's sum: left to right, every product rounded
      f32x4 sa, sq;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        sa[j] = a[j] * a[j];
        sq[j] = b[j] * b[j];
      }
      float ss = 0.f;
      for (int x = 0; x < 2 * GPH; x++) {  // the next four elements: lane t's
        const bool in_a = llama ? (x & 1) == 0 : x < GPH;
        const int t = llama ? x >> 1 : (x < GPH ? x : x - GPH);
#pragma unroll
        for (int j = 0; j < 4; j++) ss = ss + (in_a ? sa[j] : sq[j]);
        ss = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(ss), t));
      }
      const float inv = __fdiv_rn(1.f, sqrtf(__fdiv_rn(ss, (float)HD) + eps));
#pragma unroll
      for (int j = 0; j < 4; j++) {
        a[j] = (kwa[j] * a[j]) * inv;
        b[j] = (kwb[j] * b[j]) * inv;
      }
    }
    rotate(a, b);
    if constexpr (FMT == 0) {
      if (lane < GPH) {
        *reinterpret_cast<f32x4 *>(rowk + 4 * oa) = a;
        *reinterpret_cast<f32x4 *>(rowk + 4 * ob) = b;
      }
    } else {
      const float fa[4] = {a[0], a[1], a[2], a[3]}, fb[4] = {b[0], b[1], b[2], b[3]};
      float ma = 0.f, mb = 0.f;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const float x = fabsf(fa[j]), y = fabsf(fb[j]);
        ma = x > ma ? x : ma;
        mb = y > mb ? y : mb;
      }
      if (llama) {
        ma = mb > ma ? mb : ma;
        ma = mb = lanes_max_gt<4>(ma);
      } else {
        ma = lanes_max_gt<8>(ma);
        mb = lanes_max_gt<8>(mb);
      }
      if (lane < GPH) {
        wide_quant4(fa, ma, oa & 31, rowk + 34 * (oa >> 5));
        wide_quant4(fb, mb, ob & 31, rowk + 34 * (ob >> 5));
      }
    }
  }
  if (owns_new && wave == 2) {
    if constexpr (FMT == 0) {
      if (lane < DL) *reinterpret_cast<f32x4 *>(rowv + 16 * lane) = v4;
    } else {
      const float fv[4] = {v4[0], v4[1], v4[2], v4[3]};
      float mv = 0.f;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const float x = fabsf(fv[j]);
        mv = x > mv ? x : mv;
      }
      mv = lanes_max_gt<8>(mv);
      if (lane < DL) wide_quant4(fv, mv, 4 * (lane & 7), rowv + 34 * (lane >> 3));
    }
  }
  barrier_lds();
  if (owns_new) {  // both new rows to the caches
    const size_t at = (size_t)sd.pos * row;
    for (uint32_t i = tid; i < HB / 2; i += kThreads) {
      const bool is_k = i < HB / 4;
      const uint32_t j = is_k ? i : i - HB / 4;
      reinterpret_cast<uint32_t *>((is_k ? sd.k : sd.v) + lbase + at)[j] =
          reinterpret_cast<const uint32_t *>(is_k ? rowk : rowv)[j];
    }
  }
  auto load_new = [&](WideRaw<FMT, HD> &r) {
    if constexpr (FMT == 1) {
#pragma unroll
      for (int b = 0; b < NB; b++) {
        const uint32_t *w = reinterpret_cast<const uint32_t *>(rowk + 34u * b + 2u + 8u * quarter -
                                                               ((b & 1) ? 4u : 2u));
        r.k[b][0] = w[0];
        r.k[b][1] = w[1];
        r.k[b][2] = w[2];
      }
#pragma unroll
      for (int x = 0; x < WideRaw<1, HD>::NS; x++) {
        r.ks[x] = *reinterpret_cast<const uint32_t *>(rowk + soff + 136u * x);
        r.vs[x] = *reinterpret_cast<const uint32_t *>(rowv + soff + 136u * x);
      }
      const uint32_t *w = reinterpret_cast<const uint32_t *>(rowv + voff);
#pragma unroll
      for (int x = 0; x < VP; x++) {
        r.v[x][0] = w[0];
        r.v[x][1] = w[1];
      }
    } else {
#pragma unroll
      for (int j = 0; j < HD / 16; j++)
        r.k[j] = *reinterpret_cast<const f32x4 *>(rowk + 64u * j + 16u * quarter);
#pragma unroll
      for (int x = 0; x < VP; x++) r.v[x] = *reinterpret_cast<const f32x4 *>(rowv + voff);
    }
  };

  // ---- A operands ----
  uint64_t qa[FMT ? NB : 1][FMT ? SETS : 1];
  float un[FMT ? NB : 1][FMT ? SETS : 1];
  float qf[FMT ? 1 : HD / 4];
  if constexpr (FMT == 1) {
    const int ap = col & 3;
#pragma unroll
    for (int s = 0; s < SETS; s++) {
      const int ah = 4 * s + (col >> 2), ch = 4 * s + quarter;  // A row's head, C lane's head
#pragma unroll
      for (int b = 0; b < NB; b++) {
        uint64_t a = 0;
        if (ah < G) a = *reinterpret_cast<const uint64_t *>(digs + (ah * NB + b) * DS + ap * 8 + 2 * quarter);
        qa[b][s] = a;
        un[b][s] = ch < G ? __uint_as_float(digs[dig_unit_at<32>(NCH, ch * NB + b)]) : 0.f;
      }
    }
  } else {
    const int ah = 4 * (col & 3) + (col >> 2);  // A row 4h + i: head 4i + h
#pragma unroll
    for (int j = 0; j < HD / 16; j++) {
      const f32x4 x = ah < G ? *reinterpret_cast<const f32x4 *>(qs + ah * HD + 16 * j + 4 * quarter)
                             : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 4; i++) qf[4 * j + i] = x[i];
    }
  }

  float m[SETS], l[SETS];
  f32x4 acc[4][SETS];  // acc[j][s][i]: head 4s + i at dim 4*vd + j
#pragma unroll
  for (int s = 0; s < SETS; s++) {
    m[s] = kNegBig;
    l[s] = 0.f;
#pragma unroll
    for (int j = 0; j < 4; j++) acc[j][s] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  float *px = reinterpret_cast<float *>(lds) + wave * wide_px_floats(FMT, HD, SETS);
  float *pfac = px + NBX * PXB;  // [head]

  // the four scales of a position (one dword per quarter) in every lane
  auto spread = [&](const uint32_t(&raw)[FMT ? (NB + 3) / 4 : 1], float(&o)[FMT ? NB : 1]) {
    if constexpr (FMT == 1) {
#pragma unroll
      for (int x = 0; x < (NB + 3) / 4; x++) {
        const uint32_t f16 = __float_as_uint(half_bits_to_f32_hw(raw[x] >> sshift));
        const auto a = __builtin_amdgcn_permlane16_swap(f16, f16, false, false);
        if constexpr (NB == 2) {
          o[0] = __uint_as_float(a[0]);
          o[1] = __uint_as_float(a[1]);
        } else {
          // a[0]: blocks 0, 0, 2, 2 by quarter; a[1]: 1, 1, 3, 3
          const auto e = __builtin_amdgcn_permlane32_swap(a[0], a[0], false, false);
          const auto f = __builtin_amdgcn_permlane32_swap(a[1], a[1], false, false);
          o[4 * x] = __uint_as_float(e[0]);
          o[4 * x + 1] = __uint_as_float(f[0]);
          o[4 * x + 2] = __uint_as_float(e[1]);
          o[4 * x + 3] = __uint_as_float(f[1]);
        }
      }
    }
  };

  // One tile (i < mine), or the new row.
  auto consume = [&](WideRaw<FMT, HD> &cur, int it) {
    const int ts = it < mine ? tile_at(it) : sd.pos;
    const int n = it < mine ? min(kWideTile, tend - ts) : 1;
    // scores: s[set] of head 4*set + quarter at position col
    float s[SETS];
    if constexpr (FMT == 1) {
      float ks[NB];
      spread(cur.ks, ks);
      double sc[SETS];
#pragma unroll
      for (int q = 0; q < SETS; q++) sc[q] = 0.0;
#pragma unroll
      for (int b = 0; b < NB; b++) {
        constexpr uint32_t kSel[2] = {0x05040302u, 0x07060504u};
        const uint64_t bop =
            (uint64_t)__builtin_amdgcn_perm(cur.k[b][1], cur.k[b][0], kSel[b & 1]) |
            ((uint64_t)__builtin_amdgcn_perm(cur.k[b][2], cur.k[b][1], kSel[b & 1]) << 32);
#pragma unroll
        for (int q = 0; q < SETS; q++) {
          const i32x4 c = __builtin_amdgcn_mfma_i32_16x16x32_i8((long)qa[b][q], (long)bop,
                                                                i32x4{0, 0, 0, 0}, 0, 0, 0);
          sc[q] = fma(chunk_value_exact(c[0], c[1], c[2], c[3]), (double)ks[b] * (double)un[b][q],
                      sc[q]);
        }
      }
#pragma unroll
      for (int q = 0; q < SETS; q++) s[q] = (float)sc[q];
    } else {
      // fp32 sums of eight products each, added in pairs: one chain over all
      // dims leaves a larger error (rms against float64 of 16 / 8 heads of
      // 128 at 20-2000 positions: 0.82-0.985 of k_layer's, 1.05-1.09 of it in
      // two chains of 64 or in chains of 16).  Two chains at a time: with four
      // the registers pass two waves per SIMD.
      f32x4 c = {0.f, 0.f, 0.f, 0.f}, g[2][2];
#pragma unroll
      for (int j = 0; j < HD / 16; j++) {
        f32x4 t[2] = {};
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
          for (int x = 0; x < 2; x++)
            t[x] = __builtin_amdgcn_mfma_f32_16x16x4f32(qf[4 * j + 2 * x + i], cur.k[j][2 * x + i],
                                                        t[x], 0, 0, 0);
        g[0][j & 1] = t[0] + t[1];
        if ((j & 1) == 1) g[1][(j >> 1) & 1] = g[0][0] + g[0][1];
        if ((j & 3) == 3) {
          const f32x4 h = g[1][0] + g[1][1];
          c = j == 3 ? h : c + h;
        }
      }
#pragma unroll
      for (int q = 0; q < SETS; q++) s[q] = c[q];
    }
    if (att && col < n) {
#pragma unroll
      for (int q = 0; q < SETS; q++)
        if (4 * q + quarter < G)
          att[((size_t)u * n_heads + (size_t)(kvh * G + 4 * q + quarter)) * (size_t)P.att_stride +
                ts + col] = s[q];
    }
    // online softmax (the 16 lanes of a head share its reference m)
    float mt[SETS];
    bool need = false;
#pragma unroll
    for (int q = 0; q < SETS; q++) {
      if (col >= n || 4 * q + quarter >= G) s[q] = -INFINITY;
      float mx = s[q];
      mx = fmaxf(mx, dpp_f<0xB1>(mx));
      mx = fmaxf(mx, dpp_f<0x4E>(mx));
      mx = fmaxf(mx, dpp_f<0x141>(mx));
      mx = fmaxf(mx, dpp_f<0x140>(mx));
      mt[q] = fmaxf(m[q], mx);
      need |= mx > m[q] + kRescaleSlack;
    }
    const bool rescale = __any(need);
    if (rescale) {
#pragma unroll
      for (int q = 0; q < SETS; q++) {
        const float a = fast_exp2(m[q] - mt[q]);
        l[q] *= a;
        m[q] = mt[q];
        if (col == 0) pfac[4 * q + quarter] = a;
      }
    }
    float vs[NBX];
    if constexpr (FMT == 1) spread(cur.vs, vs);
#pragma unroll
    for (int q = 0; q < SETS; q++) {
      const float p = fast_exp2(s[q] - m[q]);  // 0 for masked lanes
      l[q] += p;
#pragma unroll
      for (int b = 0; b < NBX; b++) {
        float w = p;
        if constexpr (FMT == 1) w = col < n ? p * vs[b] : 0.f;
        px[b * PXB + (4 * q + quarter) * kWidePxHead + col] = w;
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (rescale) {
#pragma unroll
      for (int q = 0; q < SETS; q++) {
        const f32x4 f = *reinterpret_cast<const f32x4 *>(pfac + 4 * q);
#pragma unroll
        for (int j = 0; j < 4; j++) acc[j][q] *= f;
      }
    }
    if constexpr (FMT == 0) {
      if (n < kWideTile) {  // (0 x a row past the end's last row is not always 0)
#pragma unroll
        for (int x = 0; x < VP; x++)
          if (VP * slot + x >= n) cur.v[x] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
    }
    const float *pv = px + (FMT ? vblk : 0) * PXB + (lane & 3) * kWidePxHead + VP * slot;
#pragma unroll
    for (int x = 0; x < VP; x += 4) {
      f32x4 a[SETS];
#pragma unroll
      for (int q = 0; q < SETS; q++)
        a[q] = *reinterpret_cast<const f32x4 *>(pv + 4 * q * kWidePxHead + x);
#pragma unroll
      for (int y = 0; y < 4; y++) {
        float f[4];
        if constexpr (FMT == 1) {
          const uint32_t w = __builtin_amdgcn_perm(cur.v[x + y][1], cur.v[x + y][0], vsel);
#pragma unroll
          for (int j = 0; j < 4; j++) f[j] = i8f(w, j);
        } else {
#pragma unroll
          for (int j = 0; j < 4; j++) f[j] = cur.v[x + y][j];
        }
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
          for (int q = 0; q < SETS; q++)
            acc[j][q] = __builtin_amdgcn_mfma_f32_4x4x1f32(a[q][y], f[j], acc[j][q], 0, 0, 0);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  auto fetch = [&](WideRaw<FMT, HD> &r, int i) {
    if (i < mine)
      load(r, i);
    else if (i < total)
      load_new(r);
  };
  if (mine <= 0) fetch(ra, 0);
  if (mine <= 1) fetch(rb, 1);
  for (int it = 0; it < total; it += 2) {
    consume(ra, it);
    fetch(ra, it + 2);
    if (it + 1 < total) {
      consume(rb, it + 1);
      fetch(rb, it + 3);
    }
  }

  // ---- fold the position slots, then merge the waves in LDS ----
  barrier_lds();  // (the exchanges and the setup's scratch are dead)
  float *mg = reinterpret_cast<float *>(lds) + wave * (4 * SETS) * pstr;
#pragma unroll
  for (int q = 0; q < SETS; q++) {
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        if constexpr (DL <= 32) acc[j][q][i] += lanes_xor<32>(acc[j][q][i]);
        if constexpr (DL <= 16) acc[j][q][i] += lanes_xor<16>(acc[j][q][i]);
      }
    const float ls = group_sum<16>(l[q]);
    if (col == 0) {
      mg[(4 * q + quarter) * pstr] = m[q];
      mg[(4 * q + quarter) * pstr + 1] = ls;
    }
    if (lane < DL) {
#pragma unroll
      for (int i = 0; i < 4; i++)
        *reinterpret_cast<float4 *>(mg + (4 * q + i) * pstr + kPartHead + 4 * vd) =
            make_float4(acc[0][q][i], acc[1][q][i], acc[2][q][i], acc[3][q][i]);
    }
  }
  barrier_lds();
  for (int e = tid; e < G * DL; e += kThreads) {
    const int g = e / DL, d = e - g * DL;
    const float *b = reinterpret_cast<const float *>(lds) + g * pstr;
    constexpr int ws = 4 * SETS * pstr;
    float mw[kWavesPerSplit], M = kNegBig;
#pragma unroll
    for (int w = 0; w < kWavesPerSplit; w++) {
      mw[w] = b[w * ws];
      M = fmaxf(M, mw[w]);
    }
    double L = 0.0, o[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int w = 0; w < kWavesPerSplit; w++) {
      const double f = (double)fast_exp2(mw[w] - M);
      L = fma((double)b[w * ws + 1], f, L);
      const f32x4 x = *reinterpret_cast<const f32x4 *>(b + w * ws + kPartHead + 4 * d);
#pragma unroll
      for (int j = 0; j < 4; j++) o[j] = fma((double)x[j], f, o[j]);
    }
    const size_t head = (size_t)kvh * G + g;
    if (P.direct_out) {
      *reinterpret_cast<float4 *>(P.q_out + (size_t)u * nq + head * HD + 4 * d) =
          make_float4((float)(o[0] / L), (float)(o[1] / L), (float)(o[2] / L), (float)(o[3] / L));
    } else {
      float *pp = P.part + (((size_t)u * n_heads + head) * (size_t)max_splits + (size_t)split) * pstr;
      *reinterpret_cast<float4 *>(pp + kPartHead + 4 * d) =
          make_float4((float)o[0], (float)o[1], (float)o[2], (float)o[3]);
      if (d == 0) *reinterpret_cast<float2 *>(pp) = make_float2(M, (float)L);
    }
  }
}

// The grid: x = the splits of a (KV head, sequence, layer), a multiple of
// eight where there are eight or more, so that every KV head of a split lands
// on the same XCD (the device deals workgroups to its eight XCDs in turn by
// linear id); y = KV head; z = sequence and layer.
template <int FMT, int HD, int SETS>
hipError_t launch_wide_sets(const DecodeParams &p, int n_layers, hipStream_t s) {
  constexpr uint32_t lds = wide_lds<FMT, HD, SETS>().total;
  const unsigned x = p.max_splits < 8 ? (unsigned)p.max_splits : ((unsigned)p.max_splits + 7u) & ~7u;
  const int units = p.n_seq * n_layers;
  for (int z0 = 0; z0 < units; z0 += 65535) {
    const dim3 grid(x, (unsigned)p.sh.n_kv_heads, (unsigned)std::min(65535, units - z0));
    hipLaunchKernelGGL((k_wide<FMT, HD, SETS>), grid, dim3(kThreads), lds, s, p, z0);
    if (const hipError_t e = hipGetLastError(); e != hipSuccess) return e;
  }
  return hipSuccess;
}

template <int FMT, int HD>
hipError_t launch_wide_hd(const DecodeParams &p, int n_layers, hipStream_t s) {
  switch (wide_sets(p.sh.n_heads / p.sh.n_kv_heads)) {
    case 1: return launch_wide_sets<FMT, HD, 1>(p, n_layers, s);
    case 2: return launch_wide_sets<FMT, HD, 2>(p, n_layers, s);
    default: return launch_wide_sets<FMT, HD, 4>(p, n_layers, s);
  }
}

template <int FMT, int HD, int SETS>
int wide_occupancy_sets() {
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_wide<FMT, HD, SETS>, kThreads,
                                                   wide_lds<FMT, HD, SETS>().total) != hipSuccess) {
    (void)hipGetLastError();
    return 1;
  }
  return n > 0 ? n : 1;
}

template <int FMT, int HD>
int wide_occupancy_hd(const ShapeDev &sh) {
  switch (wide_sets(sh.n_heads / sh.n_kv_heads)) {
    case 1: return wide_occupancy_sets<FMT, HD, 1>();
    case 2: return wide_occupancy_sets<FMT, HD, 2>();
    default: return wide_occupancy_sets<FMT, HD, 4>();
  }
}

}  // namespace g2b
