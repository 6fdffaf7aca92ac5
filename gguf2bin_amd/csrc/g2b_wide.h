// g2b_wide.h - k_wide, the decode kernel for the shapes k_layer and k_tiles
// do not take: wide GQA groups (up to 16 q heads per KV head), more KV heads
// than a wave's lanes hold, rows of any length, head_dim 64, 128 or 256.
// Included only by g2b_wide_inst.hip (one KV format and head_dim at a time).
//
// Replaces the RoPE / append / score / softmax / V loops of l5_model.c:505-577
// in one launch.  A workgroup covers KW KV heads (4, 2 or 1, a divisor of the
// shape's) of one split of positions of one (sequence, layer); each of its
// four waves streams 16-position tiles of one KV head, the 4 / KW waves of a
// KV head taking every (4 / KW)th tile, so that no barrier falls inside the
// stream: a wave loads the next tile into registers while it consumes the
// current one, and the first is in flight during the setup (visit_setup of
// g2b_layer.h over the workgroup's heads).
//
// With G q heads to a KV head the arithmetic is G x 4 flop per K or V element
// - 15 per byte of Q8_0 at G = 8, above what the VALU has per HBM byte - so
// both products run on the matrix cores:
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
// the vector cache serves (default policy).
//
// What bounds it: HBM in large batches, else the chain of dependent steps of
// one tile (load, MFMA, exchange, MFMA) times the tiles of a wave.  Measured
// against the three-pass kernel that these shapes took before (one thread per
// position, every element converted on its own for every q head), per layer:
// 16 / 2 heads of 128, Q8_0, 8 sequences of 1000-4000 positions (11 MB):
// append + decode + combine 786 us, now 17.3 us + a 4.7 us combine.
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

// KV heads per workgroup: the most of 4, 2, 1 that divides the shape's and
// whose q heads the setup holds (4096 floats of rotated q in LDS).
__host__ __device__ inline int wide_kw(const ShapeDev &sh) {
  const int g = sh.n_heads / sh.n_kv_heads;
  for (int kw = 4; kw > 1; kw /= 2)
    if (sh.n_kv_heads % kw == 0 && kw * g * sh.head_dim <= 4096) return kw;
  return 1;
}

__host__ __device__ inline bool wide_shape_ok(const ShapeDev &sh) {
  if (sh.head_dim != 64 && sh.head_dim != 128 && sh.head_dim != 256) return false;
  if (sh.n_kv_heads <= 0 || sh.n_heads % sh.n_kv_heads) return false;
  return sh.n_heads / sh.n_kv_heads <= 16;
}

// Dynamic LDS: the waves' exchanges, then the setup's scratch (k_tiles'
// layout: rotated q, new k, digit planes over the norm sums' transposed copy,
// new v, the new rows, norm factors).  The merge of the waves reuses it all.
struct WideLds {
  uint32_t scr0, kr, dig, vr, rows, row_pad, scr, total;
};
__host__ __device__ inline WideLds wide_lds(const ShapeDev &sh) {
  const int hd = sh.head_dim, g = sh.n_heads / sh.n_kv_heads, kw = wide_kw(sh), nh = kw * g;
  const int sets = wide_sets(g);
  const uint32_t slice = (uint32_t)kw * (sh.kv_q8 ? (uint32_t)hd / 32u * 34u : (uint32_t)hd * 4u);
  const uint32_t kv4 = (uint32_t)(kw * hd) * 4u;
  const uint32_t trb = (uint32_t)(hd * (nh + kw + 1)) * 4u;
  const uint32_t digb = sh.kv_q8 ? (uint32_t)dig_dwords<32>(nh * (hd / 32)) * 4u : 0u;
  WideLds l;
  l.scr0 = ((uint32_t)(kWavesPerSplit * wide_px_floats(sh.kv_q8 ? 1 : 0, hd, sets)) * 4u + 15u) & ~15u;
  // (the transposed copy lies over q, k and the digit planes, which are
  // written only after its sums; the v copy is written before them)
  l.kr = (uint32_t)(nh * hd) * 4u;
  l.dig = l.kr + kv4;
  const uint32_t dig_end = l.dig + digb;
  l.vr = ((dig_end > trb ? dig_end : trb) + 15u) & ~15u;
  l.row_pad = (slice + 15u) & ~15u;
  l.rows = l.vr + kv4;
  l.scr = l.rows + 2u * l.row_pad;
  const uint32_t end = l.scr0 + l.scr + (uint32_t)(((nh + kw + 3) & ~3)) * 4u;
  const uint32_t merge = (uint32_t)(kWavesPerSplit * 4 * sets * (kPartHead + hd)) * 4u;
  l.total = ((end > merge ? end : merge) + 15u) & ~15u;
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

template <int FMT, int HD, int SETS>
__global__ __launch_bounds__(kThreads) void k_wide(DecodeParams P) {
  constexpr int NB = HD / 32, VP = HD / 16, DL = HD / 4;  // DL: V lanes per slot
  constexpr int NBX = wide_px_blocks(FMT, HD), PXB = wide_px_block(SETS);
  constexpr uint32_t HB = FMT ? HD / 32 * 34 : HD * 4;    // a KV head's bytes of a row
  constexpr int pstr = kPartHead + HD;
  extern __shared__ __align__(16) uint8_t lds[];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, col = lane & 15, quarter = lane >> 4;
  const int nkvh = P.sh.n_kv_heads, G = P.sh.n_heads / nkvh;
  const int KW = wide_kw(P.sh), WPH = kWavesPerSplit / KW;
  // grid x: the splits of KV-head group 0, then of group 1, ...
  const int nsx = (int)gridDim.x / (nkvh / KW);
  const int kvg = (int)blockIdx.x / nsx, split = (int)blockIdx.x - kvg * nsx;
  const int li = blockIdx.z, seq = static_seq((int)blockIdx.y, li, P.n_seq);
  const SeqDev sd = P.seqs ? P.seqs[seq] : P.one;
  const int npos = sd.pos + 1;
  const int t0 = split * P.split_len;
  if (t0 >= npos) return;
  int tend = min(npos, t0 + P.split_len);
  const bool owns_new = tend == npos;
  if (owns_new) tend--;  // pos itself comes from LDS
  const int layer = P.layer0 + li;
  const size_t sidx = (size_t)li * (size_t)P.n_seq + (size_t)seq;
  const uint32_t row = P.sh.row_bytes;
  const int kvl = wave / WPH, stripe = wave - kvl * WPH;  // the wave's KV head, its tiles
  const int kvh = kvg * KW + kvl;
  const size_t lbase = (size_t)layer * (size_t)sd.ctx_cap * row + (size_t)kvh * HB;
  const uint8_t *kb = sd.k + lbase, *vb = sd.v + lbase;

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

  WideRaw<FMT, HD> cur, nxt;
  // Rows [ts, ts + n) (n >= 1; positions past n read row n - 1 and count for
  // nothing), or (new_row) the workgroup's new row in LDS.
  auto load = [&](WideRaw<FMT, HD> &r, int ts, int n) {
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
      for (int u = 0; u < WideRaw<1, HD>::NS; u++) {
        r.ks[u] = gload<uint32_t>(kt + (ko + soff + 136u * u));
        r.vs[u] = gload<uint32_t>(vt + (ko + soff + 136u * u));
      }
#pragma unroll
      for (int i = 0; i < VP; i++) {
        const u32x2a w = gload<u32x2a>(vt + ((uint32_t)min(VP * slot + i, n - 1) * row + voff));
        r.v[i][0] = w.x;
        r.v[i][1] = w.y;
      }
    } else {
#pragma unroll
      for (int j = 0; j < HD / 16; j++) r.k[j] = gload<f32x4>(kt + (ko + 64u * j + 16u * quarter));
#pragma unroll
      for (int i = 0; i < VP; i++)
        r.v[i] = gload<f32x4>(vt + ((uint32_t)min(VP * slot + i, n - 1) * row + voff));
    }
  };
  auto load_new = [&](WideRaw<FMT, HD> &r, const uint8_t *krow, const uint8_t *vrow) {
    if constexpr (FMT == 1) {
#pragma unroll
      for (int b = 0; b < NB; b++) {
        const uint32_t *w = reinterpret_cast<const uint32_t *>(krow + 34u * b + 2u + 8u * quarter -
                                                               ((b & 1) ? 4u : 2u));
        r.k[b][0] = w[0];
        r.k[b][1] = w[1];
        r.k[b][2] = w[2];
      }
#pragma unroll
      for (int u = 0; u < WideRaw<1, HD>::NS; u++) {
        r.ks[u] = *reinterpret_cast<const uint32_t *>(krow + soff + 136u * u);
        r.vs[u] = *reinterpret_cast<const uint32_t *>(vrow + soff + 136u * u);
      }
      const uint32_t *w = reinterpret_cast<const uint32_t *>(vrow + voff);
#pragma unroll
      for (int i = 0; i < VP; i++) {
        r.v[i][0] = w[0];
        r.v[i][1] = w[1];
      }
    } else {
#pragma unroll
      for (int j = 0; j < HD / 16; j++)
        r.k[j] = *reinterpret_cast<const f32x4 *>(krow + 64u * j + 16u * quarter);
#pragma unroll
      for (int i = 0; i < VP; i++) r.v[i] = *reinterpret_cast<const f32x4 *>(vrow + voff);
    }
  };

  // the wave's tiles: 16-position tiles stripe, stripe + WPH, ... of the split
  const int ntile = tend > t0 ? (tend - t0 + kWideTile - 1) / kWideTile : 0;
  const int mine = ntile > stripe ? (ntile - stripe + WPH - 1) / WPH : 0;
  const bool own = owns_new && stripe == 0;
  auto tile_at = [&](int i) { return t0 + kWideTile * (stripe + WPH * i); };
  if (mine > 0) load(cur, tile_at(0), min(kWideTile, tend - tile_at(0)));

  // [QK-RMSNorm,] RoPE, digit planes and the owner's append over the
  // workgroup's heads
  const WideLds ll = wide_lds(P.sh);
  uint8_t *const sb = lds + ll.scr0;
  float *qrot = reinterpret_cast<float *>(sb);
  float *kr = reinterpret_cast<float *>(sb + ll.kr), *vr = reinterpret_cast<float *>(sb + ll.vr);
  uint32_t *digs = reinterpret_cast<uint32_t *>(sb + ll.dig);
  uint8_t *rowk = sb + ll.rows, *rowv = rowk + ll.row_pad;
  float *scr = reinterpret_cast<float *>(sb + ll.scr);
  ShapeDev sub = P.sh;
  sub.n_heads = KW * G;
  sub.n_kv_heads = KW;
  const size_t nq = (size_t)P.sh.n_heads * HD, nkv = (size_t)nkvh * HD;
  visit_setup<HD, 32, FMT == 1>(sub, sd, layer, owns_new, P.q_in + sidx * nq + (size_t)kvg * KW * G * HD,
                                P.k_in + sidx * nkv + (size_t)kvg * KW * HD,
                                P.v_in + sidx * nkv + (size_t)kvg * KW * HD, P.rope, P.norm,
                                P.qscale, qrot, kr, vr, rowk, rowv, scr, qrot, digs,
                                (uint32_t)kvg * KW * HB, (uint32_t)KW * HB);

  // A operands
  uint64_t qa[FMT ? NB : 1][FMT ? SETS : 1];
  float un[FMT ? NB : 1][FMT ? SETS : 1];
  float qf[FMT ? 1 : HD / 4];
  if constexpr (FMT == 1) {
    constexpr int DS = dig_stride<32>();
    const int nch = KW * G * NB, ap = col & 3;
#pragma unroll
    for (int s = 0; s < SETS; s++) {
      const int ah = 4 * s + (col >> 2), ch = 4 * s + quarter;  // A row's head, C lane's head
#pragma unroll
      for (int b = 0; b < NB; b++) {
        uint64_t a = 0;
        if (ah < G) {
          const uint32_t *o = digs + ((kvl * G + ah) * NB + b) * DS + ap * 8 + 2 * quarter;
          a = (uint64_t)o[0] | ((uint64_t)o[1] << 32);
        }
        qa[b][s] = a;
        un[b][s] = ch < G ? __uint_as_float(digs[dig_unit_at<32>(nch, (kvl * G + ch) * NB + b)]) : 0.f;
      }
    }
  } else {
    const int ah = 4 * (col & 3) + (col >> 2);  // A row 4h + i: head 4i + h
#pragma unroll
    for (int j = 0; j < HD / 16; j++) {
      const f32x4 x = ah < G ? *reinterpret_cast<const f32x4 *>(qrot + (kvl * G + ah) * HD + 16 * j +
                                                               4 * quarter)
                             : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 4; i++) qf[4 * j + i] = x[i] * P.qscale;
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
      for (int u = 0; u < (NB + 3) / 4; u++) {
        const uint32_t x = __float_as_uint(half_bits_to_f32_hw(raw[u] >> sshift));
        const auto a = __builtin_amdgcn_permlane16_swap(x, x, false, false);
        if constexpr (NB == 2) {
          o[0] = __uint_as_float(a[0]);
          o[1] = __uint_as_float(a[1]);
        } else {
          // a[0]: blocks 0, 0, 2, 2 by quarter; a[1]: 1, 1, 3, 3
          const auto e = __builtin_amdgcn_permlane32_swap(a[0], a[0], false, false);
          const auto f = __builtin_amdgcn_permlane32_swap(a[1], a[1], false, false);
          o[4 * u] = __uint_as_float(e[0]);
          o[4 * u + 1] = __uint_as_float(f[0]);
          o[4 * u + 2] = __uint_as_float(e[1]);
          o[4 * u + 3] = __uint_as_float(f[1]);
        }
      }
    }
  };

  const int total = mine + (own ? 1 : 0);
  const uint8_t *nk = rowk + kvl * HB, *nv = rowv + kvl * HB;
  if (mine == 0 && own) load_new(cur, nk, nv);
  for (int it = 0; it < total; it++) {
    if (it + 1 < mine)
      load(nxt, tile_at(it + 1), min(kWideTile, tend - tile_at(it + 1)));
    else if (it + 1 < total)
      load_new(nxt, nk, nv);
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
      // (two chains: half the dependent steps, and shorter fp32 sums)
      f32x4 c = {0.f, 0.f, 0.f, 0.f}, c1 = c;
#pragma unroll
      for (int j = 0; j < HD / 16; j += 2)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          c = __builtin_amdgcn_mfma_f32_16x16x4f32(qf[4 * j + i], cur.k[j][i], c, 0, 0, 0);
          c1 = __builtin_amdgcn_mfma_f32_16x16x4f32(qf[4 * j + 4 + i], cur.k[j + 1][i], c1, 0, 0, 0);
        }
      c += c1;
#pragma unroll
      for (int q = 0; q < SETS; q++) s[q] = c[q];
    }
    if (P.att && col < n) {
#pragma unroll
      for (int q = 0; q < SETS; q++)
        if (4 * q + quarter < G)
          P.att[(sidx * P.sh.n_heads + (size_t)(kvh * G + 4 * q + quarter)) * (size_t)P.att_stride +
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
        for (int i = 0; i < VP; i++)
          if (VP * slot + i >= n) cur.v[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
    }
    const float *pv = px + (FMT ? vblk : 0) * PXB + (lane & 3) * kWidePxHead + VP * slot;
#pragma unroll
    for (int i = 0; i < VP; i += 4) {
      f32x4 a[SETS];
#pragma unroll
      for (int q = 0; q < SETS; q++)
        a[q] = *reinterpret_cast<const f32x4 *>(pv + 4 * q * kWidePxHead + i);
#pragma unroll
      for (int u = 0; u < 4; u++) {
        float x[4];
        if constexpr (FMT == 1) {
          const uint32_t w = __builtin_amdgcn_perm(cur.v[i + u][1], cur.v[i + u][0], vsel);
#pragma unroll
          for (int j = 0; j < 4; j++) x[j] = i8f(w, j);
        } else {
#pragma unroll
          for (int j = 0; j < 4; j++) x[j] = cur.v[i + u][j];
        }
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
          for (int q = 0; q < SETS; q++)
            acc[j][q] = __builtin_amdgcn_mfma_f32_4x4x1f32(a[q][u], x[j], acc[j][q], 0, 0, 0);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    cur = nxt;
  }

  // Fold the position slots, then merge the WPH waves of each KV head in LDS.
  __syncthreads();  // (the exchanges and the setup's scratch are dead)
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
  __syncthreads();
  for (int e = tid; e < KW * G * DL; e += kThreads) {
    const int h = e / DL, d = e - h * DL, kk = h / G, g = h - kk * G;
    const float *b = reinterpret_cast<const float *>(lds) + (kk * WPH * (4 * SETS) + g) * pstr;
    constexpr int ws = 4 * SETS * pstr;
    float M = b[0];
    for (int w = 1; w < WPH; w++) M = fmaxf(M, b[w * ws]);
    float L = 0.f;
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int w = 0; w < WPH; w++) {
      const float f = fast_exp2(b[w * ws] - M);
      L = fmaf(b[w * ws + 1], f, L);
      const float4 x = *reinterpret_cast<const float4 *>(b + w * ws + kPartHead + 4 * d);
      o.x = fmaf(x.x, f, o.x);
      o.y = fmaf(x.y, f, o.y);
      o.z = fmaf(x.z, f, o.z);
      o.w = fmaf(x.w, f, o.w);
    }
    const size_t head = (size_t)(kvg * KW + kk) * G + g;
    if (P.direct_out) {
      const double Ld = (double)L;
      *reinterpret_cast<float4 *>(P.q_out + sidx * nq + head * HD + 4 * d) =
          make_float4((float)((double)o.x / Ld), (float)((double)o.y / Ld),
                      (float)((double)o.z / Ld), (float)((double)o.w / Ld));
    } else {
      float *pp = P.part + ((sidx * P.sh.n_heads + head) * (size_t)P.max_splits + (size_t)split) * pstr;
      *reinterpret_cast<float4 *>(pp + kPartHead + 4 * d) = o;
      if (d == 0) {
        pp[0] = M;
        pp[1] = L;
      }
    }
  }
}

template <int FMT, int HD>
hipError_t launch_wide_hd(const DecodeParams &p, int n_layers, hipStream_t s) {
  const int sets = wide_sets(p.sh.n_heads / p.sh.n_kv_heads);
  dim3 grid = static_grid(p, n_layers);
  grid.x *= (unsigned)(p.sh.n_kv_heads / wide_kw(p.sh));
  const uint32_t lds = wide_lds(p.sh).total;
  if (sets == 1)
    hipLaunchKernelGGL((k_wide<FMT, HD, 1>), grid, dim3(kThreads), lds, s, p);
  else if (sets == 2)
    hipLaunchKernelGGL((k_wide<FMT, HD, 2>), grid, dim3(kThreads), lds, s, p);
  else
    hipLaunchKernelGGL((k_wide<FMT, HD, 4>), grid, dim3(kThreads), lds, s, p);
  return hipGetLastError();
}

template <int FMT, int HD>
int wide_occupancy_hd(const ShapeDev &sh) {
  const int sets = wide_sets(sh.n_heads / sh.n_kv_heads);
  const uint32_t lds = wide_lds(sh).total;
  int n = 0;
  const hipError_t e =
      sets == 1   ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_wide<FMT, HD, 1>, kThreads, lds)
      : sets == 2 ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_wide<FMT, HD, 2>, kThreads, lds)
                  : hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_wide<FMT, HD, 4>, kThreads, lds);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    return 1;
  }
  return n > 0 ? n : 1;
}

}  // namespace g2b
