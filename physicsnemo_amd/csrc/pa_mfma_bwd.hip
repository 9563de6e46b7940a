// bf16 MFMA kernels of the backward pass (the shapes of the fused MFMA forward path).  They consume the packed
// slice weights the forward kernels leave behind (w_pack) and natural-layout (B, N, H*32) activations / gradients:
//
//   deslice_natural_kernel        out_x[n, h, :] = sum_s w[n, h, s] tok'[h, s, :]         (input of d W_out = dy^T out_x)
//   backward_tables_kernel        per-(b, h) MFMA operand fragments of tok', d num and W_slice
//   slice_softmax_backward_mfma_kernel  the per-point stage on the stored slice weights, d z out
//   point_backward_kernel         per point: d w = g tok'^T + fx_mid d num^T + d nrm, softmax backward, d T, d W_slice,
//                                 d x_mid = d z W_slice, d fx_mid = w d num                       (formulas: pa_backward.hip)
//
// Register layouts: see pa_mfma_ops.h.  Every product is arranged so that the accumulator tile has lanes <-> points and
// registers <-> slices / channels (the layout of the forward kernel's logits), i.e. the packed slice weights, the
// recomputed logits and d w line up element by element and all per-point reductions over the slices are in-lane sums
// plus one exchange with lane ^ 32.
#include "pa_common.h"
#include "pa_host.h"
#include "pa_mfma_ops.h"

namespace pa {
namespace mfma {

// ------------------------------------------------------------------------------------------------
// deslice_natural_kernel: grid (G, B, head groups), one wave per head of the group; wave h walks the batch's tiles
// g, g + G, ...
//   out_x^T_h (32 d x 32 pts) = tok'^T_h (A: tokp fragments, registers) . w_h (B: w_pack chunks)
// SPLIT: tokp is the float32 tokens (B, H, S, 32), multiplied as bf16 and remainder.
// ------------------------------------------------------------------------------------------------
template <int S, bool SPLIT>
__global__ __launch_bounds__(512) void deslice_natural_kernel(const u32x4 *__restrict__ w_pack,
                                                              const u32x4 *__restrict__ tokp,
                                                              uint16_t *__restrict__ out_x, int64_t N, int tpb, int H) {
  constexpr int NCH = S / 16;
  const int tid = threadIdx.x, lane = tid & 63, i = lane & 31, g = lane >> 5;
  const int h = blockIdx.z * (blockDim.x >> 6) + __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = blockIdx.y;
  u32x4 tp[NCH], tl[SPLIT ? NCH : 1];
#pragma unroll
  for (int cq = 0; cq < NCH; ++cq) {
    const int64_t f = ((int64_t)b * H + h) * NCH + cq;
    if constexpr (SPLIT) token_fragment(reinterpret_cast<const float *>(tokp) + f * 512 + i, g, tp[cq], tl[cq]);
    else tp[cq] = tokp[f * 64 + lane];
  }
  for (int t = blockIdx.x; t < tpb; t += gridDim.x) {
    const int64_t gt = (int64_t)b * tpb + t;
    const u32x4 *wsrc = w_pack + ((gt * H + h) * NCH) * 64 + lane;
    f32x16 ox;
#pragma unroll
    for (int r = 0; r < 16; ++r) ox[r] = 0.f;
#pragma unroll
    for (int cq = 0; cq < NCH; ++cq) {
      const u32x4 w = load_streaming(wsrc + cq * 64);
      ox = mma(tp[cq], w, ox);
      if constexpr (SPLIT) ox = mma(tl[SPLIT ? cq : 0], w, ox);
    }
    const int64_t n = (int64_t)t * 32 + i;
    const bool ok = n < N;
    store_tile_natural(ox, out_x + ((int64_t)b * N + (ok ? n : 0)) * (H * 32) + h * 32, g, ok);
  }
}

__global__ __launch_bounds__(256) void backward_tables_kernel(const float *__restrict__ w_slice,
                                                              const float *__restrict__ pt_w1,
                                                              const float *__restrict__ out_token,
                                                              const float *__restrict__ d_num, u32x4 *__restrict__ tabs,
                                                              int BH, int S, int split) {
  const BwdTablePlan tp = bwd_table_plan(S, pt_w1 != nullptr, split != 0);
  const int64_t total = tp.shared_units + (int64_t)BH * tp.per_head_units;
  for (int64_t u = (int64_t)blockIdx.x * 256 + threadIdx.x; u < total; u += (int64_t)gridDim.x * 256) {
    const int lane = (int)(u & 63), i = lane & 31, g = lane >> 5;
    int64_t f = u >> 6;  // fragment index
    const float *src;    // (S, 32) table, NULL: zeros
    bool natural;        // true: [slice 32st + i][16kk + 8g + j]; false: [16cq + rowmap(j, g)][i]
    int idx;
    bool low = false;    // the remainder of the table
    if (f < tp.nshared) {
      int r = (int)(f % tp.group);
      src = f < tp.group ? w_slice : pt_w1;
      low = r >= tp.st2 + tp.nch;
      if (low) r -= tp.st2 + tp.nch;
      natural = r < tp.st2;
      idx = natural ? r : r - tp.st2;
    } else {
      f -= tp.nshared;
      const int64_t bh = f / tp.nhead;
      int r = (int)(f - bh * tp.nhead);
      low = r >= 2 * tp.st2 + tp.nch;
      if (low) r -= 2 * tp.st2 + tp.nch;
      const float *table = r < tp.st2 ? out_token : d_num;
      src = table ? table + bh * S * 32 : nullptr;
      natural = r < 2 * tp.st2;
      idx = r < tp.st2 ? r : r < 2 * tp.st2 ? r - tp.st2 : r - 2 * tp.st2;
    }
    uint16_t e[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      int s, d;
      if (natural) {
        s = 32 * (idx >> 1) + i;
        d = 16 * (idx & 1) + 8 * g + j;
      } else {
        s = 16 * idx + rowmap(j, g);
        d = i;
      }
      const float x = src && s < S ? src[s * 32 + d] : 0.f;
      e[j] = to_bf16_bits(low ? x - (float)(__bf16)x : x);
    }
    u32x4 v;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = (uint32_t)e[2 * j] | ((uint32_t)e[2 * j + 1] << 16);
    tabs[u] = v;
  }
}

// ------------------------------------------------------------------------------------------------
// slice_softmax_backward_mfma_kernel: grid (G, B), H waves; wave h owns head h; its tok' / d num fragments stay in
// registers (S <= 64) or in LDS (S = 128, where the registers are needed for d w), the W_slice fragments are shared
// through LDS.  Per 32-point tile and head:
//   z^T  (S x pts) = W_slice . x_mid^T + b_slice                       B = x_mid rows, 16-byte natural loads
//   dw^T (S x pts) = tok' . g^T + d num . fx_mid^T + d nrm             B = g / fx_mid rows
//   w: unpacked from w_pack; dot = sum_s w dw / sum_s w; dz = (w / T) (dw - dot); dT -= sum dz z / T
//   d x_mid^T (32 x pts) = W_slice^T . dz^T (B = bf16(dz^T) straight from registers); d fx_mid^T = d num^T . w (B = w_pack)
// The stage by itself, for callers that keep d z (pa_mfma_slice_softmax_backward); training takes point_backward_kernel,
// which sums d W_slice instead of storing d z and reads no weights.
// Rows beyond N have w = 0 in w_pack (the forward writes zeros), so they contribute nothing; their loads are clamped to
// the last valid row and their stores are masked.
// ------------------------------------------------------------------------------------------------
template <int S>
__global__ __launch_bounds__(S > 64 ? 256 : 512) void slice_softmax_backward_mfma_kernel(
    const uint16_t *__restrict__ x_mid, const uint16_t *__restrict__ fx_mid, const uint16_t *__restrict__ d_out_x,
    const u32x4 *__restrict__ w_pack, const u32x4 *__restrict__ tabs, const float *__restrict__ d_norm,
    const float *__restrict__ b_slice, const float *__restrict__ temperature, uint16_t *__restrict__ d_proj,
    uint16_t *__restrict__ d_z, float *__restrict__ dT_part, int64_t N, int tpb, int H) {
  constexpr int ST = (S + 31) / 32, NCH = S / 16, ST2 = 2 * ST;
  constexpr bool LDSTAB = S > 64;  // tok' / d num fragments of d w in LDS instead of registers
  __shared__ u32x4 wsh[(ST2 + NCH) * 64];
  __shared__ float bsl[ST * 32];
  __shared__ float dnl[8 * ST * 32];  // d nrm of every head of this batch (H <= 8)
  extern __shared__ u32x4 tabl[];     // LDSTAB: [H][2 * ST2][64]
  const BwdTablePlan tp = bwd_table_plan(S, false, false);
  const int tid = threadIdx.x, lane = tid & 63, i = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = blockIdx.z * (blockDim.x >> 6) + wave;  // grid.z walks groups of heads (S = 128: 4 waves per workgroup)
  const int b = blockIdx.y;
  const int HD = H * 32;
  const int64_t bh = (int64_t)b * H + h;

  for (int u = tid; u < (ST2 + NCH) * 64; u += blockDim.x) wsh[u] = tabs[u];
  for (int s = tid; s < ST * 32; s += blockDim.x) bsl[s] = s < S ? b_slice[s] : 0.f;
  u32x4 tokA[LDSTAB ? 1 : ST2], dnA[LDSTAB ? 1 : ST2], dnT[NCH];
  {
    const u32x4 *mine = tabs + tp.shared_units + bh * tp.per_head_units + lane;
    if constexpr (LDSTAB) {
      for (int f = 0; f < 2 * ST2; ++f) tabl[(wave * 2 * ST2 + f) * 64 + lane] = mine[f * 64];
    } else {
#pragma unroll
      for (int f = 0; f < ST2; ++f) {
        tokA[f] = mine[f * 64];
        dnA[f] = mine[(ST2 + f) * 64];
      }
    }
#pragma unroll
    for (int cq = 0; cq < NCH; ++cq) dnT[cq] = mine[(2 * ST2 + cq) * 64];
  }
  const u32x4 *mytab = tabl + (wave * 2 * ST2) * 64 + lane;  // LDSTAB: this head's tok' fragments, then its d num fragments
  for (int e = tid; e < H * ST * 32; e += blockDim.x) {
    const int hh = e / (ST * 32), sl = e - hh * ST * 32;
    dnl[e] = sl < S ? d_norm[((int64_t)b * H + hh) * S + sl] : 0.f;
  }
  const float inv_t = 1.f / clamp_temperature(temperature[h]);
  float tsum = 0.f;
  __syncthreads();

  for (int t = blockIdx.x; t < tpb; t += gridDim.x) {
    const int64_t n = (int64_t)t * 32 + i;
    const bool ok = n < N;
    const int64_t row = (int64_t)b * N + (ok ? n : N - 1);
    const int64_t base = row * HD + h * 32 + 8 * g;
    u32x4 xm[2], fm[2], gg[2], wq[NCH];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      xm[kk] = *reinterpret_cast<const u32x4 *>(x_mid + base + 16 * kk);
      fm[kk] = *reinterpret_cast<const u32x4 *>(fx_mid + base + 16 * kk);
      gg[kk] = *reinterpret_cast<const u32x4 *>(d_out_x + base + 16 * kk);
    }
    {
      const u32x4 *wsrc = w_pack + ((((int64_t)b * tpb + t) * H + h) * NCH) * 64 + lane;
#pragma unroll
      for (int cq = 0; cq < NCH; ++cq) wq[cq] = load_streaming(wsrc + cq * 64);
    }
    // w of this lane's (point, slices): chunk cq = 2st + half holds registers 8 half .. 8 half + 7 as bf16
    auto w_of = [&](int st, int r) {
      const int cq = 2 * st + (r >> 3), j = r & 7;
      if (cq >= NCH) return 0.f;
      const uint32_t pair = wq[cq][j >> 1];
      return __uint_as_float((j & 1) ? (pair & 0xffff0000u) : (pair << 16));
    };
    // per point: dot = sum_s w dw;  sum_s dz z = (sum_s w dw z - dot sum_s w z) / T: the logits of a slice tile are
    // consumed as soon as they exist, only d w stays live across the tiles
    f32x16 dw[ST];
    float dot = 0.f, a1 = 0.f, a2 = 0.f, wsum = 0.f;
#pragma unroll
    for (int st = 0; st < ST; ++st) {
      f32x16 z;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        z[r] = bsl[32 * st + rowmap(r, g)];
        dw[st][r] = dnl[(h * ST + st) * 32 + rowmap(r, g)];
      }
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        z = mma(wsh[(st * 2 + kk) * 64 + lane], xm[kk], z);
        if constexpr (LDSTAB) {
          dw[st] = mma(mytab[(st * 2 + kk) * 64], gg[kk], dw[st]);
          dw[st] = mma(mytab[(ST2 + st * 2 + kk) * 64], fm[kk], dw[st]);
        } else {
          dw[st] = mma(tokA[st * 2 + kk], gg[kk], dw[st]);
          dw[st] = mma(dnA[st * 2 + kk], fm[kk], dw[st]);
        }
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float w = w_of(st, r);
        const float wd = w * dw[st][r];
        dot += wd;
        wsum += w;
        a1 = fmaf(wd, z[r], a1);
        a2 = fmaf(w, z[r], a2);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    // the bf16 weights of a point do not sum to one exactly: dividing by their sum keeps sum_s d z = 0, without which
    // the defect times the common offset of the logits leaks into d temperature and d bias
    wsum = half_sum(wsum);
    dot = wsum > 0.f ? half_sum(dot) / wsum : 0.f;
    tsum += (a1 - dot * a2) * inv_t;  // a1, a2 are this lane's halves; the halves add up in the final wave sum
    f32x16(&dz)[ST] = dw;  // d z replaces d w in place
#pragma unroll
    for (int st = 0; st < ST; ++st)
#pragma unroll
      for (int r = 0; r < 16; ++r) dz[st][r] = w_of(st, r) * inv_t * (dw[st][r] - dot);
    __builtin_amdgcn_sched_barrier(0);
    f32x16 dxm, dfm;
#pragma unroll
    for (int r = 0; r < 16; ++r) dxm[r] = dfm[r] = 0.f;
#pragma unroll
    for (int cq = 0; cq < NCH; ++cq) {
      const u32x4 dzp = (cq & 1) ? pack_half<1>(dz[cq >> 1]) : pack_half<0>(dz[cq >> 1]);
      dxm = mma(wsh[(ST2 + cq) * 64 + lane], dzp, dxm);
      dfm = mma(dnT[cq], wq[cq], dfm);
    }
    const int64_t orow = (int64_t)b * N + (ok ? n : 0);
    uint16_t *pr = d_proj + orow * 2 * HD + h * 32;
    store_tile_natural(dxm, pr, g, ok);
    store_tile_natural(dfm, pr + HD, g, ok);
#pragma unroll
    for (int st = 0; st < ST; ++st)
      store_tile_natural(dz[st], d_z + (orow * H + h) * S + 32 * st, g, ok, S - 32 * st >= 32 ? 32 : 16);
  }
  // d T of this (workgroup, head): every lane holds part of the sum over its points and slices
  tsum = wave_sum(tsum);
  if (lane == 0) dT_part[((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * H + h] = -tsum * inv_t;  // heads: disjoint
}

// ------------------------------------------------------------------------------------------------
// point_backward_kernel: everything of the backward pass that happens per point and head.  grid (G, B, head groups), one
// wave per head of the group, 32-point tiles g, g + G, ... of the batch.  Per tile and head:
//   z^T  (S x pts) = W_slice . x_mid^T + b_slice                       B = x_mid rows, 16-byte natural loads
//   dw^T (S x pts) = tok' . g^T + d num . fx_mid^T + d nrm             B = g / fx_mid rows
//   w = softmax_s(z / T), formed again in float32 (its rows sum to one, which sum_s dz = 0 needs; reading the forward's
//       bf16 weights instead costs 2 S bytes per point and head, the recomputation none that shows);
//   dz = (w / T) (dw - sum_s w dw);  dT -= sum dz z / T
//   d x_mid^T (32 x pts) = W_slice^T . dz^T;  d fx_mid^T = d num^T . w         B = bf16 tiles straight from registers
//       (SPLIT: dz, and d a1 below, as bf16 and remainder too: 16 bits on both sides)
//   d W_slice (S x 32) += dz^T . x_mid,  d b_slice += sum dz:  both operands turned around by an exact MFMA product with
//       0/1 selection matrices (lanes <-> slices / channels, k = points), accumulated in registers over the whole kernel:
//       d z itself never reaches memory.
// PLUS (Transolver++; a2 comes from the forward pass, fx_mid is x_mid, d_proj holds the sum of both gradients): the softmax argument is
//   (z + Gumbel noise) / temp,  temp = max(temperature[h] + gelu(a2), 0.01),  a2 = b2 + sum_s w2[s] gelu(a1[s]),
//   a1 = W1 x_mid + b1;  d temp flows back into temperature[h] and through the small MLP (d W1, d b1, d w2, d b2, d x_mid).
// Rows beyond N repeat the batch's last row: their stores write that row's values again, their sums are masked.
// Each workgroup leaves one row of partial parameter gradients (point_grads() floats: d W_slice, d b_slice, d T per head,
// and for PLUS d W1, d b1, d w2, d b2).
// Bound by HBM, (3 + 2) 64 bytes per point and head, and behind it by the vector work of the softmax and its backward:
// 1 048 576 points, 8 heads, S = 64: 0.74 ms = 3.7 TB/s; reading the stored weights and writing d z the same step took 1.29 ms,
// and d W_slice another 0.3 ms behind it.  PLUS is bound by vector issue (1 900 instructions per tile and head, 9 500 cycles of issue
// in 11 000 at two waves per SIMD): 100 003 points 0.148 ms.  With one wave per SIMD, the temperature's hidden layer formed once more
// for a2 and the noise read where it is used it took 0.221 ms; 8 192 points 25 us against 74.
// ------------------------------------------------------------------------------------------------
struct PointArgs {
  const uint16_t *x_mid, *fx_mid, *g;  // (B, N, H*32)
  const uint16_t *uniform;             // PLUS: (B, N, H, S)
  const float *a2;                     // PLUS: [tile][H][32]
  const u32x4 *tabs;
  const float *d_norm, *b_slice, *temperature;
  const float *pt_b1, *pt_w2, *pt_b2;  // PLUS
  uint16_t *d_proj;                    // (B, N, 2*H*32); PLUS: (B, N, H*32)
  float *partials;
  int64_t N;
  int tpb, H;
};

// heads per workgroup.  1, 2: what the split tables of S = 128 leave room for
constexpr int point_waves(int S, bool plus, bool split) { return S > 64 ? (split ? (plus ? 1 : 2) : 4) : plus || (split && S == 64) ? 4 : 8; }

// Waves per head, each with tiles of its own.  PLUS: 2 where the head's sums and one tile's values fit 256 registers (S = 128: the
// sums alone take 256), so that a SIMD holds two waves; they share the head's tables in LDS, which leave no room for eight heads.
// The plain form on float32 tables takes 30.6 us with two and 34.1 with one (2 x 16 384 points, S = 64), but the step around it
// 3 785 us against 3 695: the convolutions behind it then run at a lower clock.
constexpr int point_streams(int S, bool plus) { return S <= 64 && plus ? 2 : 1; }

// S >= 64: the head's tok' / d num fragments stay in (dynamic) LDS, the registers are needed for z, dw and the sums
constexpr int point_table_units(int S, bool split) { return S >= 64 ? (4 * ((S + 31) / 32) + S / 16) * 64 * (split ? 2 : 1) : 0; }

// a2 alone, for callers that do not have it from a forward pass: grid (G, B, H), one wave
template <int S>
__global__ __launch_bounds__(64) void temperature_hidden_kernel(PointArgs a, float *__restrict__ a2_out) {
  constexpr int ST = (S + 31) / 32, GRP = (2 * ST + S / 16) * 2;  // fragments of W1 behind those of W_slice, each with remainders
  const int lane = threadIdx.x, i = lane & 31, g = lane >> 5, b = blockIdx.y, h = blockIdx.z, HD = a.H * 32;
  const u32x4 *w1 = a.tabs + GRP * 64 + lane;
  for (int t = blockIdx.x; t < a.tpb; t += gridDim.x) {
    const int64_t n = (int64_t)t * 32 + i;
    const uint16_t *row = a.x_mid + ((int64_t)b * a.N + (n < a.N ? n : a.N - 1)) * HD + h * 32 + 8 * g;
    const u32x4 x0 = *reinterpret_cast<const u32x4 *>(row), x1 = *reinterpret_cast<const u32x4 *>(row + 16);
    float a2 = 0.f;
    for (int st = 0; st < ST; ++st) {
      f32x16 hd;
#pragma unroll
      for (int r = 0; r < 16; ++r) hd[r] = 32 * st + rowmap(r, g) < S ? a.pt_b1[32 * st + rowmap(r, g)] : 0.f;
#pragma unroll
      for (int lo = 0; lo < 2; ++lo) {
        hd = mma(w1[(lo * (GRP / 2) + st * 2 + 0) * 64], x0, hd);
        hd = mma(w1[(lo * (GRP / 2) + st * 2 + 1) * 64], x1, hd);
      }
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (32 * st + rowmap(r, g) < S) a2 = fmaf(a.pt_w2[32 * st + rowmap(r, g)], gelu_fit(hd[r]), a2);
    }
    a2 = half_sum(a2) + a.pt_b2[0];
    if (g == 0) a2_out[(((int64_t)b * a.tpb + t) * a.H + h) * 32 + i] = a2;
  }
}

// keeps the phases of a tile apart: the scheduler's freedom to fetch operands of a later one costs registers that are not there
#define PHASE __builtin_amdgcn_sched_barrier(0)
template <int S, bool PLUS, bool SPLIT>
__global__ __launch_bounds__((point_waves(S, PLUS, SPLIT) * point_streams(S, PLUS) * 64)) void point_backward_kernel(PointArgs a) {
  constexpr int ST = (S + 31) / 32, NCH = S / 16, ST2 = 2 * ST, GRP = (ST2 + NCH) * (SPLIT ? 2 : 1), NSH = GRP * (PLUS ? 2 : 1);
  constexpr int NTAB = 2 * ST2 + NCH;  // per-head fragments (and as many remainders)
  constexpr int TU = point_table_units(S, SPLIT);
  constexpr bool LDSTAB = TU > 0;
  extern __shared__ u32x4 tabl[];  // LDSTAB: [head][TU]; at the end [wave][ST * 32][33] floats
  constexpr int W = point_waves(S, PLUS, SPLIT), STREAMS = point_streams(S, PLUS);
  constexpr float kLn2 = 0.6931471805599453f;
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  __shared__ u32x4 wsh[NSH * 64];
  __shared__ u32x4 sel[4 * 64];  // 0, 1: k in kperm order; 2, 3: k in natural order
  __shared__ float bsl[ST * 32], dnl[W][ST * 32], b1l[PLUS ? ST * 32 : 1], w2l[PLUS ? ST * 32 : 1];
  __shared__ float red_t[W * STREAMS], red_b2[W * STREAMS], red_w2[PLUS ? W * STREAMS : 1][PLUS ? ST * 32 : 1];
  const BwdTablePlan tp = bwd_table_plan(S, PLUS, SPLIT);
  const int tid = threadIdx.x, lane = tid & 63, i = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), nwaves = blockDim.x >> 6, heads = nwaves / STREAMS;
  const int stream = wave / heads, hw = wave - stream * heads;  // which of the head's waves, head within the workgroup
  const int h = blockIdx.z * heads + hw, b = blockIdx.y, H = a.H, HD = H * 32;
  const int64_t bh = (int64_t)b * H + h, N = a.N;

  for (int u = tid; u < NSH * 64; u += blockDim.x) wsh[u] = a.tabs[u];
  for (int u = tid; u < 4 * 64; u += blockDim.x) {
    const int ui = u & 31, ug = (u >> 5) & 1, f = u >> 6;
    bf16x8 e;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      e[j] = (__bf16)(ui == (f < 2 ? kperm(f & 1, ug, j) : 16 * (f & 1) + 8 * ug + j) ? 1.f : 0.f);
    sel[u] = __builtin_bit_cast(u32x4, e);
  }
  for (int s = tid; s < ST * 32; s += blockDim.x) {
    bsl[s] = s < S ? a.b_slice[s] : -1e30f;  // slices beyond S: weight 0
    if constexpr (PLUS) {
      b1l[s] = s < S ? a.pt_b1[s] : 0.f;
      w2l[s] = s < S ? a.pt_w2[s] : 0.f;
    }
  }
  for (int e = lane; e < ST * 32; e += 64) dnl[hw][e] = e < S ? a.d_norm[bh * S + e] : 0.f;
  u32x4 treg[LDSTAB ? 1 : NTAB * (SPLIT ? 2 : 1)];
  u32x4 *mytab = tabl + hw * TU + lane;
  {
    const u32x4 *mine = a.tabs + tp.shared_units + bh * tp.per_head_units + lane;
#pragma unroll
    for (int f = 0; f < NTAB * (SPLIT ? 2 : 1); ++f) {
      if constexpr (LDSTAB) mytab[f * 64] = mine[f * 64];
      else treg[LDSTAB ? 0 : f] = mine[f * 64];
    }
  }
  // acc += table fragment f (tok', d num, d num turned) . v, and shared fragment f (lo: its remainder) . v
  auto table = [&](int f) { return LDSTAB ? mytab[f * 64] : treg[LDSTAB ? 0 : f]; };
  auto mma_head = [&](int f, u32x4 v, f32x16 acc) {
    acc = mma(table(f), v, acc);
    if constexpr (SPLIT) acc = mma(table(NTAB + f), v, acc);
    return acc;
  };
  auto mma_shared = [&](int group, int f, u32x4 v, f32x16 acc) {  // W_slice (group 0), W1 (1): ST2 straight, NCH turned
    acc = mma(wsh[(group * GRP + f) * 64 + lane], v, acc);
    if constexpr (SPLIT) acc = mma(wsh[(group * GRP + ST2 + NCH + f) * 64 + lane], v, acc);
    return acc;
  };
  // SPLIT: shared fragment f . what bf16 leaves over of eight registers of v, the third term of the product of both
  auto mma_rest = [&](int group, int f, const f32x16 &v, int half, f32x16 acc) {
    if constexpr (SPLIT) acc = mma(wsh[(group * GRP + f) * 64 + lane], half ? pack_half_rest<1>(v) : pack_half_rest<0>(v), acc);
    return acc;
  };
  const float t_raw = a.temperature[h], inv_t = 1.f / clamp_temperature(t_raw);
  const bool odd = lane & 1;
  const bf16x2 ones = {(__bf16)1.f, (__bf16)1.f};
  f32x16 dws[ST], dw1[PLUS ? ST : 1];  // this wave's sums
  float dw2[PLUS ? ST : 1][8];         // d w2: register q of an even lane is slice rowmap(2 q, g), of an odd one rowmap(2 q + 1, g)
  float csum[ST], csum1[PLUS ? ST : 1], tsum = 0.f, b2sum = 0.f;
#pragma unroll
  for (int st = 0; st < ST; ++st) {
    csum[st] = 0.f;
    if constexpr (PLUS) csum1[st] = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      dws[st][r] = 0.f;
      if constexpr (PLUS) dw1[st][r] = dw2[st][r >> 1] = 0.f;
    }
  }
  __syncthreads();

  u32x4 xm[2], fm[PLUS ? 1 : 2], gg[2];  // fetched one tile ahead
  // a tile's first row (wave-uniform) and this lane's row within it, the last one again beyond N
  auto tile_row = [&](int t) { return (int64_t)b * N + (int64_t)t * 32; };
  auto lane_row = [&](int t) {
    const int64_t last = N - 1 - (int64_t)t * 32;
    return min(i, (int)(last < 31 ? last : 31));
  };
  auto load = [&](const uint16_t *src, int t, u32x4(&v)[2]) {
    const char *p = reinterpret_cast<const char *>(src + tile_row(t) * HD + h * 32);
    const unsigned at = (unsigned)(lane_row(t) * HD + 8 * g) * 2u;  // bytes: a scalar base and 32 bits per lane
    v[0] = *reinterpret_cast<const u32x4 *>(p + at);
    v[1] = *reinterpret_cast<const u32x4 *>(p + at + 32u);
  };
  // PLUS: the noise's samples, slices 32 st + rowmap(4 q .. 4 q + 3, g), and a2
  uint2 noise[PLUS ? ST : 1][4];
  float a2_next = 0.f;
  auto load_noise = [&](int t) {
    if constexpr (PLUS) {
      const char *p = reinterpret_cast<const char *>(a.uniform + tile_row(t) * (H * S) + h * S);
      const unsigned at = (unsigned)(lane_row(t) * (H * S) + 4 * g) * 2u;
#pragma unroll
      for (int st = 0; st < ST; ++st)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (S % 32 == 0 || 32 * st + 8 * q + 4 * g < S)
            noise[st][q] = *reinterpret_cast<const uint2 *>(p + at + (unsigned)(64 * st + 16 * q));
      const char *p2 = reinterpret_cast<const char *>(a.a2 + (((int64_t)b * a.tpb + t) * H + h) * 32);
      a2_next = *reinterpret_cast<const float *>(p2 + (unsigned)i * 4u);
    }
  };
  // streams take turns over the grid, so that few tiles meet as many workgroups as there are
  const int t0 = blockIdx.x + stream * gridDim.x, tstep = gridDim.x * STREAMS;
  if (t0 < a.tpb) {
    load(a.x_mid, t0, xm);
    load(a.g, t0, gg);
    if constexpr (!PLUS) load(a.fx_mid, t0, fm);
    load_noise(t0);
  }

  for (int t = t0; t < a.tpb; t += tstep) {
    asm volatile("" ::: "memory");  // the tables are read from LDS where they are used, not kept in registers from here on
    const bool valid = (int64_t)t * 32 + i < N;
    const int tn = t + tstep < a.tpb ? t + tstep : t;

    float it = inv_t, traw = 0.f, a2 = 0.f;  // 1 / temperature of this lane's point
    GeluParts ga2{};
    auto hidden = [&](int st) {              // the first Linear of proj_temperature, slices 32 st ..
      f32x16 hd;
#pragma unroll
      for (int r = 0; r < 16; ++r) hd[r] = b1l[PLUS ? 32 * st + rowmap(r, g) : 0];
      hd = mma_shared(1, st * 2 + 0, xm[0], hd);
      return mma_shared(1, st * 2 + 1, xm[1], hd);
    };
    if constexpr (PLUS) {
      a2 = a2_next;
      ga2 = gelu_parts(a2);
      traw = t_raw + a2 * ga2.phi;
      it = 1.f / (float)(__bf16)fmaxf(traw, 0.01f);  // the forward rounds it to bf16
    }
    f32x16 z[ST], dw[ST];
    float mx = -INFINITY;
#pragma unroll
    for (int st = 0; st < ST; ++st) {
      if constexpr (PLUS) PHASE;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        z[st][r] = bsl[32 * st + rowmap(r, g)];
        dw[st][r] = dnl[hw][32 * st + rowmap(r, g)];
      }
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        z[st] = mma_shared(0, st * 2 + kk, xm[kk], z[st]);
        dw[st] = mma_head(st * 2 + kk, gg[kk], dw[st]);
        dw[st] = mma_head(ST2 + st * 2 + kk, PLUS ? xm[kk] : fm[PLUS ? 0 : kk], dw[st]);
      }
      if constexpr (PLUS) {
        PHASE;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          if (S % 32 == 0 || 32 * st + 8 * q + 4 * g < S) {
            const uint2 v = noise[st][q];
            const float uu[4] = {__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u),
                                 __uint_as_float(v.y << 16), __uint_as_float(v.y & 0xffff0000u)};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const float inner = fmaf(-kLn2, __builtin_amdgcn_logf(uu[j] + 1e-8f), 1e-8f);  // -ln(u + eps) + eps
              z[st][4 * q + j] = fmaf(-kLn2, __builtin_amdgcn_logf(inner), z[st][4 * q + j]);
            }
          }
        }
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, z[st][r]);
    }
    PHASE;
    if constexpr (!PLUS) {
      load(a.g, tn, gg);
      load(a.fx_mid, tn, fm);
    }
    mx = half_max(mx);
    const float sc = kLog2e * it, off = mx * sc;
    float sum = 0.f, dot = 0.f, a1 = 0.f, az = 0.f;
#pragma unroll
    for (int st = 0; st < ST; ++st)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float zz = z[st][r], e = __builtin_amdgcn_exp2f(fmaf(zz, sc, -off)), ed = e * dw[st][r];
        sum += e;
        dot += ed;
        a1 = fmaf(ed, zz, a1);
        az = fmaf(e, zz, az);
        z[st][r] = e;
      }
    const float inv = 1.f / half_sum(sum);
    dot = half_sum(dot) * inv;
    // sum_s dl z of this lane's slices (dl = w (dw - dot)); the halves add up in the sums below
    float dlz = (a1 - dot * az) * inv;
    float d_a2 = 0.f;
    if constexpr (PLUS) {
      dlz = half_sum(dlz);
      const float d_temp = traw >= 0.01f ? -dlz * it * it : 0.f;  // clamp(min): gradient where not clamped
      d_a2 = d_temp * gelu_grad(a2, ga2);  // also in rows beyond N, which write the last row's d x_mid again
      if (g == 0 && valid) {
        tsum += d_temp;
        b2sum += d_a2;
      }
    } else {
      tsum += valid ? dlz : 0.f;
    }
    PHASE;
    const float wi = inv * it;
    u32x4 wq[NCH], dzp[NCH];
#pragma unroll
    for (int cq = 0; cq < NCH; ++cq) wq[cq] = (cq & 1) ? pack_half<1>(z[cq >> 1], inv) : pack_half<0>(z[cq >> 1], inv);
#pragma unroll
    for (int st = 0; st < ST; ++st)
#pragma unroll
      for (int r = 0; r < 16; ++r) dw[st][r] = z[st][r] * wi * (dw[st][r] - dot);
#pragma unroll
    for (int cq = 0; cq < NCH; ++cq) dzp[cq] = (cq & 1) ? pack_half<1>(dw[cq >> 1]) : pack_half<0>(dw[cq >> 1]);
    f32x16 dxm, dfm;
#pragma unroll
    for (int r = 0; r < 16; ++r) dxm[r] = dfm[r] = 0.f;
    PHASE;
#pragma unroll
    for (int cq = 0; cq < NCH; ++cq) {
      dxm = mma_shared(0, ST2 + cq, dzp[cq], dxm);
      dxm = mma_rest(0, ST2 + cq, dw[cq >> 1], cq & 1, dxm);
      if constexpr (PLUS) dxm = mma_head(2 * ST2 + cq, wq[cq], dxm);
      else dfm = mma_head(2 * ST2 + cq, wq[cq], dfm);
    }
    u32x4 xn[2];
    if constexpr (!PLUS) load(a.x_mid, tn, xn);
    PHASE;
    // x_mid with its points as the reduction index
    f32x16 tr;
#pragma unroll
    for (int r = 0; r < 16; ++r) tr[r] = 0.f;
    tr = mma(xm[0], sel[2 * 64 + lane], tr);
    tr = mma(xm[1], sel[3 * 64 + lane], tr);
    const u32x4 xt0 = pack_half<0>(tr), xt1 = pack_half<1>(tr);
    // acc += chunks of the slices 32 st .. (lanes <-> points) turned around . x_mid; cs: their sums over the points
    auto accumulate = [&](u32x4 c0, u32x4 c1, int st, f32x16 &acc, float &cs) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        c0[j] = valid ? c0[j] : 0u;
        c1[j] = valid ? c1[j] : 0u;
      }
      f32x16 tt;
#pragma unroll
      for (int r = 0; r < 16; ++r) tt[r] = 0.f;
      tt = mma(c0, sel[lane], tt);
      if (2 * st + 1 < NCH) tt = mma(c1, sel[64 + lane], tt);
      const u32x4 t0 = pack_half<0>(tt), t1 = pack_half<1>(tt);
      acc = mma(t0, xt0, acc);
      acc = mma(t1, xt1, acc);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t w0 = t0[j], w1 = t1[j];
        cs = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, w0), ones, cs, false);
        cs = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, w1), ones, cs, false);
      }
    };
#pragma unroll
    for (int st = 0; st < ST; ++st) {
      PHASE;
      accumulate(dzp[2 * st], dzp[2 * st + 1 < NCH ? 2 * st + 1 : 0], st, dws[st], csum[st]);
    }
    if constexpr (PLUS) {
      const float d_sum = valid ? d_a2 : 0.f;
#pragma unroll
      for (int st = 0; st < ST; ++st) {  // the hidden values again: 8 matrix instructions against 32 registers held since a2
        PHASE;
        f32x16 hd = hidden(st);
        if (st == ST - 1) {  // the next tile, under the activations: earlier, its registers would have to be spilled
          load(a.x_mid, tn, xm);
          load(a.g, tn, gg);
          load_noise(tn);
          PHASE;
        }
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          float act[2];
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            const float v = hd[2 * q + k];
            const GeluParts p = gelu_parts(v);
            act[k] = d_sum * (v * p.phi);
            hd[2 * q + k] = d_a2 * w2l[32 * st + rowmap(2 * q + k, g)] * gelu_grad(v, p);
          }
          // two lanes share two slices' sums: half the registers
          const float keep = odd ? act[1] : act[0], give = odd ? act[0] : act[1];
          dw2[st][q] += keep + __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(give), 0xB1, 0xf, 0xf, true));
        }
        const u32x4 c0 = pack_half<0>(hd), c1 = pack_half<1>(hd);
        dxm = mma_shared(1, ST2 + 2 * st, c0, dxm);
        dxm = mma_rest(1, ST2 + 2 * st, hd, 0, dxm);
        if (2 * st + 1 < NCH) {
          dxm = mma_shared(1, ST2 + 2 * st + 1, c1, dxm);
          dxm = mma_rest(1, ST2 + 2 * st + 1, hd, 1, dxm);
        }
        accumulate(c0, c1, st, dw1[st], csum1[st]);
      }
    }
    PHASE;
    constexpr int NP = PLUS ? 1 : 2;
    char *pb = reinterpret_cast<char *>(a.d_proj + tile_row(t) * (NP * HD) + h * 32);
    uint16_t *pr = reinterpret_cast<uint16_t *>(pb + (unsigned)(lane_row(t) * (NP * HD)) * 2u);
    store_tile_natural(dxm, pr, g, true);
    if constexpr (!PLUS) store_tile_natural(dfm, pr + HD, g, true);
    if constexpr (!PLUS) xm[0] = xn[0], xm[1] = xn[1];
  }

  // One row of partial gradients per workgroup.  The waves leave their sums side by side in LDS, over the tables, and all threads
  // add them up in the waves' order: the waves in turn, each with the shuffles of d w2, took 40 us behind the last tile (8 192
  // points, S = 64: 74 us, PLUS).
  const int n = point_grads(S, H, PLUS);
  float *dst = a.partials + (((int64_t)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x) * n;
  float *sums = reinterpret_cast<float *>(tabl);
  auto total = [&](const f32x16(&acc)[ST], const float(&cs)[ST], float *out) {  // (S, 32) and behind it (S)
    __syncthreads();
    float *mine = sums + wave * (ST * 32 * 33);
#pragma unroll
    for (int st = 0; st < ST; ++st) {
#pragma unroll
      for (int r = 0; r < 16; ++r) mine[(32 * st + rowmap(r, g)) * 33 + i] = acc[st][r];
      const float c = half_sum(cs[st]);
      if (g == 0) mine[(32 * st + i) * 33 + 32] = c;
    }
    __syncthreads();
    for (int e = tid; e < S * 33; e += blockDim.x) {
      float v = 0.f;
      for (int w = 0; w < nwaves; ++w) v += sums[w * (ST * 32 * 33) + e];
      const int sl = e / 33, c = e - sl * 33;
      out[c < 32 ? sl * 32 + c : S * 32 + sl] = v;
    }
  };
  float ts = wave_sum(tsum), bs = PLUS ? wave_sum(b2sum) : 0.f;
  if constexpr (!PLUS) ts = t_raw >= kTempMin && t_raw <= kTempMax ? -ts * inv_t * inv_t : 0.f;  // clamp's gradient
  if (lane == 0) {
    red_t[wave] = ts;
    red_b2[wave] = bs;
  }
  if constexpr (PLUS) {
#pragma unroll
    for (int st = 0; st < ST; ++st)
#pragma unroll
      for (int q = 0; q < 8; ++q) {  // over the lanes of this half with the same parity
        float v = dw2[st][q];
        auto step = [](float x, auto ctrl) {
          constexpr int c = decltype(ctrl)::value;
          return x + __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(x), c, 0xf, 0xf, true));
        };
        v = step(v, std::integral_constant<int, 0x4E>{});   // quad_perm [2,3,0,1]
        v = step(v, std::integral_constant<int, 0x124>{});  // row_ror:4
        v = step(v, std::integral_constant<int, 0x128>{});  // row_ror:8
        const auto o = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        if (i < 2) red_w2[wave][32 * st + rowmap(2 * q + i, g)] = __uint_as_float(o[0]) + __uint_as_float(o[1]);
      }
  }
  total(dws, csum, dst);
  const int h0 = blockIdx.z * heads;
  for (int e = tid; e < H; e += blockDim.x) {
    float v = 0.f;
    if (e >= h0 && e < h0 + heads)
      for (int q = 0; q < STREAMS; ++q) v += red_t[q * heads + e - h0];
    dst[S * 33 + e] = v;
  }
  if constexpr (PLUS) {
    dst += S * 33 + H;
    total(dw1, csum1, dst);
    for (int s = tid; s < S; s += blockDim.x) {
      float v = 0.f;
      for (int w = 0; w < nwaves; ++w) v += red_w2[w][s];
      dst[S * 33 + s] = v;
    }
    if (tid == 0) {
      float v = 0.f;
      for (int w = 0; w < nwaves; ++w) v += red_b2[w];
      dst[S * 34] = v;
    }
  }
}

// ================================================================================================
// host side
// ================================================================================================
bool backward_supported(const pa_shape &s) { return supported(PA_BF16, s); }

int64_t backward_groups(const pa_shape &s, int num_cu) {
  int64_t g = (2 * (int64_t)num_cu + s.B - 1) / s.B;
  const int64_t tpb = tiles_per_batch(s);
  if (g > tpb) g = tpb;
  return g < 1 ? 1 : g;
}

int64_t backward_tables_bytes(const pa_shape &s) {
  const BwdTablePlan tp = bwd_table_plan((int)s.S, false, false);
  return (tp.shared_units + s.B * s.H * tp.per_head_units) * 16;
}

template <bool SPLIT>
static int deslice_natural_t(const pa_shape &s, const void *w_pack, const void *tokp, void *out_x, int num_cu, hipStream_t st) {
  const int waves = (int)(s.H < 8 ? s.H : 8);
  if (s.H % waves != 0) return PA_ERR_UNSUPPORTED;
  const int groups = (int)(s.H / waves);
  int64_t gx = backward_groups(s, num_cu) / groups;
  if (gx < 1) gx = 1;
  const dim3 grid((unsigned)gx, (unsigned)s.B, (unsigned)groups), block((unsigned)(waves * 64));
  const u32x4 *wp = static_cast<const u32x4 *>(w_pack), *tp = static_cast<const u32x4 *>(tokp);
  uint16_t *ox = static_cast<uint16_t *>(out_x);
  const int tpb = (int)tiles_per_batch(s);
  switch (s.S) {
    case 16: hipLaunchKernelGGL((deslice_natural_kernel<16, SPLIT>), grid, block, 0, st, wp, tp, ox, s.N, tpb, (int)s.H); break;
    case 32: hipLaunchKernelGGL((deslice_natural_kernel<32, SPLIT>), grid, block, 0, st, wp, tp, ox, s.N, tpb, (int)s.H); break;
    case 64: hipLaunchKernelGGL((deslice_natural_kernel<64, SPLIT>), grid, block, 0, st, wp, tp, ox, s.N, tpb, (int)s.H); break;
    case 128: hipLaunchKernelGGL((deslice_natural_kernel<128, SPLIT>), grid, block, 0, st, wp, tp, ox, s.N, tpb, (int)s.H); break;
    default: return PA_ERR_UNSUPPORTED;
  }
  return launch_status();
}

int deslice_natural(const pa_shape &s, const void *w_pack, const void *tokp, void *out_x, int num_cu, hipStream_t st) {
  return deslice_natural_t<false>(s, w_pack, tokp, out_x, num_cu, st);
}

int deslice_tokens(const pa_shape &s, const void *w_pack, const float *tokens, void *out_x, int num_cu, hipStream_t st) {
  return deslice_natural_t<true>(s, w_pack, tokens, out_x, num_cu, st);
}

int slice_softmax_backward(const pa_shape &s, const pa_params &p, const void *x_mid, const void *fx_mid,
                           const void *d_out_x, const void *w_pack, const float *out_token, const float *d_num,
                           const float *d_norm, void *tables, void *d_proj, void *d_z, float *dT_part, int num_cu,
                           hipStream_t st) {
  if (!backward_supported(s)) return PA_ERR_UNSUPPORTED;
  u32x4 *tabs = static_cast<u32x4 *>(tables);
  hipLaunchKernelGGL(backward_tables_kernel, dim3(64), dim3(256), 0, st, p.in_project_slice_weight,
                     (const float *)nullptr, out_token, d_num, tabs, (int)(s.B * s.H), (int)s.S, 0);
  int rc = launch_status();
  if (rc) return rc;
  // S = 128: 4 waves (heads) per workgroup, one wave per SIMD, their tok' / d num fragments in (dynamic) LDS
  const int waves = (int)(s.S > 64 ? 4 : s.H);
  const int groups = (int)(s.H / waves);
  const dim3 grid((unsigned)backward_groups(s, num_cu), (unsigned)s.B, (unsigned)groups), block((unsigned)(waves * 64));
  const int tpb = (int)tiles_per_batch(s);
  const size_t lds = s.S > 64 ? (size_t)waves * 2 * 2 * ((s.S + 31) / 32) * 64 * 16 : 0;
  if ((rc = allow_dynamic_lds(slice_softmax_backward_mfma_kernel<128>, lds))) return rc;
#define PA_LAUNCH_BWD(SS)                                                                                              \
  hipLaunchKernelGGL((slice_softmax_backward_mfma_kernel<SS>), grid, block, lds, st, static_cast<const uint16_t *>(x_mid), \
                     static_cast<const uint16_t *>(fx_mid), static_cast<const uint16_t *>(d_out_x),                     \
                     static_cast<const u32x4 *>(w_pack), tabs, d_norm, p.in_project_slice_bias, p.temperature,          \
                     static_cast<uint16_t *>(d_proj), static_cast<uint16_t *>(d_z), dT_part, s.N, tpb, (int)s.H)
  switch (s.S) {
    case 16: PA_LAUNCH_BWD(16); break;
    case 32: PA_LAUNCH_BWD(32); break;
    case 64: PA_LAUNCH_BWD(64); break;
    case 128: PA_LAUNCH_BWD(128); break;
    default: return PA_ERR_UNSUPPORTED;
  }
#undef PA_LAUNCH_BWD
  return launch_status();
}

// ---- the per-point backward ----
bool point_backward_supported(const pa_shape &s) {
  if (s.D != 32 || s.C != s.H * 32 || (s.C != 128 && s.C != 256 && s.C != 512)) return false;
  if (s.S != 16 && s.S != 32 && s.S != 64 && s.S != 128) return false;
  return tiles_per_batch(s) * s.B <= ((int64_t)1 << 31) / 16 && s.B <= 65535;
}

int64_t point_backward_grads(const pa_shape &s, bool plus) { return point_grads((int)s.S, (int)s.H, plus); }

// Irregular layers of 128 and 256 channels multiply with bf16 tables, all others with float32 ones kept as bf16 and its
// remainder: at 512 channels and 128 slices, 4 096 points, plain bf16 tables leave d b_slice 1.6e-2, d W_slice 1.0e-2 and
// d W_x 6.9e-3 from float64, the split ones 2.7e-3, 2.2e-3 and 2.5e-3 (as fma loops on float32 tables do).
bool float_tables(const pa_shape &s, bool plus) { return plus || s.conv_k > 0 || s.C == 512; }

static int point_head_waves(const pa_shape &s, bool plus) {  // waves (heads) per workgroup
  const int most = point_waves((int)s.S, plus, float_tables(s, plus));
  return (int)(s.H < most ? s.H : most);
}

// workgroups along the points: the chip filled once by the workgroups that fit it (8 waves of 256 registers or 4 of 512 per CU), so that a workgroup's tables and its partial row are paid for once
static int64_t point_groups(const pa_shape &s, bool plus, int num_cu) {
  const int w = point_head_waves(s, plus), most = point_waves((int)s.S, plus, float_tables(s, plus));
  const int64_t resident = (int64_t)num_cu * (most / w), other = s.B * (s.H / w), tpb = tiles_per_batch(s);
  int64_t g = resident / other;
  if (g > tpb) g = tpb;
  return g < 1 ? 1 : g;
}

int64_t point_backward_workspace_bytes(const pa_shape &s, bool plus, int num_cu) {
  const BwdTablePlan tp = bwd_table_plan((int)s.S, plus, float_tables(s, plus));
  const int64_t wgs = point_groups(s, plus, num_cu) * s.B * (s.H / point_head_waves(s, plus));
  return (tp.shared_units + s.B * s.H * tp.per_head_units) * 16 + wgs * point_backward_grads(s, plus) * 4;
}
int64_t temperature_hidden_bytes(const pa_shape &s) { return s.B * tiles_per_batch(s) * s.H * 32 * 4; }

// the operand fragments of W_slice (Transolver++: and W1), out_token (NULL: zeros) and d_num
int backward_tables(const pa_shape &s, const float *w_slice, const float *pt_w1, const float *out_token, const float *d_num,
                    bool split, void *tabs, hipStream_t st) {
  const BwdTablePlan tp = bwd_table_plan((int)s.S, pt_w1 != nullptr, split);
  const int64_t grid = (tp.shared_units + s.B * s.H * tp.per_head_units + 255) / 256;
  hipLaunchKernelGGL(backward_tables_kernel, dim3((unsigned)(grid < 256 ? grid : 256)), dim3(256), 0, st, w_slice, pt_w1,
                     out_token, d_num, static_cast<u32x4 *>(tabs), (int)(s.B * s.H), (int)s.S, split ? 1 : 0);
  return launch_status();
}

// x_mid, fx_mid, d_out_x natural rows (PLUS: fx_mid unused); out_token may be NULL (no deslice term); grads:
// point_backward_grads() floats
int point_backward(const pa_shape &s, const pa_params &p, const pa_plus_params *plus, const void *x_mid,
                   const void *fx_mid, const void *d_out_x, const void *uniform, const float *out_token,
                   const float *d_num, const float *d_norm, void *workspace, void *d_proj, float *grads, int num_cu,
                   hipStream_t st, wgrad::Sums *later, const float *a2) {
  if (!point_backward_supported(s)) return PA_ERR_UNSUPPORTED;
  const bool split = float_tables(s, plus != nullptr);
  const BwdTablePlan tp = bwd_table_plan((int)s.S, plus != nullptr, split);
  u32x4 *tabs = static_cast<u32x4 *>(workspace);
  const int64_t table_units = tp.shared_units + s.B * s.H * tp.per_head_units;
  PointArgs a{};
  a.x_mid = static_cast<const uint16_t *>(x_mid);
  a.fx_mid = static_cast<const uint16_t *>(fx_mid);
  a.g = static_cast<const uint16_t *>(d_out_x);
  a.uniform = static_cast<const uint16_t *>(uniform);
  a.a2 = a2;
  a.tabs = tabs;
  a.d_norm = d_norm, a.b_slice = p.in_project_slice_bias, a.temperature = p.temperature;
  if (plus) a.pt_b1 = plus->proj_temperature_0_bias, a.pt_w2 = plus->proj_temperature_2_weight, a.pt_b2 = plus->proj_temperature_2_bias;
  a.d_proj = static_cast<uint16_t *>(d_proj);
  a.partials = reinterpret_cast<float *>(tabs + table_units);
  a.N = s.N, a.tpb = (int)tiles_per_batch(s), a.H = (int)s.H;
  int rc = backward_tables(s, p.in_project_slice_weight, plus ? plus->proj_temperature_0_weight : nullptr, out_token, d_num, split,
                           tabs, st);
  if (rc) return rc;
  if (plus && !a2) {  // behind the partial gradients
    float *own = a.partials + point_groups(s, true, num_cu) * s.B * (s.H / point_head_waves(s, true)) * point_backward_grads(s, true);
    const int64_t gx = a.tpb < 1024 ? a.tpb : 1024;
    const dim3 grid((unsigned)gx, (unsigned)s.B, (unsigned)s.H);
    switch (s.S) {
      case 16: hipLaunchKernelGGL(temperature_hidden_kernel<16>, grid, dim3(64), 0, st, a, own); break;
      case 32: hipLaunchKernelGGL(temperature_hidden_kernel<32>, grid, dim3(64), 0, st, a, own); break;
      case 64: hipLaunchKernelGGL(temperature_hidden_kernel<64>, grid, dim3(64), 0, st, a, own); break;
      default: hipLaunchKernelGGL(temperature_hidden_kernel<128>, grid, dim3(64), 0, st, a, own); break;
    }
    if ((rc = launch_status())) return rc;
    a.a2 = own;
  }
  const int w = point_head_waves(s, plus != nullptr);
  const int64_t G = point_groups(s, plus != nullptr, num_cu), Z = s.H / w;
  const int streams = point_streams((int)s.S, plus != nullptr);
  const dim3 grid((unsigned)G, (unsigned)s.B, (unsigned)Z), block((unsigned)(w * streams * 64));
#define PA_POINT(SS)                                                                             \
  case SS: {                                                                                     \
    auto kernel = plus    ? point_backward_kernel<SS, true, true>                                \
                  : split ? point_backward_kernel<SS, false, true>                               \
                          : point_backward_kernel<SS, false, false>;                             \
    const size_t tables = (size_t)w * point_table_units(SS, split) * 16;                         \
    const size_t totals = (size_t)w * streams * ((SS + 31) / 32 * 32) * 33 * 4;                  \
    const size_t lds = tables > totals ? tables : totals;                                        \
    if ((rc = allow_dynamic_lds(kernel, lds))) return rc;                                        \
    hipLaunchKernelGGL(kernel, grid, block, lds, st, a);                                         \
  } break
  switch (s.S) {
    PA_POINT(16);
    PA_POINT(32);
    PA_POINT(64);
    PA_POINT(128);
    default: return PA_ERR_UNSUPPORTED;
  }
#undef PA_POINT
  if ((rc = launch_status())) return rc;
  wgrad::Sums own, &sums = later ? *later : own;
  sums.add(a.partials, grads, point_backward_grads(s, plus != nullptr), G * s.B * Z);
  return later ? PA_OK : wgrad::launch_sums(own, st);
}

}  // namespace mfma
}  // namespace pa
