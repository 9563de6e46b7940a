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
// PLUS (Transolver++; fx_mid is x_mid, d_proj holds the sum of both gradients): the softmax argument is
//   (z + Gumbel noise) / temp,  temp = max(temperature[h] + gelu(a2), 0.01),  a2 = b2 + sum_s w2[s] gelu(a1[s]),
//   a1 = W1 x_mid + b1;  d temp flows back into temperature[h] and through the small MLP (d W1, d b1, d w2, d b2, d x_mid).
// Rows beyond N repeat the batch's last row: their stores write that row's values again, their sums are masked.
// Each workgroup leaves one row of partial parameter gradients (point_grads() floats: d W_slice, d b_slice, d T per head,
// and for PLUS d W1, d b1, d w2, d b2).
// Bound by HBM, (3 + 2) 64 bytes per point and head, and behind it by the vector work of the softmax and its backward:
// 1 048 576 points, 8 heads, S = 64: 0.74 ms = 3.7 TB/s; reading the stored weights and writing d z the same step took 1.29 ms,
// and d W_slice another 0.3 ms behind it.  PLUS is bound by its vector work, 27 instructions to a matrix instruction and one
// wave per SIMD: 100 003 points 0.219 ms = 1.2 TB/s, against 1.83 ms of the fma kernel on natural layouts; of these the
// remainder of d z and d a1 takes 0.014 ms, GELU to float32 accuracy 0.010 ms.
// ------------------------------------------------------------------------------------------------
struct PointArgs {
  const uint16_t *x_mid, *fx_mid, *g;  // (B, N, H*32)
  const uint16_t *uniform;             // PLUS: (B, N, H, S)
  const u32x4 *tabs;
  const float *d_norm, *b_slice, *temperature;
  const float *pt_b1, *pt_w2, *pt_b2;  // PLUS
  uint16_t *d_proj;                    // (B, N, 2*H*32); PLUS: (B, N, H*32)
  float *partials;
  int64_t N;
  int tpb, H;
};

// heads (waves) per workgroup.  4: one wave per SIMD, 512 registers; 1, 2: what the split tables of S = 128 leave room for
constexpr int point_waves(int S, bool plus, bool split) { return S > 64 ? (split ? (plus ? 1 : 2) : 4) : plus || (split && S == 64) ? 4 : 8; }

// S >= 64: the head's tok' / d num fragments stay in (dynamic) LDS, the registers are needed for z, dw and the sums
constexpr int point_table_units(int S, bool split) { return S >= 64 ? (4 * ((S + 31) / 32) + S / 16) * 64 * (split ? 2 : 1) : 0; }

template <int S, bool PLUS, bool SPLIT>
__global__ __launch_bounds__((point_waves(S, PLUS, SPLIT) * 64)) void point_backward_kernel(PointArgs a) {
  constexpr int ST = (S + 31) / 32, NCH = S / 16, ST2 = 2 * ST, GRP = (ST2 + NCH) * (SPLIT ? 2 : 1), NSH = GRP * (PLUS ? 2 : 1);
  constexpr int NTAB = 2 * ST2 + NCH;  // per-head fragments (and as many remainders)
  constexpr int TU = point_table_units(S, SPLIT);
  constexpr bool LDSTAB = TU > 0;
  extern __shared__ u32x4 tabl[];  // LDSTAB: [wave][TU]
  constexpr int W = point_waves(S, PLUS, SPLIT);
  constexpr float kLn2 = 0.6931471805599453f;
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  __shared__ u32x4 wsh[NSH * 64];
  __shared__ u32x4 sel[4 * 64];  // 0, 1: k in kperm order; 2, 3: k in natural order
  __shared__ float bsl[ST * 32], dnl[W][ST * 32], b1l[PLUS ? ST * 32 : 1], w2l[PLUS ? ST * 32 : 1];
  __shared__ float red[PLUS ? 2 : 1][ST * 32][33];
  __shared__ float red_t[W];
  __shared__ float red_w2[PLUS ? ST * 32 : 1], red_b2[W];
  const BwdTablePlan tp = bwd_table_plan(S, PLUS, SPLIT);
  const int tid = threadIdx.x, lane = tid & 63, i = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), nwaves = blockDim.x >> 6;
  const int h = blockIdx.z * nwaves + wave, b = blockIdx.y, H = a.H, HD = H * 32;
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
  for (int e = lane; e < ST * 32; e += 64) dnl[wave][e] = e < S ? a.d_norm[bh * S + e] : 0.f;
  u32x4 treg[LDSTAB ? 1 : NTAB * (SPLIT ? 2 : 1)];
  u32x4 *mytab = tabl + wave * TU + lane;
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
  const float b2 = PLUS ? a.pt_b2[0] : 0.f;
  const bf16x2 ones = {(__bf16)1.f, (__bf16)1.f};
  f32x16 dws[ST], dw1[PLUS ? ST : 1], dw2[PLUS ? ST : 1];
  float csum[ST], csum1[PLUS ? ST : 1], tsum = 0.f, b2sum = 0.f;
#pragma unroll
  for (int st = 0; st < ST; ++st) {
    csum[st] = 0.f;
    if constexpr (PLUS) csum1[st] = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      dws[st][r] = 0.f;
      if constexpr (PLUS) dw1[st][r] = dw2[st][r] = 0.f;
    }
  }
  __syncthreads();

  u32x4 xm[2], fm[PLUS ? 1 : 2], gg[2];
  auto row_of = [&](int t) {
    const int64_t n = (int64_t)t * 32 + i;
    return (int64_t)b * N + (n < N ? n : N - 1);
  };
  auto load = [&](int t, u32x4(&x)[2], u32x4(&f)[PLUS ? 1 : 2], u32x4(&q)[2]) {
    const int64_t base = row_of(t) * HD + h * 32 + 8 * g;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      x[kk] = *reinterpret_cast<const u32x4 *>(a.x_mid + base + 16 * kk);
      q[kk] = *reinterpret_cast<const u32x4 *>(a.g + base + 16 * kk);
      if constexpr (!PLUS) f[kk] = *reinterpret_cast<const u32x4 *>(a.fx_mid + base + 16 * kk);
    }
  };
  if ((int)blockIdx.x < a.tpb) load(blockIdx.x, xm, fm, gg);

  for (int t = blockIdx.x; t < a.tpb; t += gridDim.x) {
    asm volatile("" ::: "memory");  // the tables are read from LDS where they are used, not kept in registers from here on
    const bool valid = (int64_t)t * 32 + i < N;
    const int64_t row = row_of(t);
    u32x4 xn[2], fn[PLUS ? 1 : 2], gn[2];
    load(t + (int)gridDim.x < a.tpb ? t + gridDim.x : t, xn, fn, gn);  // the tile after this one

    float it = inv_t, traw = 0.f, a2 = 0.f;  // 1 / temperature of this lane's point
    f32x16 hd[PLUS ? ST : 1];
    if constexpr (PLUS) {
#pragma unroll
      for (int st = 0; st < ST; ++st) {
#pragma unroll
        for (int r = 0; r < 16; ++r) hd[st][r] = b1l[32 * st + rowmap(r, g)];
        hd[st] = mma_shared(1, st * 2 + 0, xm[0], hd[st]);
        hd[st] = mma_shared(1, st * 2 + 1, xm[1], hd[st]);
#pragma unroll
        for (int r = 0; r < 16; ++r) a2 = fmaf(w2l[32 * st + rowmap(r, g)], gelu_fit(hd[st][r]), a2);
      }
      a2 = half_sum(a2) + b2;
      traw = t_raw + gelu_fit(a2);
      it = 1.f / bf16_bits_to_f32(f32_to_bf16_bits(fmaxf(traw, 0.01f)));  // the forward rounds it to bf16
    }
    f32x16 z[ST], dw[ST];
    float mx = -INFINITY;
#pragma unroll
    for (int st = 0; st < ST; ++st) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        z[st][r] = bsl[32 * st + rowmap(r, g)];
        dw[st][r] = dnl[wave][32 * st + rowmap(r, g)];
      }
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        z[st] = mma_shared(0, st * 2 + kk, xm[kk], z[st]);
        dw[st] = mma_head(st * 2 + kk, gg[kk], dw[st]);
        dw[st] = mma_head(ST2 + st * 2 + kk, PLUS ? xm[kk] : fm[PLUS ? 0 : kk], dw[st]);
      }
      if constexpr (PLUS) {
        const uint16_t *urow = a.uniform + row * (H * S) + h * S;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int s0 = 32 * st + 8 * q + 4 * g;  // slices rowmap(4 q .. 4 q + 3, g)
          if (S % 32 == 0 || s0 < S) {
            const uint2 raw = *reinterpret_cast<const uint2 *>(urow + s0);
            const float uu[4] = {__uint_as_float(raw.x << 16), __uint_as_float(raw.x & 0xffff0000u),
                                 __uint_as_float(raw.y << 16), __uint_as_float(raw.y & 0xffff0000u)};
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
      const float d_temp = valid && traw >= 0.01f ? -dlz * it * it : 0.f;  // clamp(min): gradient where not clamped
      d_a2 = d_temp * gelu_erf_grad(a2);
      if (g == 0) {
        tsum += d_temp;
        b2sum += d_a2;
      }
    } else {
      tsum += valid ? dlz : 0.f;
    }
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
#pragma unroll
    for (int cq = 0; cq < NCH; ++cq) {
      dxm = mma_shared(0, ST2 + cq, dzp[cq], dxm);
      dxm = mma_rest(0, ST2 + cq, dw[cq >> 1], cq & 1, dxm);
      if constexpr (PLUS) dxm = mma_head(2 * ST2 + cq, wq[cq], dxm);
      else dfm = mma_head(2 * ST2 + cq, wq[cq], dfm);
    }
    // x_mid with its points as the reduction index
    f32x16 tr;
#pragma unroll
    for (int r = 0; r < 16; ++r) tr[r] = 0.f;
    tr = mma(xm[0], sel[2 * 64 + lane], tr);
    tr = mma(xm[1], sel[3 * 64 + lane], tr);
    const u32x4 xt0 = pack_half<0>(tr), xt1 = pack_half<1>(tr);
    auto accumulate = [&](u32x4(&chunk)[NCH], f32x16(&acc)[ST], float(&cs)[ST]) {
#pragma unroll
      for (int st = 0; st < ST; ++st) {
        f32x16 tt;
#pragma unroll
        for (int r = 0; r < 16; ++r) tt[r] = 0.f;
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          if (2 * st + half >= NCH) continue;
          u32x4 c = chunk[2 * st + half];
#pragma unroll
          for (int j = 0; j < 4; ++j) c[j] = valid ? c[j] : 0u;
          tt = mma(c, sel[half * 64 + lane], tt);
        }
        const u32x4 t0 = pack_half<0>(tt), t1 = pack_half<1>(tt);
        acc[st] = mma(t0, xt0, acc[st]);
        acc[st] = mma(t1, xt1, acc[st]);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const uint32_t w0 = t0[j], w1 = t1[j];
          cs[st] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, w0), ones, cs[st], false);
          cs[st] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, w1), ones, cs[st], false);
        }
      }
    };
    accumulate(dzp, dws, csum);
    if constexpr (PLUS) {
#pragma unroll
      for (int st = 0; st < ST; ++st)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float v = hd[st][r];
          const GeluParts p = gelu_parts(v);
          dw2[st][r] = fmaf(d_a2, v * p.phi, dw2[st][r]);
          hd[st][r] = d_a2 * w2l[32 * st + rowmap(r, g)] * gelu_grad(v, p);
        }
#pragma unroll
      for (int cq = 0; cq < NCH; ++cq) dzp[cq] = (cq & 1) ? pack_half<1>(hd[cq >> 1]) : pack_half<0>(hd[cq >> 1]);
#pragma unroll
      for (int cq = 0; cq < NCH; ++cq) {
        dxm = mma_shared(1, ST2 + cq, dzp[cq], dxm);
        dxm = mma_rest(1, ST2 + cq, hd[cq >> 1], cq & 1, dxm);
      }
      accumulate(dzp, dw1, csum1);
    }
    uint16_t *pr = a.d_proj + row * (PLUS ? HD : 2 * HD) + h * 32;
    store_tile_natural(dxm, pr, g, true);
    if constexpr (!PLUS) store_tile_natural(dfm, pr + HD, g, true);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      xm[kk] = xn[kk];
      gg[kk] = gn[kk];
      if constexpr (!PLUS) fm[kk] = fn[kk];
    }
  }

  // one row of partial gradients per workgroup: the waves (heads) add up in order
  for (int w = 0; w < nwaves; ++w) {
    if (wave == w) {
#pragma unroll
      for (int st = 0; st < ST; ++st) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          float &at = red[0][32 * st + rowmap(r, g)][i];
          at = w == 0 ? dws[st][r] : at + dws[st][r];
          if constexpr (PLUS) {
            float &a1t = red[PLUS ? 1 : 0][32 * st + rowmap(r, g)][i];
            a1t = w == 0 ? dw1[st][r] : a1t + dw1[st][r];
            float v = dw2[st][r];
#pragma unroll
            for (int o = 16; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
            if (i == 0) red_w2[32 * st + rowmap(r, g)] = w == 0 ? v : red_w2[32 * st + rowmap(r, g)] + v;
          }
        }
        const float c = half_sum(csum[st]);
        if (g == 0) red[0][32 * st + i][32] = w == 0 ? c : red[0][32 * st + i][32] + c;
        if constexpr (PLUS) {
          const float c1 = half_sum(csum1[st]);
          if (g == 0) red[PLUS ? 1 : 0][32 * st + i][32] = w == 0 ? c1 : red[PLUS ? 1 : 0][32 * st + i][32] + c1;
        }
      }
      float ts = wave_sum(tsum), bs = PLUS ? wave_sum(b2sum) : 0.f;
      if constexpr (!PLUS) ts = t_raw >= kTempMin && t_raw <= kTempMax ? -ts * inv_t * inv_t : 0.f;  // clamp's gradient
      if (lane == 0) {
        red_t[wave] = ts;
        red_b2[wave] = bs;
      }
    }
    __syncthreads();
  }
  const int n = point_grads(S, H, PLUS);
  float *dst = a.partials + (((int64_t)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x) * n;
  for (int e = tid; e < S * 32; e += blockDim.x) dst[e] = red[0][e >> 5][e & 31];
  for (int s = tid; s < S; s += blockDim.x) dst[S * 32 + s] = red[0][s][32];
  const int h0 = blockIdx.z * nwaves;
  for (int e = tid; e < H; e += blockDim.x) dst[S * 33 + e] = e >= h0 && e < h0 + nwaves ? red_t[e - h0] : 0.f;
  if constexpr (PLUS) {
    dst += S * 33 + H;
    for (int e = tid; e < S * 32; e += blockDim.x) dst[e] = red[PLUS ? 1 : 0][e >> 5][e & 31];
    for (int s = tid; s < S; s += blockDim.x) {
      dst[S * 32 + s] = red[PLUS ? 1 : 0][s][32];
      dst[S * 33 + s] = red_w2[s];
    }
    if (tid == 0) {
      float v = red_b2[0];
      for (int w = 1; w < nwaves; ++w) v += red_b2[w];
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

// workgroups along the points: the chip filled once by the workgroups that fit it (8 waves of 256 or 4 of 512 registers
// per CU), so that a workgroup's tables and its partial row are paid for once
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
                   hipStream_t st, wgrad::Sums *later) {
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
  a.tabs = tabs;
  a.d_norm = d_norm, a.b_slice = p.in_project_slice_bias, a.temperature = p.temperature;
  if (plus) a.pt_b1 = plus->proj_temperature_0_bias, a.pt_w2 = plus->proj_temperature_2_weight, a.pt_b2 = plus->proj_temperature_2_bias;
  a.d_proj = static_cast<uint16_t *>(d_proj);
  a.partials = reinterpret_cast<float *>(tabs + table_units);
  a.N = s.N, a.tpb = (int)tiles_per_batch(s), a.H = (int)s.H;
  int rc = backward_tables(s, p.in_project_slice_weight, plus ? plus->proj_temperature_0_weight : nullptr, out_token, d_num, split,
                           tabs, st);
  if (rc) return rc;
  const int w = point_head_waves(s, plus != nullptr);
  const int64_t G = point_groups(s, plus != nullptr, num_cu), Z = s.H / w;
  const dim3 grid((unsigned)G, (unsigned)s.B, (unsigned)Z), block((unsigned)(w * 64));
#define PA_POINT(SS)                                                                             \
  case SS: {                                                                                     \
    auto kernel = plus    ? point_backward_kernel<SS, true, true>                                \
                  : split ? point_backward_kernel<SS, false, true>                               \
                          : point_backward_kernel<SS, false, false>;                             \
    const size_t lds = (size_t)w * point_table_units(SS, split) * 16;                            \
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
