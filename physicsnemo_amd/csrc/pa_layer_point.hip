// The per-point stage of an irregular layer's backward pass in bf16, with the products in front of it (formulas and operand
// fragments: pa_mfma_bwd.hip, pa_mfma_ops.h).  This file is compiled with matrix instructions writing ordinary registers
// (-amdgpu-mfma-vgpr-form): its kernel keeps weights in the accumulation registers as operands, and the compiler's other
// form would put the results there too and copy each of them out again (200 copies per tile and wave).
#include "pa_common.h"
#include "pa_host.h"
#include "pa_mfma_ops.h"

namespace pa {
namespace mfma {

// ------------------------------------------------------------------------------------------------
// layer_point_backward_kernel: point_backward_kernel of an irregular layer together with the three products in front of it,
//   x_mid = W_x x + b_x,  fx_mid = W_fx x + b_fx,  g = W_out^T dy,
// so that none of the three (6 C bytes per point written, and read again) reaches memory.  Workgroups of four waves, one
// head each, with the head's 32 rows of the three weights in registers for the whole kernel (3 C / 4 of 512: one wave per
// SIMD).  The 32-point tiles of x and dy pass through LDS, two stages of direct loads; row r's 16-byte unit u lies at
// u ^ (r % 16), which puts what a load instruction reads on all banks.  The products of a tile are formed one tile ahead,
// one matrix instruction behind each value of the softmax of the tile before, and its logits and d w behind that tile's
// stores: with one wave per SIMD nothing else would fill the matrix cores meanwhile.  A lane's rows of the weights are
// taken in the order (bits 2 and 3 of i exchanged) in which the accumulator is an operand with natural channels, what
// point_backward_kernel loads.  At C = 256 two workgroups share a tile's rows; they are neighbours on one XCD, where the
// second finds them in L2 (fetched from memory: 1.08 GB where a million points hold 1.07).
// Bound by its matrix and vector work (2 500 cycles of each per tile and wave; 5 300 pass, at the 1.5 GHz that the card
// keeps up under it): 1 048 576 points, C = 256, S = 64: 0.89 ms, in which 4 C bytes per point are read and 4 C written;
// the products and point_backward_kernel apart took 1.36 ms.  262 144 points in eight
// elements: 207 us against 336, 16 384 in two: 38 us against 57.  With the products behind the softmax instead of within it: 1.05 ms.
// ------------------------------------------------------------------------------------------------
struct LayerPointArgs {
  const uint16_t *x, *dy;           // (B, N, C)
  const uint16_t *w_in, *w_out_t;   // (2 HD, C), (HD, C)
  const float *b_x, *b_fx;          // (HD)
  const u32x4 *tabs;
  const float *d_norm, *b_slice, *temperature;
  uint16_t *d_proj;                 // (B, N, 2 HD)
  float *partials;
  int64_t N;
  int tpb, B, G;                    // tiles and workgroups per batch element
};

constexpr int kLayerPointWaves = 4;
// two stages of x and dy, the tables of four heads
constexpr int layer_point_lds(int C, int S) { return 2 * 2 * 32 * C * 2 + kLayerPointWaves * 4 * ((S + 31) / 32) * 1024; }

template <int C, int S>
__global__ __launch_bounds__(kLayerPointWaves * 64) void layer_point_backward_kernel(LayerPointArgs a) {
  constexpr int H = C / 32, HD = C, Z = H / kLayerPointWaves, KS = C / 16, UPR = C / 8;
  constexpr int ST = (S + 31) / 32, NCH = S / 16, ST2 = 2 * ST, NTAB = 2 * ST2, E = ST * 16;
  constexpr int LOADS = 8 * UPR / 64, RPL = 64 / UPR;  // loads per wave, operand and tile; rows of a load
  constexpr int STAGE = 2 * 32 * UPR;                  // units: x, then dy
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  extern __shared__ u32x4 stages[];
  __shared__ u32x4 wsh[ST2 * 64];
  __shared__ float bsl[ST * 32], dnl[kLayerPointWaves][ST * 32], bias[2][kLayerPointWaves * 32];
  __shared__ float red[ST * 32][33];
  __shared__ float red_t[kLayerPointWaves];
  const BwdTablePlan tp = bwd_table_plan(S, false, false);
  const int tid = threadIdx.x, lane = tid & 63, i = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // workgroup id: (eight of (batch element, g)) x head group x the rest, so that a tile's head groups share an XCD
  const int z = (int)(blockIdx.x >> 3) % Z, at = (int)(blockIdx.x & 7) + 8 * ((int)(blockIdx.x >> 3) / Z);
  if (at >= a.B * a.G) return;
  const int b = at / a.G, first = at - b * a.G;
  const int h = z * kLayerPointWaves + wave;
  const int64_t bh = (int64_t)b * H + h, N = a.N;

  const unsigned lds0 = (unsigned)(uintptr_t)stages + wave * (8 * UPR * 16);
  int row_in[LOADS], unit_at[LOADS];  // this lane's rows of a tile and its bytes within them
#pragma unroll
  for (int k = 0; k < LOADS; ++k) {
    row_in[k] = 8 * wave + RPL * k + lane / UPR;
    unit_at[k] = 16 * ((lane % UPR) ^ (row_in[k] & 15));
  }
  auto fetch = [&](int t, int stage, int k) {  // load k of this wave's eight rows of x and dy; past the last row: that row
    const int last = (int)(N - 1 - (int64_t)t * 32);
    const int64_t base = ((int64_t)b * N + (int64_t)t * 32) * C;
    const int off = (row_in[k] < last ? row_in[k] : last) * (2 * C) + unit_at[k];
    const unsigned dst = lds0 + (unsigned)(stage * STAGE * 16 + k * 1024);
    load_unit_to_lds(a.x + base, off, dst);
    load_unit_to_lds(a.dy + base, off, dst + 32 * UPR * 16);
  };
  auto fetch_all = [&](int t, int stage) {
#pragma unroll
    for (int k = 0; k < LOADS; ++k) fetch(t, stage, k);
  };
  auto after = [&](int t) { return t + a.G < a.tpb ? t + a.G : t; };
  fetch_all(first, 0);

  u32x4 wx[KS], wf[KS], wg[KS];
  {
    const int row = h * 32 + ((i & 0x13) | ((i & 4) << 1) | ((i & 8) >> 1));
    const uint16_t *src = a.w_in + (int64_t)row * C + 8 * g;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      wx[ks] = *reinterpret_cast<const u32x4 *>(src + 16 * ks);
      wf[ks] = *reinterpret_cast<const u32x4 *>(src + (int64_t)HD * C + 16 * ks);
      wg[ks] = *reinterpret_cast<const u32x4 *>(a.w_out_t + (int64_t)row * C + 8 * g + 16 * ks);
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+a"(wx[ks]), "+a"(wf[ks]), "+a"(wg[ks]));
  }
  u32x4 *tab = stages + 2 * STAGE + wave * (NTAB * 64) + lane;  // the head's table fragments
#pragma unroll
  for (int f = 0; f < NTAB; ++f) tab[f * 64] = a.tabs[tp.shared_units + bh * tp.per_head_units + f * 64 + lane];
  for (int u = tid; u < ST2 * 64; u += 256) wsh[u] = a.tabs[u];
  u32x4 w_turned[NCH], dn_turned[NCH];
#pragma unroll
  for (int cq = 0; cq < NCH; ++cq) {
    w_turned[cq] = a.tabs[(ST2 + cq) * 64 + lane];
    dn_turned[cq] = a.tabs[tp.shared_units + bh * tp.per_head_units + (2 * ST2 + cq) * 64 + lane];
    asm volatile("" : "+a"(w_turned[cq]), "+a"(dn_turned[cq]));
  }
  u32x4 sel[4];  // 0, 1: k in kperm order; 2, 3: k in natural order
#pragma unroll
  for (int f = 0; f < 4; ++f) {
    bf16x8 one;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      one[j] = (__bf16)(i == (f < 2 ? kperm(f & 1, g, j) : 16 * (f & 1) + 8 * g + j) ? 1.f : 0.f);
    sel[f] = __builtin_bit_cast(u32x4, one);
    asm volatile("" : "+a"(sel[f]));
  }
  for (int s = tid; s < ST * 32; s += 256) bsl[s] = s < S ? a.b_slice[s] : -1e30f;  // slices beyond S: weight 0
  for (int e = lane; e < ST * 32; e += 64) dnl[wave][e] = e < S ? a.d_norm[bh * S + e] : 0.f;
  if (tid < kLayerPointWaves * 32) {
    bias[0][tid] = a.b_x[z * kLayerPointWaves * 32 + tid];
    bias[1][tid] = a.b_fx[z * kLayerPointWaves * 32 + tid];
  }
  const float inv_t = 1.f / clamp_temperature(a.temperature[h]);
  const bf16x2 ones = {(__bf16)1.f, (__bf16)1.f};
  f32x16 dws[ST];
  float csum[ST], tsum = 0.f;
#pragma unroll
  for (int st = 0; st < ST; ++st) {
    csum[st] = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) dws[st][r] = 0.f;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  // the three products of the tile in `stage`, k-step by k-step
  f32x16 px, pf, pg;
  u32x4 xr[3], yr[3];
  const u32x4 *xs = stages;
  const int sw = i & 15;
  auto read = [&](auto ks_) {
    constexpr int ks = decltype(ks_)::value;
    if constexpr (ks < KS) {
      const u32x4 *p = xs + i * UPR + ((2 * ks + g) ^ sw);
      xr[ks % 3] = p[0];
      yr[ks % 3] = p[32 * UPR];
    }
  };
  // Matrix instructions that stay where they are written: the empty statement takes their result, without which they sink
  // behind all of the softmax.  The distances that vector instructions need to them are the compiler's.
  auto multiply = [](const u32x4 &w, const u32x4 &v, const f32x16 &onto, f32x16 &acc) {
    acc = mma(w, v, onto);
    asm volatile("" : "+v"(acc));
  };
  auto begin = [&](int stage) {
    xs = stages + stage * STAGE;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int d = wave * 32 + 16 * (r >> 3) + 8 * g + (r & 7);
      px[r] = bias[0][d], pf[r] = bias[1][d];
    }
    static_for<2>(read);
  };
  auto product = [&](auto m_) {  // the tile's matrix instruction m
    constexpr int ks = decltype(m_)::value / 3, which = decltype(m_)::value % 3;
    if constexpr (which == 0) {
      read(std::integral_constant<int, ks + 2>{});
      multiply(wx[ks], xr[ks % 3], px, px);
    } else if constexpr (which == 1) {
      multiply(wf[ks], xr[ks % 3], pf, pf);
    } else {
      multiply(wg[ks], yr[ks % 3], ks == 0 ? f32x16{} : pg, pg);
    }
  };
  // behind piece `done` of E: its share of the products `from` to `to`
  auto products = [&](auto done_, auto from_, auto to_) {
    constexpr int done = decltype(done_)::value, from = decltype(from_)::value, n = decltype(to_)::value - from,
                  lo = from + done * n / E, hi = from + (done + 1) * n / E;
    static_for<hi - lo>([&](auto k) { product(std::integral_constant<int, lo + decltype(k)::value>{}); });
    __builtin_amdgcn_sched_barrier(0);
  };
  auto between = [&](auto m) {
    __builtin_amdgcn_sched_barrier(0);
    product(m);
    __builtin_amdgcn_sched_barrier(0);
  };
  u32x4 xm[2], fm[2], gg[2];
  auto finish = [&] {
    xm[0] = pack_half<0>(px), xm[1] = pack_half<1>(px);
    fm[0] = pack_half<0>(pf), fm[1] = pack_half<1>(pf);
    gg[0] = pack_half<0>(pg), gg[1] = pack_half<1>(pg);
  };
  fetch_all(after(first), 1);
  begin(0);
  static_for<3 * KS>(product);
  finish();

  // logits (first, the next thing needed) and d w of the tile whose x_mid, fx_mid and g are at hand, on top of their biases
  f32x16 e[ST], dw[ST];
  auto biases = [&](auto cq_) {  // registers of chunk cq
    constexpr int st = decltype(cq_)::value / 2, half = decltype(cq_)::value % 2;
#pragma unroll
    for (int r = 8 * half; r < 8 * half + 8; ++r) {
      e[st][r] = bsl[32 * st + rowmap(r, g)];
      dw[st][r] = dnl[wave][32 * st + rowmap(r, g)];
    }
  };
  auto score = [&] {
#pragma unroll
    for (int st = 0; st < ST; ++st)
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) e[st] = mma(wsh[(st * 2 + kk) * 64 + lane], xm[kk], e[st]);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int st = 0; st < ST; ++st) {
        dw[st] = mma(tab[(st * 2 + kk) * 64], gg[kk], dw[st]);
        dw[st] = mma(tab[(ST2 + st * 2 + kk) * 64], fm[kk], dw[st]);
      }
  };
  static_for<2 * ST>(biases);
  score();

  constexpr std::integral_constant<int, 0> zero{};
  constexpr std::integral_constant<int, KS * 9 / 4> middle{};
  constexpr std::integral_constant<int, KS * 9 / 4 + 3> later{};
  constexpr std::integral_constant<int, KS * 3> end{};
  int stage = 0;
  for (int t = first; t < a.tpb; t += a.G, stage ^= 1) {
    // the next tile has landed (its loads are older than the four stores of the tile before this one), and every wave is
    // past this tile's stage
    if (t == first) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
    __syncthreads();
    const int t2 = after(after(t));
    begin(stage ^ 1);
    const int valid = (int)(N - (int64_t)t * 32 < 32 ? N - (int64_t)t * 32 : 32);  // points of this tile
    // x_mid with its points as the reduction index
    f32x16 tr;
#pragma unroll
    for (int r = 0; r < 16; ++r) tr[r] = 0.f;
    tr = mma(xm[0], sel[2], tr);
    tr = mma(xm[1], sel[3], tr);
    float mx = -INFINITY;
#pragma unroll
    for (int st = 0; st < ST; ++st)
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, e[st][r]);
    mx = half_max(mx);
    u32x4 xt0, xt1;
    const float sc = kLog2e * inv_t, off = mx * sc;
    float sum = 0.f, dot = 0.f, a1 = 0.f, az = 0.f, next = __builtin_amdgcn_exp2f(fmaf(e[0][0], sc, -off));
    static_for<E>([&](auto k_) {  // the exponential one element ahead
      constexpr int k = decltype(k_)::value, k1 = k + 1 < E ? k + 1 : k;
      const float zz = e[k / 16][k % 16], v = next, ed = v * dw[k / 16][k % 16];
      if constexpr (k + 1 < E) next = __builtin_amdgcn_exp2f(fmaf(e[k1 / 16][k1 % 16], sc, -off));
      sum += v;
      dot += ed;
      a1 = fmaf(ed, zz, a1);
      az = fmaf(v, zz, az);
      e[k / 16][k % 16] = v;
      if constexpr (k % 4 == 1 && k / 4 < LOADS) fetch(t2, stage, k / 4);
      if constexpr (k == 3) xt0 = pack_half<0>(tr), xt1 = pack_half<1>(tr);
      products(k_, zero, middle);
    });
    sum = half_sum(sum);
    between(std::integral_constant<int, middle>{});
    const float inv = 1.f / sum;
    between(std::integral_constant<int, middle + 1>{});
    dot = half_sum(dot) * inv;
    between(std::integral_constant<int, middle + 2>{});
    const float dlz = (a1 - dot * az) * inv;  // of this lane's slices; the halves add up in the last sum
    tsum += i < valid ? dlz : 0.f;
    // dz = w (dw - dot) / T; points beyond N leave none, so that the sums below do not count them
    const float it = i < valid ? inv_t : 0.f, shift = -dot * it;
    // d x_mid and d fx_mid chunk by chunk of 16 slices; dz with its points as the reduction index, d W_slice
    f32x16 dxm, dfm, tt;
#pragma unroll
    for (int r = 0; r < 16; ++r) dxm[r] = dfm[r] = tt[r] = 0.f;
    auto sum_slices = [&](auto st_) {
      constexpr int st = decltype(st_)::value;
      const u32x4 t0 = pack_half<0>(tt), t1 = pack_half<1>(tt);
      dws[st] = mma(t0, xt0, dws[st]);
      dws[st] = mma(t1, xt1, dws[st]);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t w0 = t0[j], w1 = t1[j];
        csum[st] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, w0), ones, csum[st], false);
        csum[st] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, w1), ones, csum[st], false);
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) tt[r] = 0.f;
    };
    static_for<E>([&](auto k_) {
      constexpr int k = decltype(k_)::value, st = k / 16, half = k / 8 % 2, cq = k / 8;
      e[st][k % 16] *= inv;
      dw[st][k % 16] = e[st][k % 16] * fmaf(dw[st][k % 16], it, shift);
      if constexpr (k % 8 == 7 && cq < NCH) {
        const u32x4 wq = pack_half<half>(e[st]), dz = pack_half<half>(dw[st]);
        dxm = mma(w_turned[cq], dz, dxm);
        dfm = mma(dn_turned[cq], wq, dfm);
        tt = mma(dz, sel[half], tt);
      }
      if constexpr (k % 8 == 7) biases(std::integral_constant<int, cq>{});
      if constexpr (k % 16 == 5 && st > 0) sum_slices(std::integral_constant<int, st - 1>{});
      products(k_, later, end);
    });
    sum_slices(std::integral_constant<int, ST - 1>{});
    finish();
    score();
    // buffer stores drop the rows past the tile's last
    const auto rows = __builtin_amdgcn_make_buffer_rsrc(a.d_proj + ((int64_t)b * N + (int64_t)t * 32) * (2 * HD), 0,
                                                        valid * (4 * HD), 0x00027000);
    const int out = i * (4 * HD) + h * 64 + 32 * g;
    u32x4 s0, s1;
    tile_natural(dxm, s0, s1);
    __builtin_amdgcn_raw_buffer_store_b128(s0, rows, out, 0, 0);
    __builtin_amdgcn_raw_buffer_store_b128(s1, rows, out + 16, 0, 0);
    tile_natural(dfm, s0, s1);
    __builtin_amdgcn_raw_buffer_store_b128(s0, rows, out + 2 * HD, 0, 0);
    __builtin_amdgcn_raw_buffer_store_b128(s1, rows, out + 2 * HD + 16, 0, 0);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing may still be landing in LDS when the workgroup ends
  const float t_raw = a.temperature[h];  // read again: no register is left to keep it over the loop

  // one row of partial gradients per workgroup: the waves (heads) add up in order
  for (int w = 0; w < kLayerPointWaves; ++w) {
    if (wave == w) {
#pragma unroll
      for (int st = 0; st < ST; ++st) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          float &to = red[32 * st + rowmap(r, g)][i];
          to = w == 0 ? dws[st][r] : to + dws[st][r];
        }
        const float c = half_sum(csum[st]);
        if (g == 0) red[32 * st + i][32] = w == 0 ? c : red[32 * st + i][32] + c;
      }
      float ts = wave_sum(tsum);
      ts = t_raw >= kTempMin && t_raw <= kTempMax ? -ts * inv_t * inv_t : 0.f;  // clamp's gradient
      if (lane == 0) red_t[wave] = ts;
    }
    __syncthreads();
  }
  float *dst = a.partials + (int64_t)(z * a.B * a.G + at) * point_grads(S, H, false);
  for (int k = tid; k < S * 32; k += 256) dst[k] = red[k >> 5][k & 31];
  for (int s = tid; s < S; s += 256) dst[S * 32 + s] = red[s][32];
  const int h0 = z * kLayerPointWaves;
  for (int k = tid; k < H; k += 256) dst[S * 33 + k] = k >= h0 && k < h0 + kLayerPointWaves ? red_t[k - h0] : 0.f;
}

// 128 slices need the registers that hold the weights here
bool layer_point_backward_supported(const pa_shape &s) { return supported(PA_BF16, s) && s.S <= 64; }

static int64_t layer_point_groups(const pa_shape &s, int num_cu) {  // per batch element: one workgroup per CU
  int64_t g = num_cu / (s.B * (s.H / kLayerPointWaves));
  const int64_t tpb = tiles_per_batch(s);
  if (g > tpb) g = tpb;
  return g < 1 ? 1 : g;
}

int64_t layer_point_backward_workspace_bytes(const pa_shape &s, int num_cu) {
  const BwdTablePlan tp = bwd_table_plan((int)s.S, false, false);
  const int64_t rows = layer_point_groups(s, num_cu) * s.B * (s.H / kLayerPointWaves);
  return (tp.shared_units + s.B * s.H * tp.per_head_units) * 16 + rows * point_grads((int)s.S, (int)s.H, false) * 4;
}

int layer_point_backward(const pa_shape &s, const pa_params &p, const void *w_out_t, const void *x, const void *dy,
                         const float *out_token, const float *d_num, const float *d_norm, void *workspace, void *d_proj,
                         wgrad::Sums &later, float *grads, int num_cu, hipStream_t st) {
  if (!layer_point_backward_supported(s)) return PA_ERR_UNSUPPORTED;
  const BwdTablePlan tp = bwd_table_plan((int)s.S, false, false);
  u32x4 *tabs = static_cast<u32x4 *>(workspace);
  const int64_t table_units = tp.shared_units + s.B * s.H * tp.per_head_units;
  int rc = backward_tables(s, p.in_project_slice_weight, nullptr, out_token, d_num, false, tabs, st);
  if (rc) return rc;
  LayerPointArgs a{};
  a.x = static_cast<const uint16_t *>(x), a.dy = static_cast<const uint16_t *>(dy);
  a.w_in = static_cast<const uint16_t *>(p.in_project_x_weight), a.w_out_t = static_cast<const uint16_t *>(w_out_t);
  a.b_x = p.in_project_x_bias, a.b_fx = p.in_project_fx_bias;
  a.tabs = tabs, a.d_norm = d_norm, a.b_slice = p.in_project_slice_bias, a.temperature = p.temperature;
  a.d_proj = static_cast<uint16_t *>(d_proj);
  a.partials = reinterpret_cast<float *>(tabs + table_units);
  const int64_t G = layer_point_groups(s, num_cu), Z = s.H / kLayerPointWaves;
  a.N = s.N, a.tpb = (int)tiles_per_batch(s), a.B = (int)s.B, a.G = (int)G;
  const size_t lds = (size_t)layer_point_lds((int)s.C, (int)s.S);
#define PA_LAYER_POINT(CC, SS)                                                                            \
  if (s.C == CC && s.S == SS) {                                                                           \
    if ((rc = allow_dynamic_lds(layer_point_backward_kernel<CC, SS>, lds))) return rc;                    \
    hipLaunchKernelGGL((layer_point_backward_kernel<CC, SS>), dim3((unsigned)((G * s.B + 7) / 8 * 8 * Z)), \
                       dim3(kLayerPointWaves * 64), lds, st, a);                                          \
  }
  PA_LAYER_POINT(128, 16)
  PA_LAYER_POINT(128, 32)
  PA_LAYER_POINT(128, 64)
  PA_LAYER_POINT(256, 16)
  PA_LAYER_POINT(256, 32)
  PA_LAYER_POINT(256, 64)
#undef PA_LAYER_POINT
  if ((rc = launch_status())) return rc;
  later.add(a.partials, grads, point_grads((int)s.S, (int)s.H, false), G * s.B * Z);
  return PA_OK;
}

}  // namespace mfma
}  // namespace pa
