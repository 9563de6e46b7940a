// Training of a bf16 layer with 32-wide heads (irregular, structured and Transolver++ variants) as two sequences of the
// library's kernels: the forward keeps what the backward needs in one buffer, the backward leaves every gradient.
// Per-point intermediates that only link two products are formed again or folded away instead of stored:
//   d tok' and d W_out come from sum_n w[n, h, s] dy[n, :] (pa_wgrad.hip), so neither out_x nor a reduction over d out_x
//   is formed; d W_slice, d b_slice are summed inside the per-point kernel, so d z is never stored (pa_mfma_bwd.hip); the
//   irregular layer's projections are computed again in the backward pass.
#include "pa_common.h"
#include "pa_host.h"
#include "pa_mfma_ops.h"

namespace pa {
namespace train {

// ------------------------------------------------------------------------------------------------
// prepare_weights_kernel: the three large weights as the two passes read them, bf16, from float32 or bf16 parameters in
// torch's layout, 32 x 32 tiles turned around through LDS (grid x: tiles, y: taps):
//   w_in   [projection][o][tap][c]          w_in_t  [c][taps - 1 - tap][projection HD + o]   (the transposed convolution)
//   w_out  [c][o]                           w_out_t [o][c]
// and, in the last kSmallBlocks x kSmallParams workgroups, the float32 parameters side by side: the backward pass reads these copies, so that
// the parameters themselves may change between the two passes.
// ------------------------------------------------------------------------------------------------
constexpr int kSmallBlocks = 8, kSmallParams = 10;
struct PrepareArgs {
  const void *w[3];  // in_project_x, in_project_fx (or NULL), out_linear
  uint16_t *w_in, *w_in_t, *w_out, *w_out_t;
  int C, HD, taps, nproj;
  const float *small[kSmallParams];
  int at[kSmallParams + 1], n[kSmallParams];  // where each begins among the copies, its length
  float *copies;
};

template <typename T>
__global__ __launch_bounds__(256) void prepare_weights_kernel(PrepareArgs a) {
  __shared__ float tile[32][33];
  const int t = threadIdx.x, col = t & 31, row0 = t >> 5;
  const int tc = a.C / 32, th = a.HD / 32, per = th * tc;
  int id = blockIdx.x;
  const int which = id / per;  // 0 .. nproj - 1: an input projection, nproj: out_linear, beyond: float32 parameters
  id -= which * per;
  if (which > a.nproj) {
    if (blockIdx.y > 0) return;
    // kSmallBlocks workgroups for each of them: one after the other they are ten trips to memory
    const int k = (int)blockIdx.x - (a.nproj + 1) * per, m = k / kSmallBlocks;
    if (const float *src = a.small[m])
      for (int e = k % kSmallBlocks * 256 + t; e < a.n[m]; e += kSmallBlocks * 256) a.copies[a.at[m] + e] = src[e];
    return;
  }
  const bool out = which == a.nproj;
  const int tap = blockIdx.y;
  if (out && tap > 0) return;
  const int r0 = 32 * (out ? id / th : id / tc), c0 = 32 * (out ? id % th : id % tc);  // rows, columns of the tile
  const T *src = static_cast<const T *>(a.w[out ? 2 : which]);
  const int64_t ld = out ? a.HD : (int64_t)a.C * a.taps;
  const int step = out ? 1 : a.taps;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int r = row0 + 8 * k;
    tile[r][col] = load_as_f32(src + (r0 + r) * ld + (int64_t)(c0 + col) * step + (out ? 0 : tap));
  }
  __syncthreads();
  const int O2 = a.nproj * a.HD;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int r = row0 + 8 * k;
    const uint16_t straight = f32_to_bf16_bits(tile[r][col]), turned = f32_to_bf16_bits(tile[col][r]);
    if (out) {
      a.w_out[(int64_t)(r0 + r) * a.HD + c0 + col] = straight;
      a.w_out_t[(int64_t)(c0 + r) * a.C + r0 + col] = turned;
    } else {
      a.w_in[((int64_t)(which * a.HD + r0 + r) * a.taps + tap) * a.C + c0 + col] = straight;
      a.w_in_t[((int64_t)(c0 + r) * a.taps + (a.taps - 1 - tap)) * O2 + which * a.HD + r0 + col] = turned;
    }
  }
}

static int64_t round_up(int64_t v) { return (v + 255) / 256 * 256; }

// ---- buffer plans ----
struct Saved {  // kept from the forward to the backward pass
  int64_t w_in, w_in_t, w_out, w_out_t, small, w_pack, tok, norm, tok_out, x_mid, fx_mid, a2, total;
};
struct Scratch {
  int64_t blob, fx_pack, partials, tokp, out_x, total;                                     // forward
  int64_t g, x_mid, fx_mid, d_proj, d_tok, d_num, d_norm, attn, parts, point, work, total_backward;  // backward
  int64_t work_bytes;
};

// how the forward hands the attended tokens back to the points
enum class HandBack {
  packed,  // kernel (d) on the bf16 tokens the slice attention packs
  tokens,  // kernel (d) on the float32 tokens
  apart    // out_x on the float32 tokens, out_linear, tail
};
static HandBack hand_back(const pa_shape &s, bool plus) {
  if (!mfma::float_tables(s, plus)) return HandBack::packed;
  return mfma::deslice_project_tokens_supported(s) ? HandBack::tokens : HandBack::apart;
}

static bool fused(const pa_shape &s, bool plus) { return !plus && mfma::supported(PA_BF16, s); }

// The projections, d out_x and the per-point stage of the backward pass in one kernel.  Its workgroups, one per CU, read 3 C / 4
// KB of weights before their first tile.  Many batch elements of one tile each do not pay that back: 2 048 clouds of 16
// points, C = 256, S = 64, 7 180 us against 7 000 for the whole step; 512 of 64 points 1 250 both ways.  Nor do, at C = 128
// where the stages move half as much, fewer than four tiles per CU: the kernels of a step at S = 32 take 165 us against 149
// for 8 192 points, 174 against 163 for 16 384, 189 against 195 for 32 768 and 222 against 246 for 65 536 (C = 256: 187
// against 193 for 2 000, 223 against 232 for 16 384, 503 against 585 for 131 072).
static bool points_in_one(const pa_shape &s, bool plus, int num_cu) {
  if (!fused(s, plus) || !mfma::layer_point_backward_supported(s)) return false;
  if (s.C == 128 && s.B * mfma::tiles_per_batch(s) < 4 * (int64_t)num_cu) return false;
  return s.N > 32 || s.B * s.H <= 4 * (int64_t)num_cu;
}

bool supported(const pa_shape &s, bool plus) {
  if (s.conv_k != 0 && s.conv_tap_major != 1) return false;
  if (!mfma::point_backward_supported(s)) return false;
  return backward::attention_lds_bytes(s) <= kMaxLdsBytes;
}

// where the float32 parameters begin among their copies, each on a 16-byte boundary: in_project_slice weight and bias,
// temperature, qkv_project, the projections' biases, then the four of proj_temperature
static void small_plan(const pa_shape &s, bool plus, int (&at)[kSmallParams + 1], int *len = nullptr) {
  const int HD = (int)s.H * 32, S = (int)s.S;
  const int n[kSmallParams] = {S * 32, S,           (int)s.H,       3 * 32 * 32,  HD, plus ? 0 : HD,
                               plus ? S * 32 : 0, plus ? S : 0, plus ? S : 0, plus ? 1 : 0};
  at[0] = 0;
  for (int m = 0; m < kSmallParams; ++m) {
    at[m + 1] = at[m] + (n[m] + 3) / 4 * 4;
    if (len) len[m] = n[m];
  }
}

static Saved plan_saved(const pa_shape &s, bool plus) {
  const int64_t HD = s.H * 32, taps = grid_taps(&s).taps, np = plus ? 1 : 2, tiles = s.B * mfma::tiles_per_batch(s);
  Saved p{};
  int64_t off = 0;
  auto take = [&](int64_t bytes) {
    const int64_t at = off;
    off += round_up(bytes);
    return at;
  };
  p.w_in = take(np * HD * taps * s.C * 2);
  p.w_in_t = take(np * HD * taps * s.C * 2);
  p.w_out = take(HD * s.C * 2);
  p.w_out_t = take(HD * s.C * 2);
  int at[kSmallParams + 1];
  small_plan(s, plus, at);
  p.small = take((int64_t)at[kSmallParams] * 4);
  p.w_pack = take(tiles * s.H * (s.S / 16) * 1024);
  p.tok = take(s.B * s.H * s.S * 32 * 4);
  p.norm = take(s.B * s.H * s.S * 4);
  p.tok_out = take(s.B * s.H * s.S * 32 * 4);
  if (!fused(s, plus)) {
    p.x_mid = take(s.B * s.N * HD * 2);
    if (!plus) p.fx_mid = take(s.B * s.N * HD * 2);
  }
  if (plus) p.a2 = take(mfma::temperature_hidden_bytes(s));
  p.total = off;
  return p;
}

static int64_t forward_groups(const pa_shape &s, bool plus, int num_cu) {
  return fused(s, plus) && mfma::fuse_reduce(s) ? mfma::project_groups(s, num_cu, true) : mfma::reduce_groups(s);
}

static Scratch plan_scratch(const pa_shape &s, bool plus, int num_cu) {
  const int64_t HD = s.H * 32, M = s.B * s.N, tiles = s.B * mfma::tiles_per_batch(s), BHS = s.B * s.H * s.S;
  Scratch p{};
  int64_t off = 0;
  auto take = [&](int64_t bytes) {
    const int64_t at = off;
    off += round_up(bytes);
    return at;
  };
  p.blob = take(hand_back(s, plus) != HandBack::apart ? mfma::blob_bytes(s) : 0);
  p.fx_pack = take(plus ? 0 : tiles * s.H * 2 * 1024);
  p.partials = take((forward_groups(s, plus, num_cu) + 1) * BHS * 33 * 4);
  p.tokp = take(mfma::tokp_bytes(s));
  p.out_x = take(hand_back(s, plus) == HandBack::apart ? M * HD * 2 : 0);
  p.total = off;

  off = 0;
  const int np = plus ? 1 : 2;
  const bool one = points_in_one(s, plus, num_cu);
  p.g = take(one ? 0 : M * HD * 2);
  if (fused(s, plus) && !one) {
    p.x_mid = take(M * HD * 2);
    p.fx_mid = take(M * HD * 2);
  }
  p.d_proj = take(M * np * HD * 2);
  p.d_tok = take(BHS * 32 * 4);
  p.d_num = take(BHS * 32 * 4);
  p.d_norm = take(BHS * 4);
  p.attn = take(s.B * s.H * 2 * s.S * s.S * 4);
  p.parts = take(s.B * s.H * 3 * 32 * 32 * 4);
  p.work_bytes = wgrad::workspace_bytes(PA_BF16, M, np * HD, s.C, grid_taps(&s).taps, num_cu);
  auto more = [&](int64_t bytes) { p.work_bytes = bytes > p.work_bytes ? bytes : p.work_bytes; };
  more(wgrad::output_backward_workspace_bytes(s, num_cu));
  p.point = take(one ? mfma::layer_point_backward_workspace_bytes(s, num_cu) : mfma::point_backward_workspace_bytes(s, plus, num_cu));
  p.work = take(p.work_bytes);
  p.total_backward = off;
  return p;
}

int64_t saved_bytes(const pa_shape &s, bool plus) { return plan_saved(s, plus).total; }
int64_t forward_workspace_bytes(const pa_shape &s, bool plus, int num_cu) { return plan_scratch(s, plus, num_cu).total; }
int64_t backward_workspace_bytes(const pa_shape &s, bool plus, int num_cu) {
  return plan_scratch(s, plus, num_cu).total_backward;
}

// gradients in one float buffer: d in_project_x (then d in_project_fx) weights, their biases, d W_out, d b_out, d W_qkv,
// then the per-point kernel's (d W_slice, d b_slice, d temperature, Transolver++: d W1, d b1, d w2, d b2)
int64_t grad_floats(const pa_shape &s, bool plus) {
  const int64_t HD = s.H * 32, np = plus ? 1 : 2;
  return np * HD * s.C * grid_taps(&s).taps + np * HD + s.C * HD + s.C + 3 * 32 * 32 + mfma::point_backward_grads(s, plus);
}

// the parameters for the kernels behind prepare_weights: the copies in the saved buffer
struct Prepared {
  pa_params p;
  pa_plus_params q;
};
static Prepared prepared(const pa_shape &s, bool plus, char *sv, const Saved &sp) {
  int at[kSmallParams + 1];
  small_plan(s, plus, at);
  const float *small = reinterpret_cast<const float *>(sv + sp.small);
  Prepared r{};
  r.p.in_project_x_weight = sv + sp.w_in;
  r.p.in_project_fx_weight = plus ? nullptr : sv + sp.w_in + s.H * 32 * s.C * grid_taps(&s).taps * 2;
  r.p.out_linear_weight = sv + sp.w_out;
  r.p.in_project_slice_weight = small + at[0], r.p.in_project_slice_bias = small + at[1];
  r.p.temperature = small + at[2], r.p.qkv_project_weight = small + at[3];
  r.p.in_project_x_bias = small + at[4], r.p.in_project_fx_bias = plus ? nullptr : small + at[5];
  r.q.proj_temperature_0_weight = small + at[6], r.q.proj_temperature_0_bias = small + at[7];
  r.q.proj_temperature_2_weight = small + at[8], r.q.proj_temperature_2_bias = small + at[9];
  return r;
}

int forward(const pa_shape &s, int weight_dtype, const pa_params &params, const pa_plus_params *plus, const void *x,
            const void *uniform, void *y, const pa_block_tail *tail, void *saved, void *workspace, int num_cu, hipStream_t st) {
  const bool pl = plus != nullptr;
  const Saved sp = plan_saved(s, pl);
  const Scratch sc = plan_scratch(s, pl, num_cu);
  char *sv = static_cast<char *>(saved), *ws = static_cast<char *>(workspace);
  const int taps = grid_taps(&s).taps;
  PrepareArgs pa{};
  pa.w[0] = params.in_project_x_weight, pa.w[1] = params.in_project_fx_weight, pa.w[2] = params.out_linear_weight;
  pa.w_in = reinterpret_cast<uint16_t *>(sv + sp.w_in), pa.w_in_t = reinterpret_cast<uint16_t *>(sv + sp.w_in_t);
  pa.w_out = reinterpret_cast<uint16_t *>(sv + sp.w_out), pa.w_out_t = reinterpret_cast<uint16_t *>(sv + sp.w_out_t);
  pa.C = (int)s.C, pa.HD = (int)(s.H * 32), pa.taps = taps, pa.nproj = pl ? 1 : 2;
  const float *small[kSmallParams] = {params.in_project_slice_weight,
                                      params.in_project_slice_bias,
                                      params.temperature,
                                      params.qkv_project_weight,
                                      params.in_project_x_bias,
                                      pl ? nullptr : params.in_project_fx_bias,
                                      pl ? plus->proj_temperature_0_weight : nullptr,
                                      pl ? plus->proj_temperature_0_bias : nullptr,
                                      pl ? plus->proj_temperature_2_weight : nullptr,
                                      pl ? plus->proj_temperature_2_bias : nullptr};
  for (int m = 0; m < kSmallParams; ++m) pa.small[m] = small[m];
  small_plan(s, pl, pa.at, pa.n);
  pa.copies = reinterpret_cast<float *>(sv + sp.small);
  const dim3 grid((unsigned)((pa.nproj + 1) * (s.C / 32) * s.H + kSmallBlocks * kSmallParams), (unsigned)taps);
  if (weight_dtype == PA_F32) hipLaunchKernelGGL(prepare_weights_kernel<float>, grid, dim3(256), 0, st, pa);
  else hipLaunchKernelGGL(prepare_weights_kernel<bf16>, grid, dim3(256), 0, st, pa);
  int rc = launch_status();
  if (rc) return rc;
  Prepared prep = prepared(s, pl, sv, sp);
  prep.p.out_linear_bias = params.out_linear_bias;  // read by the forward pass only
  const pa_params &p = prep.p;
  void *blob = ws + sc.blob, *fx_pack = ws + sc.fx_pack, *tokp = ws + sc.tokp, *w_pack = sv + sp.w_pack;
  float *partials = reinterpret_cast<float *>(ws + sc.partials), *tok = reinterpret_cast<float *>(sv + sp.tok),
        *norm = reinterpret_cast<float *>(sv + sp.norm), *tok_out = reinterpret_cast<float *>(sv + sp.tok_out);
  const int64_t G = forward_groups(s, pl, num_cu);
  const float *fx_bias = nullptr;
  const HandBack how = hand_back(s, pl);
  if (fused(s, pl)) {
    if ((rc = mfma::pack_params(s, p, blob, st))) return rc;
    const bool one = mfma::fuse_reduce(s);
    if ((rc = mfma::project_softmax(s, blob, x, fx_pack, w_pack, one ? partials : nullptr, num_cu, st))) return rc;
    if (!one && (rc = mfma::slice_reduce(s, w_pack, fx_pack, partials, st))) return rc;
    fx_bias = p.in_project_fx_bias;
  } else {
    void *x_mid = sv + sp.x_mid, *fx_mid = pl ? nullptr : sv + sp.fx_mid;
    GemmArgs a{};
    a.in = x;
    a.w[0] = p.in_project_x_weight, a.w[1] = p.in_project_fx_weight;
    a.bias[0] = p.in_project_x_bias, a.bias[1] = p.in_project_fx_bias;
    a.out[0] = x_mid, a.out[1] = fx_mid;
    if (!pl) a.out_pack[1] = fx_pack;  // Transolver++: fx_mid is x_mid, read as rows
    a.M = s.B * s.N;
    a.N = (int)s.N, a.C = (int)s.C, a.O = (int)(s.H * 32);
    a.gh = (int)s.grid_h, a.gw = (int)s.grid_w, a.gd = (int)s.grid_d, a.ks = (int)s.conv_k;
    a.w_tap_major = 1;
    a.K = taps * (int)s.C;
    if (!pl) a.pack_tpb = (int)mfma::tiles_per_batch(s), a.pack_heads = (int)s.H;
    if (!gemm::serves(a, pl ? 1 : 2, 2)) return PA_ERR_UNSUPPORTED;
    if ((rc = gemm::launch(a, pl ? 1 : 2, PA_BF16, st))) return rc;
    rc = pl ? mfma::slice_softmax_pack_plus(s, p, prep.q, x_mid, uniform, w_pack, true, reinterpret_cast<float *>(sv + sp.a2), num_cu, st)
            : mfma::slice_softmax_pack(s, p, x_mid, w_pack, num_cu, st);
    if (rc) return rc;
    rc = pl ? mfma::slice_reduce_rows(s, w_pack, x_mid, partials, st) : mfma::slice_reduce(s, w_pack, fx_pack, partials, st);
    if (rc) return rc;
    if (how != HandBack::apart && (rc = mfma::pack_out_linear(s, p.out_linear_weight, nullptr, p.out_linear_bias, blob, st)))
      return rc;
  }
  if ((rc = mfma::combine_attention(s, p, fx_bias, partials, G, tok, norm, tok_out, tokp, st))) return rc;
  if (how == HandBack::packed) return mfma::deslice_project(s, blob, w_pack, tokp, y, tail, num_cu, st);
  if (how == HandBack::tokens) return mfma::deslice_project_tokens(s, blob, w_pack, tok_out, y, tail, num_cu, st);
  if ((rc = mfma::deslice_tokens(s, w_pack, tok_out, ws + sc.out_x, num_cu, st))) return rc;
  if ((rc = general::out_linear(PA_BF16, s, p, ws + sc.out_x, y, st)) || !tail) return rc;
  return general::residual_ln(PA_BF16, s, y, *tail, st);
}

int backward(const pa_shape &s, bool pl, const void *x, const void *uniform, const void *dy, const void *saved, void *dx,
             float *grads, void *workspace, int num_cu, hipStream_t st) {
  const Saved sp = plan_saved(s, pl);
  const Scratch sc = plan_scratch(s, pl, num_cu);
  char *sv = static_cast<char *>(const_cast<void *>(saved)), *ws = static_cast<char *>(workspace);
  const Prepared prep = prepared(s, pl, sv, sp);
  const pa_params &p = prep.p;
  const int64_t HD = s.H * 32, M = s.B * s.N, taps = grid_taps(&s).taps, np = pl ? 1 : 2;
  float *d_w_in = grads, *d_b_in = d_w_in + np * HD * s.C * taps, *d_w_out = d_b_in + np * HD, *d_b_out = d_w_out + s.C * HD,
        *d_wqkv = d_b_out + s.C, *small = d_wqkv + 3 * 32 * 32;
  const float *tok = reinterpret_cast<float *>(sv + sp.tok), *norm = reinterpret_cast<float *>(sv + sp.norm),
              *tok_out = reinterpret_cast<float *>(sv + sp.tok_out);
  float *d_tok = reinterpret_cast<float *>(ws + sc.d_tok), *d_num = reinterpret_cast<float *>(ws + sc.d_num),
        *d_norm = reinterpret_cast<float *>(ws + sc.d_norm), *parts = reinterpret_cast<float *>(ws + sc.parts);
  void *g = ws + sc.g, *d_proj = ws + sc.d_proj, *point = ws + sc.point, *work = ws + sc.work;
  pa_shape lin = s;
  lin.conv_k = lin.grid_h = lin.grid_w = lin.grid_d = 0;
  int rc = wgrad::output_backward(s, sv + sp.w_pack, dy, tok_out, p.out_linear_weight, work, d_tok, d_w_out, d_b_out, num_cu, st);
  if (rc) return rc;
  if ((rc = backward::slice_attention(s, p, tok, norm, d_tok, reinterpret_cast<float *>(ws + sc.attn), d_num, d_norm, parts, st)))
    return rc;
  wgrad::Sums sums;  // formed together at the end: what their partial results lie in is not used again until then
  sums.add(parts, d_wqkv, 3 * 32 * 32, s.B * s.H);
  if (points_in_one(s, pl, num_cu)) {
    if ((rc = mfma::layer_point_backward(s, p, sv + sp.w_out_t, x, dy, tok_out, d_num, d_norm, point, d_proj, sums, small,
                                         num_cu, st)))
      return rc;
  } else {
    if ((rc = general::rows_gemm(PA_BF16, lin, s.C, HD, dy, sv + sp.w_out_t, nullptr, 0, g, st))) return rc;
    const void *x_mid = sv + sp.x_mid, *fx_mid = pl ? nullptr : sv + sp.fx_mid;
    if (fused(s, pl)) {
      x_mid = ws + sc.x_mid, fx_mid = ws + sc.fx_mid;
      if ((rc = general::project_inputs(PA_BF16, s, p, x, ws + sc.x_mid, ws + sc.fx_mid, st))) return rc;
    }
    if ((rc = mfma::point_backward(s, p, pl ? &prep.q : nullptr, x_mid, fx_mid, g, uniform, tok_out, d_num, d_norm, point, d_proj,
                                   small, num_cu, st, &sums, pl ? reinterpret_cast<const float *>(sv + sp.a2) : nullptr)))
      return rc;
  }
  if (dx && (rc = general::rows_gemm(PA_BF16, s, np * HD, s.C, d_proj, sv + sp.w_in_t, nullptr, 0, dx, st))) return rc;
  if ((rc = wgrad::product(PA_BF16, M, d_proj, np * HD, np * HD, x, s.C, s.C, s.conv_k > 0 ? &s : nullptr, work, d_w_in, d_b_in,
                           num_cu, st, &sums)))
    return rc;
  return wgrad::launch_sums(sums, st);
}

}  // namespace train
}  // namespace pa
