// Training of a float32 layer (irregular and structured, any head width of the general kernels) as two sequences of the
// library's kernels, one call each way: the stages keep what they kept one by one (x_mid, fx_mid, slice weights, tokens, out_x),
// the weights are turned around by one kernel, and the gradients leave in one buffer.  The sums of the small gradients over
// heads are one kernel instead of tensor operations.  Bound by the stages (their own files); what this saves is launches and
// the host's way between them: a training step of four blocks on a 60 x 60 grid, 128 channels, 4 300 us on the stages one by one,
// 3 170 us here; on 4 x 85 x 85 grids, where the kernels count, 5 100 and 4 760 us.
#include "pa_common.h"
#include "pa_host.h"

namespace pa {
namespace train_f32 {

// ------------------------------------------------------------------------------------------------
// prepare_weights_kernel: the three large weights as the two passes read them, 32 x 32 tiles turned around through LDS (grid x:
// tiles, y: taps), and in the last workgroups the small parameters that the backward pass reads:
//   w_in [projection][o][tap][c] (taps > 1)    w_in_t [c][taps - 1 - tap][projection HD + o]    w_out_t [o][c]
// ------------------------------------------------------------------------------------------------
constexpr int kSmallBlocks = 4, kSmallParams = 4;
struct PrepareArgs {
  const float *w[3];  // in_project_x, in_project_fx, out_linear
  float *w_in, *w_in_t, *w_out_t;
  int C, HD, taps;
  const float *small[kSmallParams];
  int at[kSmallParams], n[kSmallParams];
  float *copies;
};

__global__ __launch_bounds__(256) void prepare_weights_kernel(PrepareArgs a) {
  __shared__ float tile[32][33];
  const int t = threadIdx.x, col = t & 31, row0 = t >> 5;
  const int tc = (a.C + 31) / 32, th = (a.HD + 31) / 32, per = th * tc;
  const int which = blockIdx.x / per, id = blockIdx.x - which * per;
  if (which > 2) {
    if (blockIdx.y > 0) return;
    for (int m = 0; m < kSmallParams; ++m)
      for (int e = (blockIdx.x - 3 * per) * 256 + t; e < a.n[m]; e += kSmallBlocks * 256) a.copies[a.at[m] + e] = a.small[m][e];
    return;
  }
  const bool out = which == 2;
  const int tap = blockIdx.y;
  if (out && tap > 0) return;
  const int r0 = 32 * (out ? id / th : id / tc), c0 = 32 * (out ? id % th : id % tc);  // rows, columns of the tile
  const int R = out ? a.C : a.HD, Q = out ? a.HD : a.C;
  const int64_t ld = out ? a.HD : (int64_t)a.C * a.taps;
  const int step = out ? 1 : a.taps;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int r = row0 + 8 * k;
    if (r0 + r < R && c0 + col < Q) tile[r][col] = a.w[which][(r0 + r) * ld + (int64_t)(c0 + col) * step + (out ? 0 : tap)];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int r = row0 + 8 * k;
    if (!out && a.w_in && r0 + r < R && c0 + col < Q)
      a.w_in[((int64_t)(which * a.HD + r0 + r) * a.taps + tap) * a.C + c0 + col] = tile[r][col];
    if (c0 + r >= Q || r0 + col >= R) continue;
    if (out) a.w_out_t[(int64_t)(c0 + r) * a.C + r0 + col] = tile[col][r];
    else a.w_in_t[((int64_t)(c0 + r) * a.taps + (a.taps - 1 - tap)) * 2 * a.HD + which * a.HD + r0 + col] = tile[col][r];
  }
}

// tokens[bhs][d] = sums[bhs][d]: the weighted sums without the column of their counts
__global__ __launch_bounds__(256) void take_tokens_kernel(const float *__restrict__ sums, float *__restrict__ tokens, int64_t n, int D) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e < n) tokens[e] = sums[e / D * (D + 1) + e % D];
}

// The gradients that are sums over heads: d W_slice and d b_slice from the diagonal blocks of P = d z^T x_mid ((H S) x (H D)) and
// its column sums; d temperature where the clamp lets it through.
__global__ __launch_bounds__(256) void head_sums_kernel(const float *__restrict__ P, const float *__restrict__ sums,
                                                        const float *__restrict__ d_clamped, const float *__restrict__ temperature,
                                                        float *__restrict__ d_ws, float *__restrict__ d_bs, float *__restrict__ d_t,
                                                        int H, int S, int D) {
  const int e = blockIdx.x * 256 + threadIdx.x;
  if (e < S * D) {
    const int s = e / D, d = e - s * D;
    float v = 0.f;
    for (int h = 0; h < H; ++h) v += P[(int64_t)(h * S + s) * H * D + h * D + d];
    d_ws[e] = v;
  } else if (e < S * D + S) {
    const int s = e - S * D;
    float v = 0.f;
    for (int h = 0; h < H; ++h) v += sums[h * S + s];
    d_bs[s] = v;
  } else if (e < S * D + S + H) {
    const int h = e - S * D - S;
    const float t = temperature[h];
    d_t[h] = t >= kTempMin && t <= kTempMax ? d_clamped[h] : 0.f;
  }
}

static int64_t round_up(int64_t v) { return (v + 255) / 256 * 256; }

struct Saved {  // kept from the forward to the backward pass
  int64_t w_in_t, w_out_t, small, x_mid, fx_mid, w, tok, norm, tok_out, out_x, total;
};
struct Scratch {
  int64_t w_in, partials, total;                                                                                    // forward
  int64_t g, d_tok, d_num, d_norm, attn, parts, d_proj, d_z, d_t, t_sum, heads, work[3], total_backward;
  bool served;  // by the row-axis products
  bool narrow;  // the per-point stages on the kernels of narrow heads
};
struct Taker {
  int64_t off = 0;
  int64_t operator()(int64_t bytes) {
    const int64_t at = off;
    off += round_up(bytes);
    return at;
  }
};

// where the small parameters begin among their copies: in_project_slice weight and bias, temperature, qkv_project
static void small_plan(const pa_shape &s, int (&at)[kSmallParams], int (&n)[kSmallParams], int *total) {
  const int len[kSmallParams] = {(int)(s.S * s.D), (int)s.S, (int)s.H, (int)(3 * s.D * s.D)};
  int off = 0;
  for (int m = 0; m < kSmallParams; ++m) at[m] = off, n[m] = len[m], off += (len[m] + 3) / 4 * 4;
  *total = off;
}

static Saved plan_saved(const pa_shape &s) {
  const int64_t HD = s.H * s.D, M = s.B * s.N, BHS = s.B * s.H * s.S;
  Saved p{};
  Taker take;
  int at[kSmallParams], n[kSmallParams], small;
  small_plan(s, at, n, &small);
  p.w_in_t = take(2 * HD * grid_taps(&s).taps * s.C * 4);
  p.w_out_t = take(HD * s.C * 4);
  p.small = take((int64_t)small * 4);
  p.x_mid = take(M * HD * 4), p.fx_mid = take(M * HD * 4), p.out_x = take(M * HD * 4);
  p.w = take(M * s.H * s.S * 4);
  p.tok = take(BHS * s.D * 4), p.norm = take(BHS * 4), p.tok_out = take(BHS * s.D * 4);
  p.total = take.off;
  return p;
}

static int64_t sum_groups(const pa_shape &s, int num_cu) {  // partial token sums
  return narrow::points_supported(s) ? narrow::point_groups(s, num_cu) : general::partial_count(s);
}

static Scratch plan_scratch(const pa_shape &s, int num_cu) {
  const int64_t HD = s.H * s.D, HS = s.H * s.S, M = s.B * s.N, BHS = s.B * HS, taps = grid_taps(&s).taps;
  Scratch p{};
  Taker take;
  p.narrow = narrow::points_supported(s);
  p.partials = take((sum_groups(s, num_cu) + 1) * BHS * (s.D + 1) * 4);
  Taker back = take;
  p.w_in = take(taps > 1 ? 2 * HD * taps * s.C * 4 : 0);
  p.total = take.off;
  p.g = back(M * HD * 4);
  p.d_tok = back(BHS * s.D * 4), p.d_num = back(BHS * s.D * 4), p.d_norm = back(BHS * 4);
  p.attn = back(s.B * s.H * 2 * s.S * s.S * 4);
  p.parts = back(s.B * s.H * 3 * s.D * s.D * 4);
  p.d_proj = back(M * 2 * HD * 4), p.d_z = back(p.narrow ? 0 : M * HS * 4);
  p.d_t = back(p.narrow ? narrow::point_backward_rows(s, num_cu) * (s.S * (s.D + 1) + s.H) * 4 : backward::point_tiles(s) * s.H * 4);
  p.t_sum = back(s.H * 4);
  p.heads = back(p.narrow ? 0 : (HS * HD + HS) * 4);
  const int64_t work[3] = {wgrad::workspace_bytes(PA_F32, M, s.C, HD, 1, num_cu),
                           p.narrow ? 256 : wgrad::workspace_bytes(PA_F32, M, HS, HD, 1, num_cu),
                           wgrad::workspace_bytes(PA_F32, M, 2 * HD, s.C, (int)taps, num_cu)};
  p.served = true;
  for (int k = 0; k < 3; ++k) {
    p.served = p.served && work[k] > 0;
    p.work[k] = back(work[k] > 0 ? work[k] : 0);
  }
  p.total_backward = back.off;
  return p;
}

// The shapes of the general backward kernels whose weight gradients the row-axis products serve and whose d W_slice is the
// diagonal of one product over whole points (wider ones are formed head by head).
bool supported(const pa_shape &s, int num_cu) {
  if (s.conv_k != 0 && s.conv_tap_major != 1) return false;
  if (backward::attention_lds_bytes(s) > kMaxLdsBytes || backward::point_tile_rows(s) == 0) return false;
  if (s.H < 2 || s.H * s.S > 512 || s.C % 4 != 0 || s.H * s.D % 4 != 0) return false;
  return plan_scratch(s, num_cu).served;
}

int64_t saved_bytes(const pa_shape &s) { return plan_saved(s).total; }
int64_t forward_workspace_bytes(const pa_shape &s, int num_cu) { return plan_scratch(s, num_cu).total; }
int64_t backward_workspace_bytes(const pa_shape &s, int num_cu) { return plan_scratch(s, num_cu).total_backward; }
int64_t grad_floats(const pa_shape &s) {
  const int64_t HD = s.H * s.D;
  return 2 * HD * s.C * grid_taps(&s).taps + 2 * HD + s.C * HD + s.C + 3 * s.D * s.D + s.S * s.D + s.S + s.H;
}

int forward(const pa_shape &s, const pa_params &params, const void *x, void *y, const pa_block_tail *tail, void *saved,
            void *workspace, int num_cu, hipStream_t st) {
  const Saved sp = plan_saved(s);
  const Scratch sc = plan_scratch(s, num_cu);
  char *sv = static_cast<char *>(saved), *ws = static_cast<char *>(workspace);
  auto f = [](char *p, int64_t at) { return reinterpret_cast<float *>(p + at); };
  const int taps = grid_taps(&s).taps, HD = (int)(s.H * s.D), C = (int)s.C;
  PrepareArgs pa{};
  pa.w[0] = static_cast<const float *>(params.in_project_x_weight), pa.w[1] = static_cast<const float *>(params.in_project_fx_weight);
  pa.w[2] = static_cast<const float *>(params.out_linear_weight);
  pa.w_in = taps > 1 ? f(ws, sc.w_in) : nullptr, pa.w_in_t = f(sv, sp.w_in_t), pa.w_out_t = f(sv, sp.w_out_t);
  pa.C = C, pa.HD = HD, pa.taps = taps;
  const float *small[kSmallParams] = {params.in_project_slice_weight, params.in_project_slice_bias, params.temperature,
                                      params.qkv_project_weight};
  int total;
  small_plan(s, pa.at, pa.n, &total);
  for (int m = 0; m < kSmallParams; ++m) pa.small[m] = small[m];
  pa.copies = f(sv, sp.small);
  const int tiles = ((C + 31) / 32) * ((HD + 31) / 32);
  hipLaunchKernelGGL(prepare_weights_kernel, dim3((unsigned)(3 * tiles + kSmallBlocks), (unsigned)taps), dim3(256), 0, st, pa);
  int rc = launch_status();
  if (rc) return rc;
  pa_params p = params;
  if (taps > 1) {
    p.in_project_x_weight = pa.w_in;
    p.in_project_fx_weight = pa.w_in + (int64_t)HD * taps * C;
  }
  float *partials = f(ws, sc.partials), *tok = f(sv, sp.tok), *norm = f(sv, sp.norm), *tok_out = f(sv, sp.tok_out);
  void *x_mid = sv + sp.x_mid, *fx_mid = sv + sp.fx_mid, *w = sv + sp.w, *out_x = sv + sp.out_x;
  if ((rc = general::project_inputs(PA_F32, s, p, x, x_mid, fx_mid, st))) return rc;
  if (sc.narrow) {
    pa_params copies{};  // on their 16-byte boundaries
    copies.in_project_slice_weight = pa.copies + pa.at[0], copies.in_project_slice_bias = pa.copies + pa.at[1];
    copies.temperature = pa.copies + pa.at[2];
    rc = narrow::point_sums(s, &copies, static_cast<float *>(x_mid), static_cast<float *>(fx_mid), static_cast<float *>(w), partials,
                            num_cu, st);
  } else {
    if ((rc = general::slice_softmax(PA_F32, s, p, x_mid, w, st))) return rc;
    rc = general::slice_partial(PA_F32, s, w, fx_mid, partials, st);
  }
  if (rc) return rc;
  if ((rc = general::combine_attention(s, p, partials, sum_groups(s, num_cu), tok, norm, tok_out, st))) return rc;
  if ((rc = general::deslice(PA_F32, s, w, tok_out, out_x, st))) return rc;
  if ((rc = general::out_linear(PA_F32, s, p, out_x, y, st)) || !tail) return rc;
  return general::residual_ln(PA_F32, s, y, *tail, st);
}

int backward(const pa_shape &s, const void *x, const void *dy, const void *saved, void *dx, float *grads, void *workspace,
             int num_cu, hipStream_t st) {
  const Saved sp = plan_saved(s);
  const Scratch sc = plan_scratch(s, num_cu);
  char *sv = static_cast<char *>(const_cast<void *>(saved)), *ws = static_cast<char *>(workspace);
  auto f = [](char *p, int64_t at) { return reinterpret_cast<float *>(p + at); };
  const int64_t HD = s.H * s.D, HS = s.H * s.S, M = s.B * s.N, BHS = s.B * HS, taps = grid_taps(&s).taps;
  float *d_w_in = grads, *d_b_in = d_w_in + 2 * HD * s.C * taps, *d_w_out = d_b_in + 2 * HD, *d_b_out = d_w_out + s.C * HD,
        *d_wqkv = d_b_out + s.C, *d_ws = d_wqkv + 3 * s.D * s.D, *d_bs = d_ws + s.S * s.D, *d_t = d_bs + s.S;
  int at[kSmallParams], n[kSmallParams], total;
  small_plan(s, at, n, &total);
  const float *small = f(sv, sp.small);
  pa_params p{};
  p.in_project_slice_weight = small + at[0], p.in_project_slice_bias = small + at[1], p.temperature = small + at[2];
  p.qkv_project_weight = small + at[3];
  const float *tok = f(sv, sp.tok), *norm = f(sv, sp.norm), *tok_out = f(sv, sp.tok_out);
  float *partials = f(ws, sc.partials), *d_tok = f(ws, sc.d_tok), *d_num = f(ws, sc.d_num), *d_norm = f(ws, sc.d_norm),
        *parts = f(ws, sc.parts), *t_tiles = f(ws, sc.d_t), *t_sum = f(ws, sc.t_sum), *heads = f(ws, sc.heads);
  void *g = ws + sc.g, *d_proj = ws + sc.d_proj, *d_z = ws + sc.d_z;
  const void *x_mid = sv + sp.x_mid, *fx_mid = sv + sp.fx_mid, *w = sv + sp.w, *out_x = sv + sp.out_x;
  pa_shape lin = s;
  lin.conv_k = lin.grid_h = lin.grid_w = lin.grid_d = 0;
  int rc = general::rows_gemm(PA_F32, lin, s.C, HD, dy, sv + sp.w_out_t, nullptr, 0, g, st);
  if (rc) return rc;
  // adjoint of the deslice w.r.t. the attended tokens, then the slice attention and the normalisation
  const float *sums = nullptr;
  rc = sc.narrow ? narrow::point_sums(s, nullptr, nullptr, static_cast<float *>(g), const_cast<float *>(static_cast<const float *>(w)),
                                      partials, num_cu, st)
                 : general::slice_partial(PA_F32, s, w, g, partials, st);
  if (rc) return rc;
  if ((rc = general::combine_partials(s, partials, sum_groups(s, num_cu), &sums, st))) return rc;
  hipLaunchKernelGGL(take_tokens_kernel, dim3((unsigned)((BHS * s.D + 255) / 256)), dim3(256), 0, st, sums, d_tok, BHS * s.D, (int)s.D);
  if ((rc = launch_status())) return rc;
  if ((rc = backward::slice_attention(s, p, tok, norm, d_tok, f(ws, sc.attn), d_num, d_norm, parts, st))) return rc;
  wgrad::Sums totals;  // formed together at the end: what their partial results lie in is not used again until then
  totals.add(parts, d_wqkv, 3 * s.D * s.D, s.B * s.H);
  // per point: slice softmax, aggregation and deslice adjoints
  if (sc.narrow) {
    auto in = [](const void *q) { return static_cast<const float *>(q); };
    rc = narrow::point_backward(s, p, in(x_mid), in(fx_mid), in(g), tok_out, d_num, d_norm, static_cast<float *>(d_proj), t_tiles, num_cu, st);
    totals.add(t_tiles, d_ws, s.S * (s.D + 1) + s.H, narrow::point_backward_rows(s, num_cu));  // d_ws, d_bs, d_t
  } else {
    rc = backward::slice_softmax(PA_F32, s, p, x_mid, fx_mid, w, g, tok_out, d_num, d_norm, d_proj, d_z, t_tiles, st);
    totals.add(t_tiles, t_sum, s.H, backward::point_tiles(s));
  }
  if (rc) return rc;
  if ((rc = wgrad::product(PA_F32, M, dy, s.C, s.C, out_x, HD, HD, nullptr, ws + sc.work[0], d_w_out, d_b_out, num_cu, st, &totals)))
    return rc;
  if (!sc.narrow && (rc = wgrad::product(PA_F32, M, d_z, HS, HS, x_mid, HD, HD, nullptr, ws + sc.work[1], heads, heads + HS * HD, num_cu,
                                         st, &totals)))
    return rc;
  if (dx && (rc = general::rows_gemm(PA_F32, s, 2 * HD, s.C, d_proj, sv + sp.w_in_t, nullptr, 0, dx, st))) return rc;
  if ((rc = wgrad::product(PA_F32, M, d_proj, 2 * HD, 2 * HD, x, s.C, s.C, s.conv_k > 0 ? &s : nullptr, ws + sc.work[2], d_w_in, d_b_in,
                           num_cu, st, &totals)))
    return rc;
  if ((rc = wgrad::launch_sums(totals, st)) || sc.narrow) return rc;
  hipLaunchKernelGGL(head_sums_kernel, dim3((unsigned)((s.S * s.D + s.S + s.H + 255) / 256)), dim3(256), 0, st, heads, heads + HS * HD,
                     t_sum, small + at[2], d_ws, d_bs, d_t, (int)s.H, (int)s.S, (int)s.D);
  return launch_status();
}

}  // namespace train_f32
}  // namespace pa
