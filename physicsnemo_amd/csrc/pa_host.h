// Host-side declarations shared by the kernel translation units and the C ABI.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "../../include/physattn.h"

namespace pa {

constexpr size_t kMaxLdsBytes = 160 * 1024;  // LDS per workgroup on gfx950

// result of the launch just enqueued, as a C-ABI return code
inline int launch_status() {
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? PA_OK : (int)e;
}

// opt a kernel in to more than the default 48 KiB of dynamic LDS
// (the attribute is per kernel and per device: remembered for the device it was last set on, so the steady state of a
// process that stays on one GPU makes no runtime call here)
template <typename F>
inline int allow_dynamic_lds(F kernel, size_t bytes) {
  if (bytes > kMaxLdsBytes) return PA_ERR_UNSUPPORTED;
  if (bytes > 48 * 1024) {
    static thread_local const void *last_kernel = nullptr;
    static thread_local size_t last_bytes = 0;
    static thread_local int last_dev = -1;
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess) dev = -1;
    const void *k = reinterpret_cast<const void *>(kernel);
    if (k == last_kernel && bytes <= last_bytes && dev == last_dev && dev >= 0) return PA_OK;
    hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
    if (e != hipSuccess) return (int)e;
    last_kernel = k;
    last_bytes = bytes;
    last_dev = dev;
  }
  return PA_OK;
}

// Arguments of the row GEMMs: out[m, o] = bias[o] + sum_k A(m, k) * W[o, k]
//   linear: A(m, k) = in[m*K + k]
//   conv  : K = taps*C, k = tap*C + c; 2-D: taps = ks^2, tap = u*ks + v, A(m,k) = in[b, (i+u-p)*gw + (j+v-p), c];
//           3-D: taps = ks^3, tap = (u*ks + v)*ks + z, A(m,k) = in[b, ((i+u-p)*gw + (j+v-p))*gd + (l+z-p), c];
//           0 outside the grid; the PyTorch weight element is W[o, c, u, v(, z)] = W[o*K + c*taps + tap].
// Up to two (W, bias, out) sets share the same input (x_mid and fx_mid), selected by blockIdx.z.
struct GemmArgs {
  const void *in;
  const void *w[2];
  const float *bias[2];
  void *out[2];
  int64_t M;   // rows = B*N
  int K, O;    // reduction length, output columns
  int C, N, gh, gw, ks;  // conv geometry (ks = 0: linear)
  int gd;                // depth of a 3-D grid (0: 2-D)
  int w_tap_major;       // conv weights as (O, taps, C) (= the reduction order k = tap * C + c) instead of (O, C, taps)
  // MFMA kernel only, bf16, Linear, O = 32 * pack_heads: pack_tpb > 0 walks the rows batch by batch in tiles of 32
  // points (pack_tpb tiles per batch, the last one padded) and also writes each (tile, head) block of the result in
  // the packed operand layout of the MFMA slice kernels (fx_pack).  out[z] may then be NULL.
  void *out_pack[2];
  int pack_tpb, pack_heads;
  int act;  // applied to out (not to out_pack): 0 none, 1 GELU in its erf form (torch.nn.GELU default)
};

namespace gemm {
// MFMA row GEMM (fp32: v_mfma_f32_32x32x2_f32, bf16: v_mfma_f32_32x32x16_bf16); `serves` tells whether the shape and
// the pointers meet its 16-byte granularity, otherwise the scalar kernel of the general family runs.
bool serves(const GemmArgs &a, int nsets, size_t elem_bytes);
int launch(const GemmArgs &a, int nsets, int dtype, hipStream_t st);
// weight-gradient products over the row axis: partials[g][oa][ob] = sum over chunk g of A[m][oa] * B[m][ob] (bf16 in)
int64_t cols_gemm_chunks(int64_t M, int64_t OA, int num_cu);
int cols_gemm(const void *A, int64_t lda, int64_t OA, const void *B, int64_t ldb, int64_t OB, int64_t M,
              float *partials, float *col_sums, int num_cu, hipStream_t st);
// the same for float32 operands (fp32 MFMA)
int64_t cols_gemm_f32_chunks(int64_t M, int64_t OA, int64_t OB, int num_cu);
int cols_gemm_f32(const void *A, int64_t lda, int64_t OA, const void *B, int64_t ldb, int64_t OB, int64_t M,
                  const pa_shape *shape, float *partials, float *col_sums, int num_cu, hipStream_t st);
}  // namespace gemm

namespace wgrad {
// Totals of partial results, dst[e] = sum over g < G of src[g][e], collected so that one launch forms several of them: every
// result's partials stay where they are until then.
struct Sums {
  static constexpr int kMost = 8;
  struct One {
    const float *src;
    float *dst;
    int64_t n, first;     // elements; the launch's first workgroup for them
    int G, taps, OB;      // taps > 1: src is [oa][tap][ob], dst the order of a convolution's weight, [oa][ob][tap]
    int lanes;            // of a workgroup along the elements, 4 elements each (0: 32 lanes, one element each;
                          // < 0: the taps together)
  } r[kMost];
  int count = 0;
  int64_t blocks = 0;
  bool by_taps = false;  // one of them takes the taps of a convolution's weight together
  static constexpr int kTaps = 9;
  // Large results stream rows of 256 to 1024 bytes per partial, more workgroups rather than longer rows where there are
  // few elements; small results have too few elements to fill the chip and split the partials instead, 32 ways.
  void add(const float *src, float *dst, int64_t n, int64_t G, int taps = 1, int64_t OB = 1) {
    const bool units = n % 4 == 0 && reinterpret_cast<uintptr_t>(src) % 16 == 0;
    // A workgroup takes 256 neighbouring ob of one oa, all taps, where there are enough of those (lanes < 0): three for every two
    // CUs.  By taps / by rows, us, results of 256, 320, 384, 448, 512 workgroups: 9 taps, 14 partials 11.6 / 10.3, 13.1 / 11.9,
    // 13.8 / 13.9, 14.2 / 17.2, 15.2 / 18.4; 25 taps 19.6 / 19.6, 21.2 / 21.8, 22.5 / 25.3 (OB = 512: 22.4 / 20.5), 24.2 / 29.5,
    // 26.1 / 33.0; 27 taps 24.9 / 23.7, 17.5 / 21.4, 19.0 / 25.9, 20.2 / 28.9, 22.2 / 32.6.  With 128 they take 1.7 to 1.9 times as long.
    if (units && taps > 1 && OB % 256 == 0 && n / (taps * 256) >= 384) {
      r[count++] = One{src, dst, n, blocks, (int)G, taps, (int)OB, -1};
      blocks += n / (taps * 256);
      by_taps = true;
      return;
    }
    const int lanes = !units ? 0 : n < 65536 ? 8 : G < 32 ? 64 : n < 262144 ? 16 : 32, per = lanes ? 4 * lanes : 32;
    r[count++] = One{src, dst, n, blocks, (int)G, taps, (int)OB, lanes};
    blocks += (n + per - 1) / per;
  }
};
int launch_sums(const Sums &sums, hipStream_t st);
// out[oa][ob] (grid: [oa][ob][tap]) = sum_m A[m][oa] B[m][ob] and the column sums of A; `workspace`: workspace_bytes()
int64_t workspace_bytes(int dtype, int64_t M, int64_t OA, int64_t OB, int taps, int num_cu);
int product(int dtype, int64_t M, const void *A, int64_t lda, int64_t OA, const void *B, int64_t ldb, int64_t OB,
            const pa_shape *grid, void *workspace, float *out, float *col_sums, int num_cu, hipStream_t st,
            Sums *later = nullptr);  // later: the totals are left to its launch
// the bf16 tile kernel alone, G partial results
int launch_wide(const void *A, int64_t lda, int64_t OA, const void *B, int64_t ldb, int64_t OB, int64_t M, int64_t G,
                const pa_shape *grid, float *partials, float *col_sums, hipStream_t st);
int sum_rows(const float *src, int64_t rows, int64_t n, float *dst, hipStream_t st);
int64_t output_backward_workspace_bytes(const pa_shape &s, int num_cu);
int output_backward(const pa_shape &s, const void *w_pack, const void *dy, const float *out_token, const void *w_out,
                    void *workspace, float *d_out_token, float *d_w_out, float *d_b_out, int num_cu, hipStream_t st);
}  // namespace wgrad

namespace train {
// training of a bf16 layer (32-wide heads): see pa_layer_train_forward / _backward
bool supported(const pa_shape &s, bool plus);
int64_t saved_bytes(const pa_shape &s, bool plus);
int64_t forward_workspace_bytes(const pa_shape &s, bool plus, int num_cu);
int64_t backward_workspace_bytes(const pa_shape &s, bool plus, int num_cu);
int64_t grad_floats(const pa_shape &s, bool plus);
int forward(const pa_shape &s, int weight_dtype, const pa_params &p, const pa_plus_params *plus, const void *x,
            const void *uniform, void *y, const pa_block_tail *tail, void *saved, void *workspace, int num_cu, hipStream_t st);
int backward(const pa_shape &s, bool plus, const void *x, const void *uniform, const void *dy, const void *saved, void *dx,
             float *grads, void *workspace, int num_cu, hipStream_t st);
}  // namespace train

namespace train_f32 {
// the same for float32 layers: see pa_layer_train_f32_forward / _backward
bool supported(const pa_shape &s, int num_cu);
int64_t saved_bytes(const pa_shape &s);
int64_t forward_workspace_bytes(const pa_shape &s, int num_cu);
int64_t backward_workspace_bytes(const pa_shape &s, int num_cu);
int64_t grad_floats(const pa_shape &s);
int forward(const pa_shape &s, const pa_params &p, const void *x, void *y, const pa_block_tail *tail, void *saved, void *workspace,
            int num_cu, hipStream_t st);
int backward(const pa_shape &s, const void *x, const void *dy, const void *saved, void *dx, float *grads, void *workspace,
             int num_cu, hipStream_t st);
}  // namespace train_f32

namespace general {
int dequant_e4m3(const void *in, const float *scale, void *out, int64_t rows, int64_t cols, hipStream_t st);
int project_inputs(int dtype, const pa_shape &s, const pa_params &p, const void *x, void *x_mid, void *fx_mid,
                   hipStream_t st);
int out_linear(int dtype, const pa_shape &s, const pa_params &p, const void *out_x, void *y, hipStream_t st);
int rows_gemm(int dtype, const pa_shape &grid, int64_t c_in, int64_t c_out, const void *in, const void *weight,
              const float *bias, int act, void *out, hipStream_t st);
int rows_gemm_packed(const pa_shape &s, int64_t c_in, const void *in, const void *weight, const float *bias, void *out,
                     void *out_pack, hipStream_t st);
int slice_softmax(int dtype, const pa_shape &s, const pa_params &p, const void *x_mid, void *w, hipStream_t st);
int slice_softmax_plus(int dtype, const pa_shape &s, const pa_params &p, const pa_plus_params &pp, const void *x_mid,
                       const void *uniform, void *w, void *scratch, hipStream_t st);
int64_t partial_count(const pa_shape &s);
size_t combine_attn_lds_bytes(const pa_shape &s);
int slice_partial(int dtype, const pa_shape &s, const void *w, const void *fx_mid, float *partials, hipStream_t st);
int combine_partials(const pa_shape &s, const float *partials, int64_t G, const float **combined, hipStream_t st);
int combine_attention(const pa_shape &s, const pa_params &p, const float *partials, int64_t G, float *slice_token,
                      float *slice_norm, float *out_token, hipStream_t st);
int deslice(int dtype, const pa_shape &s, const void *w, const float *out_token, void *out_x, hipStream_t st);
int residual_ln(int dtype, const pa_shape &s, void *y, const pa_block_tail &tail, hipStream_t st);
int64_t layernorm_backward_groups(int64_t rows);
int layernorm_backward(int dtype, int64_t rows, int64_t C, const void *x, const void *dy, const void *add, const float *gamma,
                       float eps, void *dx, float *partials, float *grads, hipStream_t st);
}  // namespace general

namespace conv {
// float32 structured 2-D front end (C = 128, 8 heads of 16, 32 slices): both convolutions on split-bf16 MFMA products,
// slice softmax and partial token sums in one launch.  `w`: (B, N, H, S) float32; `partials`: groups(s) partials of
// B * H * S * (D + 1) floats each, in the layout the general combine kernels read.
bool supported(int dtype, const pa_shape &s);
int64_t groups(const pa_shape &s);
int64_t blob_bytes(const pa_shape &s);
// blob_out (may be NULL): f32rows::backend_blob_bytes() that receive out_linear's weight in the form f32rows::backend
// reads, cut by the same launch that cuts the convolution weights
// (with mlp: f32rows::block_blob_bytes(mlp->F), and the block MLP's weights behind it, as f32rows::block_tail reads)
int front(const pa_shape &s, const pa_params &p, const void *x, void *blob, void *w, float *partials, void *blob_out,
          const pa_block_mlp *mlp, hipStream_t st);
}  // namespace conv

namespace f32rows {
// float32 per-point kernels of a 128-wide block on split-bf16 products.  backend: out_x = w . out_token per head
// (8 heads of 16, 32 slices; w (B, N, H, S), out_token (B, H, S, D)), y = out_x W_out^T + b_out and the tail, one
// launch; blob: backend_blob_bytes() of scratch for the repacked W_out.  mlp_*: Mlp(128 -> F -> 128), F a multiple of
// 128, with the same tail; blob: mlp_blob_bytes(F) written by mlp_pack.
bool backend_supported(int dtype, const pa_shape &s);
int64_t backend_blob_bytes();
int backend(const pa_shape &s, const pa_params &p, const void *w, const float *out_token, void *y,
            const pa_block_tail *tail, void *blob, bool blob_ready, hipStream_t st);
bool mlp_supported(int dtype, int64_t rows, int64_t C, int64_t F);
int64_t mlp_blob_bytes(int64_t F);
int mlp_pack(int64_t F, const void *w1, const void *w2, void *blob, hipStream_t st);
int mlp_forward(int64_t rows, int64_t F, const void *blob, const float *b1, const float *b2, const void *u, void *y,
                const pa_block_tail *tail, hipStream_t st);
// the whole per-point tail of a block in one launch: hand-back, out_linear, + fx_in, LayerNorm, Mlp, + residual, next
// LayerNorm (see pa_block_forward); blob: block_blob_bytes(F) of scratch
bool block_supported(int dtype, const pa_shape &s, int64_t F);
int64_t block_blob_bytes(int64_t F);
int block_tail(const pa_shape &s, const pa_params &p, const pa_block_mlp &m, const void *w, const float *out_token,
               const void *fx_in, void *fx_out, const pa_block_tail *next, const pa_block_head *head, void *blob,
               bool blob_ready, hipStream_t st);
// the model's preprocess Mlp, Linear(c_in -> F) -> GELU -> Linear(F -> 128), c_in <= 8, with the tail (the first
// LayerNorm); blob: premlp_blob_bytes(F) of scratch
bool premlp_supported(int dtype, int64_t rows, int64_t c_in, int64_t F, int64_t C);
int64_t premlp_blob_bytes(int64_t F);
int premlp_forward(int64_t rows, int64_t c_in, int64_t F, const void *w1, const float *b1, const void *w2,
                   const float *b2, const void *u, void *y, const pa_block_tail *tail, void *blob, hipStream_t st);
}  // namespace f32rows

namespace narrow {
// float32 blocks of 32 or 64 channels (heads of 8 or 16, 32 slices, irregular mesh): `front` leaves the slice weights
// (B, N, H, S) and groups() partial token sums as the general combine kernels read them, block_tail is
// f32rows::block_tail for these widths
bool block_supported(int dtype, const pa_shape &s, int64_t F);
int64_t groups(const pa_shape &s, int num_cu);
int front(const pa_shape &s, const pa_params &p, const void *x, float *w, float *partials, int num_cu, hipStream_t st);
int block_tail(const pa_shape &s, const pa_params &p, const pa_block_mlp &m, const float *w, const float *out_token,
               const void *fx_in, void *fx_out, const pa_block_tail *next, const pa_block_head *head, int num_cu,
               hipStream_t st);
// float32 training, heads of 16 channels and 32 slices: the slice softmax of x_mid's rows with the token sums of v's (p NULL: the
// sums alone, of the weights w), point_groups() partials as the general combine kernels read them; and the per-point adjoints
// with d W_slice | d b_slice | d temperature (masked where clamped), point_backward_rows() partial rows of S 17 + H floats
bool points_supported(const pa_shape &s);
int64_t point_groups(const pa_shape &s, int num_cu);
int64_t point_backward_rows(const pa_shape &s, int num_cu);
int point_sums(const pa_shape &s, const pa_params *p, const float *x_mid, const float *v, float *w, float *partials, int num_cu,
               hipStream_t st);
int point_backward(const pa_shape &s, const pa_params &p, const float *x_mid, const float *fx_mid, const float *g,
                   const float *out_token, const float *d_num, const float *d_norm, float *d_proj, float *partials, int num_cu,
                   hipStream_t st);
}  // namespace narrow

namespace backward {
size_t attention_lds_bytes(const pa_shape &s);
int slice_attention(const pa_shape &s, const pa_params &p, const float *slice_token, const float *slice_norm,
                    const float *d_out_token, float *scratch, float *d_num, float *d_norm, float *d_wqkv_part,
                    hipStream_t st);
int point_tile_rows(const pa_shape &s, bool plus = false);  // plus: the Transolver++ form of the per-point kernel
int64_t point_tiles(const pa_shape &s, bool plus = false);
int slice_softmax(int dtype, const pa_shape &s, const pa_params &p, const void *x_mid, const void *fx_mid,
                  const void *w, const void *d_out_x, const float *out_token, const float *d_num, const float *d_norm,
                  void *d_proj, void *d_z, float *dT_part, hipStream_t st);
int slice_softmax_plus(int dtype, const pa_shape &s, const pa_params &p, const pa_plus_params &pp, const void *x_mid,
                       const void *uniform, const void *w, const void *d_out_x, const float *out_token,
                       const float *d_num, const float *d_norm, void *d_x_mid, void *d_z, void *d_a1, float *d_a2,
                       float *dT_part, hipStream_t st);
}  // namespace backward

namespace flare {
int64_t column_max_chunks(const pa_shape &s);
int column_weights(int dtype, const pa_shape &s, const void *a, float *partial, float *colmax, void *wc,
                   hipStream_t st);
// temperature: NULL, or (H) float32 -- the entries are then divided by clamp(temperature[head], 0.5, 5) first
int softmax_rows(int dtype, const pa_shape &s, void *a, const float *temperature, hipStream_t st);
int column_max(int dtype, const pa_shape &s, const void *a, float *partial, float *colmax, hipStream_t st);
// bf16 scores (B,N,H,S) -> exp(A - column max) and softmax_s(A) in the packed layout of the MFMA slice kernels
int pack_weights(const pa_shape &s, const void *scores, const float *colmax, void *wc_pack, void *wr_pack, int num_cu,
                 hipStream_t st);
int normalise(const pa_shape &s, const float *sums, float *z, hipStream_t st);
int backward_tile_rows(const pa_shape &s);
int backward_points(int dtype, const pa_shape &s, const void *wr, const void *wc, const void *v, const void *g,
                    const float *z, const float *d_num, const float *d_den, void *d_a, void *d_v, hipStream_t st);
}  // namespace flare

namespace gale {
size_t lds_bytes(const pa_shape &s, int64_t Sc, int64_t Dc);
int pack_tokens(const pa_shape &s, const float *out_token, void *tokp, hipStream_t st);
int slice_cross_mix(const pa_shape &s, const pa_gale_params &gp, int64_t Sc, int64_t Dc, const float *slice_token,
                    const float *self_token, const float *context, float *out_token, void *tokp, hipStream_t st);
}  // namespace gale

namespace ballquery {
int ball_query(int64_t B, int64_t Np, int64_t Nq, int64_t K, float radius, const float *points, const float *queries,
               int64_t *indices, float *out_points, float *out_dists, int32_t *counts, hipStream_t st);
int ball_query_cells(int64_t B, int64_t Np, int64_t Nq, int64_t K, float radius, int64_t G, const float *grid,
                     const float *sorted_points, const int32_t *sorted_index, const int32_t *cell_start,
                     const float *queries, const int32_t *query_order, int64_t *indices, float *out_points,
                     float *out_dists, int32_t *counts, hipStream_t st);
}  // namespace ballquery

namespace mfma {
bool staged_supported(int dtype, const pa_shape &s);
int slice_softmax_pack_plus(const pa_shape &s, const pa_params &p, const pa_plus_params &pp, const void *x_mid,
                            const void *uniform, void *w_pack, bool split, float *a2_out, int num_cu, hipStream_t st);
int slice_softmax_pack(const pa_shape &s, const pa_params &p, const void *x_mid, void *w_pack, int num_cu,
                       hipStream_t st);
// the same weights recomputed where they are used, never stored: token sums (softmax_reduce_groups partials) and
// the hand-back to the points (out_x may be x_mid)
int64_t softmax_reduce_groups(const pa_shape &s, int num_cu);
// packed_x: x_mid (and out_x) are packed operand tiles [tile][head][2][64 lanes] of 16 bytes instead of rows
int slice_softmax_reduce(const pa_shape &s, const pa_params &p, const void *x_mid, bool packed_x, const void *fx_pack,
                         float *partials, int num_cu, hipStream_t st);
// token sums of inputs with few channels, straight from x (softmax_reduce_groups partials)
bool thin_tokens_supported(const pa_shape &s);
int thin_tokens(const pa_shape &s, const pa_params &p, const void *x, float *partials, int num_cu, hipStream_t st);
int deslice_recompute(const pa_shape &s, const pa_params &p, const void *x_mid, bool packed_x, const void *tokp,
                      void *out_x, int num_cu, hipStream_t st);
bool backward_supported(const pa_shape &s);
int64_t backward_groups(const pa_shape &s, int num_cu);
int64_t backward_tables_bytes(const pa_shape &s);
int slice_softmax_backward(const pa_shape &s, const pa_params &p, const void *x_mid, const void *fx_mid,
                           const void *d_out_x, const void *w_pack, const float *out_token, const float *d_num,
                           const float *d_norm, void *tables, void *d_proj, void *d_z, float *dT_part, int num_cu,
                           hipStream_t st);
int deslice_natural(const pa_shape &s, const void *w_pack, const void *tokp, void *out_x, int num_cu, hipStream_t st);
// out_x and, further down, the whole hand-back on the float32 attended tokens (B, H, S, 32) instead of bf16 fragments
int deslice_tokens(const pa_shape &s, const void *w_pack, const float *tokens, void *out_x, int num_cu, hipStream_t st);
bool deslice_project_tokens_supported(const pa_shape &s);
int deslice_project_tokens(const pa_shape &s, const void *blob, const void *w_pack, const float *tokens, void *y,
                           const pa_block_tail *tail, int num_cu, hipStream_t st);
bool float_tables(const pa_shape &s, bool plus);  // training multiplies with float32 tables and tokens, not bf16 ones
bool layer_point_backward_supported(const pa_shape &s);
int64_t layer_point_backward_workspace_bytes(const pa_shape &s, int num_cu);
int layer_point_backward(const pa_shape &s, const pa_params &p, const void *w_out_t, const void *x, const void *dy,
                         const float *out_token, const float *d_num, const float *d_norm, void *workspace, void *d_proj,
                         wgrad::Sums &later, float *grads, int num_cu, hipStream_t st);
int backward_tables(const pa_shape &s, const float *w_slice, const float *pt_w1, const float *out_token, const float *d_num,
                    bool split, void *tabs, hipStream_t st);
bool point_backward_supported(const pa_shape &s);
int64_t point_backward_grads(const pa_shape &s, bool plus);
int64_t point_backward_workspace_bytes(const pa_shape &s, bool plus, int num_cu);
// Transolver++: a2 [tile][H][32], what proj_temperature's second Linear gives; without one from the forward pass the workspace
// ends in as many bytes to form it in
int64_t temperature_hidden_bytes(const pa_shape &s);
int point_backward(const pa_shape &s, const pa_params &p, const pa_plus_params *plus, const void *x_mid,
                   const void *fx_mid, const void *d_out_x, const void *uniform, const float *out_token,
                   const float *d_num, const float *d_norm, void *workspace, void *d_proj, float *grads, int num_cu,
                   hipStream_t st, wgrad::Sums *later = nullptr, const float *a2 = nullptr);
bool supported(int dtype, const pa_shape &s);
int64_t tiles_per_batch(const pa_shape &s);
int64_t reduce_groups(const pa_shape &s);
int64_t blob_bytes(const pa_shape &s);
int64_t fx_pack_bytes(const pa_shape &s);
int64_t w_pack_bytes(const pa_shape &s);
int64_t tokp_bytes(const pa_shape &s);
int pack_params(const pa_shape &s, const pa_params &p, void *blob, hipStream_t st);
int pack_out_linear(const pa_shape &s, const void *w_out, const float *w_scale, const float *b_out, void *blob,
                    hipStream_t st);
int64_t project_groups(const pa_shape &s, int num_cu, bool fused);
bool fuse_reduce(const pa_shape &s);
int project_softmax(const pa_shape &s, const void *blob, const void *x, void *fx_pack, void *w_pack, float *partials,
                    int num_cu, hipStream_t st);
// the fused form with the shader clock of one of its workgroups reported (C = 256, S <= 64): clock_out[0] = shader
// cycles, clock_out[1] = ticks of the 100 MHz wall clock
int project_softmax_clocked(const pa_shape &s, const void *blob, const void *x, void *w_pack, float *partials,
                            uint64_t *clock_out, int num_cu, hipStream_t st);
int slice_reduce(const pa_shape &s, const void *w_pack, const void *fx_pack, float *partials, hipStream_t st);
// the same on fx_mid as (B, N, H*32) rows
int slice_reduce_rows(const pa_shape &s, const void *w_pack, const void *fx_mid, float *partials, hipStream_t st);
int combine_attention(const pa_shape &s, const pa_params &p, const float *fx_bias, const float *partials, int64_t G,
                      float *slice_token, float *slice_norm, float *out_token, void *tokp, hipStream_t st);
int deslice_project(const pa_shape &s, const void *blob, const void *w_pack, const void *tokp, void *y,
                    const pa_block_tail *tail, int num_cu, hipStream_t st);
// kernel (d) fed with x_mid tiles: the slice weights are recomputed per tile and never stored (S = 128)
bool deslice_recompute_project_supported(const pa_shape &s);
int deslice_recompute_project(const pa_shape &s, const pa_params &p, const void *blob, const void *xm_pack,
                              const void *tokp, void *y, const pa_block_tail *tail, int num_cu, hipStream_t st);
}  // namespace mfma

namespace mlp {
bool supported(int dtype, int64_t rows, int64_t C, int64_t F);
int64_t blob_bytes(int64_t C, int64_t F);
// w*_scale: nullptr for bf16 weights; else the weight is fp8-e4m3 bytes with one float32 scale per output row
int pack(int64_t C, int64_t F, const void *w1, const float *w1_scale, const void *w2, const float *w2_scale, void *blob,
         hipStream_t st);
// LayerNorm applied to the input rows on their way into the first product (gamma == nullptr: none)
struct InputLn {
  const float *gamma = nullptr, *beta = nullptr;
  float eps = 0.f;
};
bool input_ln_supported(int dtype, int64_t rows, int64_t C, int64_t F);
int forward(int64_t rows, int64_t C, int64_t F, const void *blob, const float *b1, const float *b2, const void *u,
            void *y, const pa_block_tail *tail, const InputLn &in, int num_cu, hipStream_t st);
// the same with GELU to float32 accuracy (C = 256)
int train_forward(int64_t rows, int64_t C, int64_t F, const void *blob, const float *b1, const float *b2, const void *u,
                  void *y, const pa_block_tail *tail, int num_cu, hipStream_t st);
// backward of the hidden layer (pa_mlp_bwd.hip): act = gelu(W1 u + b1), dh = (W2^T dy) * gelu'(W1 u + b1), (rows, F) bf16
bool hidden_backward_supported(int64_t rows, int64_t C, int64_t F);
int64_t hidden_backward_blob_bytes(int64_t C, int64_t F);
int hidden_backward(int64_t rows, int64_t C, int64_t F, const void *w1, const float *b1, const void *w2, const void *u,
                    const void *dy, void *act, void *dh, void *blob, void *w1_t, int num_cu, hipStream_t st);
// the preprocess MLP (c_in <= 16 inputs -> F -> C in {256, 512}) with the hidden layer kept on chip; bf16 rows and weights
bool premlp_supported(int dtype, int64_t rows, int64_t c_in, int64_t F, int64_t C);
int64_t premlp_blob_bytes(int64_t F, int64_t C);
int premlp(int64_t rows, int64_t c_in, int64_t F, int64_t C, const void *w1, const float *b1, const void *w2,
           const float *b2, const void *u, void *y, const float *ln_gamma, const float *ln_beta, float ln_eps,
           void *ln_out, void *blob, int num_cu, hipStream_t st);
// y = W x + bias [+ residual] [-> LayerNorm] for bf16 rows, W (C x C) bf16 row-major; blob: linear_blob_bytes(C) of scratch
bool linear_supported(int dtype, int64_t rows, int64_t C);
int64_t linear_blob_bytes(int64_t C);
int linear(int64_t rows, int64_t C, const void *w, const float *w_scale, const float *bias, const void *x, void *y,
           const pa_block_tail *tail, void *blob, int num_cu, hipStream_t st);
// the same with x as packed operand tiles [B tpb][C / 32][2][64 lanes] (k order kperm within a head)
int linear_packed(int64_t B, int64_t N, int64_t C, const void *w, const float *w_scale, const float *bias,
                  const void *x_pack, void *y, const pa_block_tail *tail, void *blob, int num_cu, hipStream_t st);
// the layer's two Linear input projections as packed operand tiles; blob: 2 linear_blob_bytes(C) of scratch
int project_packed(int64_t B, int64_t N, int64_t C, const void *w_x, const float *s_x, const float *b_x, const void *w_fx,
                   const float *s_fx, const float *b_fx, const void *x, void *xm_pack, void *fx_pack, void *blob,
                   int num_cu, hipStream_t st);
// the same for the k x k (x k) grid convolutions of the structured layers, as an implicit GEMM over taps x channels;
// blob: conv_project_blob_bytes(C, taps) of scratch
bool conv_project_supported(int dtype, int64_t B, int64_t N, int64_t C);
int64_t conv_project_blob_bytes(int64_t C, int64_t taps);
int conv_project_packed(int64_t B, int64_t N, int64_t C, int64_t gh, int64_t gw, int64_t gd, int64_t k, int tap_major,
                        const void *w_x, const float *b_x, const void *w_fx, const float *b_fx, const void *x,
                        void *xm_pack, void *fx_pack, void *blob, int num_cu, hipStream_t st);
}  // namespace mlp

namespace norm {
bool rows_ln_backward_supported(int64_t rows, int64_t C, int64_t K);
int64_t rows_ln_backward_groups(int64_t rows, int num_cu);
int rows_ln_backward(int64_t rows, int64_t K, const void *dh, const void *wt, const void *x, const float *gamma, float eps,
                     const void *add, void *dx, float *partials, float *grads, int num_cu, hipStream_t st, wgrad::Sums &later);
}  // namespace norm

}  // namespace pa
