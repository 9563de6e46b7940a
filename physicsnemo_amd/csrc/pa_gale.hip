// GALE (geometry-aware latent embeddings) slice-token stage: cross-attention of the slice tokens to a context and
// the blend with the slice self-attention output (physicsnemo/nn/module/gale.py:87-145 and :43-84).  Everything else of a GALE
// layer (projections, slice softmax, aggregation, slice self-attention, deslice + out_linear) is the PhysicsAttention
// layer's own kernels; this stage sits between the slice self-attention and the deslice.
//
// Workgroups (batch * head, blocks of 16 slice tokens), operands and weights in LDS (every workgroup forms k and v of
// its (batch, head) itself); fp32 arithmetic on the vector ALUs (the stage is S x D work, independent of the
// number of points):
//   q = tok Wq^T + bq (S x D);  k = ctx Wk^T + bk,  v = ctx Wv^T + bv (Sc x D)
//   cross = softmax(q k^T / sqrt(D)) v
//   weighted:        out = sigmoid(m) self + (1 - sigmoid(m)) cross
//   concat_project:  out = gelu([self | cross] Wc^T + bc)
// Bound by latency; the dot products read eight terms ahead (8 heads, 64 slices, 64 context tokens: 27 us, term by term 42).
// The result goes out as float32 (B,H,S,D) and, optionally, as the bf16 operands of the MFMA deslice kernel.
#include "pa_common.h"
#include "pa_host.h"
#include "pa_mfma_ops.h"

namespace pa {
namespace gale {

constexpr int kThreads = 256;
constexpr int kQueryBlock = 16;  // slice tokens per workgroup: grid.y = ceil(S / 16) workgroups share a (batch, head)

__global__ __launch_bounds__(kThreads) void slice_cross_mix_kernel(
    const float *__restrict__ slice_token, const float *__restrict__ self_token, const float *__restrict__ context,
    pa_gale_params gp, float *__restrict__ out_token, uint16_t *__restrict__ tokp, int S, int D, int Sc, int Dc) {
  extern __shared__ float lds[];
  const int D1 = D + 1, Dc1 = Dc + 1;
  float *tok = lds;               // S * D1, later: cross
  float *ctx = tok + S * D1;      // Sc * Dc1
  float *q = ctx + Sc * Dc1;      // S * D1
  float *k = q + S * D1;          // Sc * D1
  float *v = k + Sc * D1;         // Sc * D1
  float *prow = v + Sc * D1;      // (kThreads / 64) * Sc
  float *wq = prow + (kThreads / 64) * Sc;  // D * D1   cross_q weight rows
  float *wk = wq + D * D1;                  // D * Dc1  cross_k weight rows
  float *wv = wk + D * Dc1;                 // D * Dc1  cross_v weight rows
  float *wc = wv + D * Dc1;                 // D * (2D + 1)  concat_project weight rows (that blend mode only)
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
  const int64_t bh = blockIdx.x;
  const int s0 = blockIdx.y * kQueryBlock, s1 = min(S, s0 + kQueryBlock);  // this workgroup's slice tokens
  const float *tk = slice_token + bh * S * D;
  const float *cx = context + bh * Sc * Dc;

#pragma unroll 4
  for (int i = s0 * D + t; i < s1 * D; i += kThreads) tok[(i / D) * D1 + (i % D)] = tk[i];
#pragma unroll 8
  for (int i = t; i < Sc * Dc; i += kThreads) ctx[(i / Dc) * Dc1 + (i % Dc)] = cx[i];
  // the three weights go through LDS: read from global memory inside the dot products, every term waits for its load
#pragma unroll 8
  for (int i = t; i < D * D; i += kThreads) wq[(i / D) * D1 + (i % D)] = gp.cross_q_weight[i];
#pragma unroll 8
  for (int i = t; i < D * Dc; i += kThreads) {
    wk[(i / Dc) * Dc1 + (i % Dc)] = gp.cross_k_weight[i];
    wv[(i / Dc) * Dc1 + (i % Dc)] = gp.cross_v_weight[i];
  }
  if (!gp.state_mixing)
#pragma unroll 8
    for (int i = t; i < D * 2 * D; i += kThreads) wc[(i / (2 * D)) * (2 * D + 1) + (i % (2 * D))] = gp.concat_project_weight[i];
  __syncthreads();
  for (int i = s0 * D + t; i < s1 * D; i += kThreads) {
    const int s = i / D, e = i - s * D;
    const float *wr = wq + e * D1;
    float acc = gp.cross_q_bias[e];
#pragma unroll 8
    for (int d = 0; d < D; ++d) acc = fmaf(tok[s * D1 + d], wr[d], acc);
    q[s * D1 + e] = acc;
  }
  for (int i = t; i < Sc * D; i += kThreads) {
    const int u = i / D, e = i - u * D;
    const float *wkr = wk + e * Dc1, *wvr = wv + e * Dc1;
    float ak = gp.cross_k_bias[e], av = gp.cross_v_bias[e];
#pragma unroll 8
    for (int c = 0; c < Dc; ++c) {
      ak = fmaf(ctx[u * Dc1 + c], wkr[c], ak);
      av = fmaf(ctx[u * Dc1 + c], wvr[c], av);
    }
    k[u * D1 + e] = ak;
    v[u * D1 + e] = av;
  }
  __syncthreads();  // tok is dead from here on: its rows receive the cross-attention output

  const float scale = rsqrtf((float)D);
  float *pr = prow + wave * Sc;
  for (int s = s0 + wave; s < s1; s += kThreads / 64) {
    const float *qs = q + s * D1;
    float mx = -INFINITY;
    for (int u = lane; u < Sc; u += 64) {
      float acc = 0.f;
#pragma unroll 8
      for (int e = 0; e < D; ++e) acc = fmaf(qs[e], k[u * D1 + e], acc);
      acc *= scale;
      pr[u] = acc;
      mx = fmaxf(mx, acc);
    }
    mx = wave_max(mx);
    float sum = 0.f;
    for (int u = lane; u < Sc; u += 64) {
      const float e = expf(pr[u] - mx);
      pr[u] = e;
      sum += e;
    }
    sum = wave_sum(sum);
    const float inv = 1.f / sum;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    for (int e = lane; e < D; e += 64) {
      float acc = 0.f;
#pragma unroll 8
      for (int u = 0; u < Sc; ++u) acc = fmaf(pr[u], v[u * D1 + e], acc);
      tok[s * D1 + e] = acc * inv;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();

  const float *sf = self_token + bh * S * D;
  float mixw = 0.f;
  if (gp.state_mixing) mixw = 1.f / (1.f + expf(-gp.state_mixing[0]));
  const int NCH = S / 16;
  for (int i = s0 * D + t; i < s1 * D; i += kThreads) {
    const int s = i / D, e = i - s * D;
    float o;
    if (gp.state_mixing) {
      o = mixw * sf[i] + (1.f - mixw) * tok[s * D1 + e];
    } else {
      const float *wr = wc + e * (2 * D + 1);
      float acc = gp.concat_project_bias[e];
#pragma unroll 8
      for (int d = 0; d < D; ++d) acc = fmaf(sf[s * D + d], wr[d], acc);
#pragma unroll 8
      for (int d = 0; d < D; ++d) acc = fmaf(tok[s * D1 + d], wr[D + d], acc);
      o = gelu_erf(acc);
    }
    out_token[bh * S * D + i] = o;
    if (tokp) {  // operand order of the MFMA deslice product (D = 32): chunk of 16 slices, lane = 32 g' + d, element j
      const int cq = s >> 4, ss = s & 15, gq = (ss >> 2) & 1, j = 4 * (ss >> 3) + (ss & 3);
      tokp[(((bh * NCH + cq) * 64 + 32 * gq + e) * 8) + j] = f32_to_bf16_bits(o);
    }
  }
}

// ------------------------------------------------------------------------------------------------
// slice_cross_mix_mfma_kernel: the same stage for heads of 32 channels on the float32 matrix instructions.  Workgroup = one
// (batch, head), 4 waves; UT tiles of 32 context tokens.  Every product is arranged so that what it leaves in registers is an
// operand of the next one (accumulator register r of lane half g is row rowmap(r, g), which is also the pair of reduction
// indices that step r of a 32 x 32 x 2 product takes from the two halves):
//   k^T (e x u) = Wk ctx^T + bk,  v (u x e) = ctx Wv^T + bv      one tile per wave, shared through LDS as they lie
//   q^T (e x s) = Wq tok^T + bq;  z^T (u x s) = k q^T;  softmax over u in lane;  cross^T (e x s) = v^T p^T
//   weighted: blend;  concat_project: out^T = Wc [self | cross]^T + bc, GELU      32 slice tokens per wave
// Operands that come from memory are float4 of a row, lane half g holding elements 8 j + 4 g .. + 3.
// Bound by latency (loads, then 90 dependent products of 64 cycles each): 8 heads, 64 slices, 64 context tokens 13 us; the
// kernel on the vector ALUs above, which stays for other widths and longer contexts, 27 us.
// ------------------------------------------------------------------------------------------------
typedef float f32x4 __attribute__((ext_vector_type(4)));
using mfma::f32x16;

__device__ __forceinline__ f32x16 product32(float a, float b, f32x16 acc) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc, 0, 0, 0);
}
// acc += A B^T over n (a multiple of 8) columns of this lane's rows of A and B
__device__ __forceinline__ f32x16 rows_product(const float *a, const float *b, int n, int g, f32x16 acc) {
#pragma unroll 8
  for (int c = 0; c < n; c += 8) {
    const f32x4 x = *reinterpret_cast<const f32x4 *>(a + c + 4 * g), y = *reinterpret_cast<const f32x4 *>(b + c + 4 * g);
#pragma unroll
    for (int m = 0; m < 4; ++m) acc = product32(x[m], y[m], acc);
  }
  return acc;
}

template <int UT>
__global__ __launch_bounds__(kThreads) void slice_cross_mix_mfma_kernel(
    const float *__restrict__ slice_token, const float *__restrict__ self_token, const float *__restrict__ context,
    pa_gale_params gp, float *__restrict__ out_token, uint16_t *__restrict__ tokp, int S, int Sc, int Dc) {
  __shared__ f32x4 tiles[2 * UT][4][64];  // k^T, then v: registers 4 q .. + 3 of a lane
  const int lane = threadIdx.x & 63, i = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t bh = blockIdx.x;
  for (int n = wave; n < 2 * UT; n += kThreads / 64) {
    const int u = 32 * (n % UT) + i;
    const float *cx = context + (bh * Sc + (u < Sc ? u : Sc - 1)) * Dc;
    f32x16 acc;
    if (n < UT) {
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] = gp.cross_k_bias[mfma::rowmap(r, g)];
      acc = rows_product(gp.cross_k_weight + i * Dc, cx, Dc, g, acc);
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] = gp.cross_v_bias[i];
      acc = rows_product(cx, gp.cross_v_weight + i * Dc, Dc, g, acc);
#pragma unroll
      for (int r = 0; r < 16; ++r)  // rows past the context weigh nothing, which an infinity would not survive
        if (32 * (n - UT) + mfma::rowmap(r, g) >= Sc) acc[r] = 0.f;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) tiles[n][q][lane] = f32x4{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
  }
  const int first = wave;
  f32x16 qt;  // of the wave's first tile, ahead of the barrier
  auto query = [&](int st) {
    const int s = 32 * st + i;
#pragma unroll
    for (int r = 0; r < 16; ++r) qt[r] = gp.cross_q_bias[mfma::rowmap(r, g)];
    qt = rows_product(gp.cross_q_weight + i * 32, slice_token + (bh * S + (s < S ? s : S - 1)) * 32, 32, g, qt);
  };
  if (32 * first < S) query(first);
  __syncthreads();
  const float scale = rsqrtf(32.f);
  const float mixw = gp.state_mixing ? 1.f / (1.f + expf(-gp.state_mixing[0])) : 0.f;
  for (int st = first; 32 * st < S; st += kThreads / 64) {
    if (st != first) query(st);
    const int s = 32 * st + i;
    const float *sf = self_token + (bh * S + (s < S ? s : S - 1)) * 32;
    f32x16 z[UT];
    float mx = -INFINITY;
#pragma unroll
    for (int n = 0; n < UT; ++n) {
#pragma unroll
      for (int r = 0; r < 16; ++r) z[n][r] = 0.f;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4 kt = tiles[n][q][lane];
#pragma unroll
        for (int m = 0; m < 4; ++m) z[n] = product32(kt[m], qt[4 * q + m], z[n]);
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        z[n][r] = 32 * n + mfma::rowmap(r, g) < Sc ? z[n][r] * scale : -INFINITY;
        mx = fmaxf(mx, z[n][r]);
      }
    }
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    float sum = 0.f;
#pragma unroll
    for (int n = 0; n < UT; ++n)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        z[n][r] = expf(z[n][r] - mx);
        sum += z[n][r];
      }
    sum += __shfl_xor(sum, 32, 64);
    f32x16 cross;
#pragma unroll
    for (int r = 0; r < 16; ++r) cross[r] = 0.f;
#pragma unroll
    for (int n = 0; n < UT; ++n)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4 v = tiles[UT + n][q][lane];
#pragma unroll
        for (int m = 0; m < 4; ++m) cross = product32(v[m], z[n][4 * q + m], cross);
      }
    const float inv = 1.f / sum;
#pragma unroll
    for (int r = 0; r < 16; ++r) cross[r] *= inv;
    f32x16 o;
    if (gp.state_mixing) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4 own = *reinterpret_cast<const f32x4 *>(sf + 8 * q + 4 * g);
#pragma unroll
        for (int m = 0; m < 4; ++m) o[4 * q + m] = mixw * own[m] + (1.f - mixw) * cross[4 * q + m];
      }
    } else {
      const float *wc = gp.concat_project_weight + i * 64;
#pragma unroll
      for (int r = 0; r < 16; ++r) o[r] = gp.concat_project_bias[mfma::rowmap(r, g)];
      o = rows_product(wc, sf, 32, g, o);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4 w = *reinterpret_cast<const f32x4 *>(wc + 32 + 8 * q + 4 * g);
#pragma unroll
        for (int m = 0; m < 4; ++m) o = product32(w[m], cross[4 * q + m], o);
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) o[r] = gelu_erf(o[r]);
    }
    if (s < S) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<f32x4 *>(out_token + (bh * S + s) * 32 + 8 * q + 4 * g) =
            f32x4{o[4 * q], o[4 * q + 1], o[4 * q + 2], o[4 * q + 3]};
      if (tokp) {  // the operand order of the deslice product, as above
        const int cq = s >> 4, ss = s & 15, gq = (ss >> 2) & 1, j = 4 * (ss >> 3) + (ss & 3);
        uint16_t *to = tokp + ((bh * (S / 16) + cq) * 64 + 32 * gq) * 8 + j;
#pragma unroll
        for (int r = 0; r < 16; ++r) to[mfma::rowmap(r, g) * 8] = f32_to_bf16_bits(o[r]);
      }
    }
  }
}

// out_token (B,H,S,32) float32 -> the bf16 operands of the MFMA deslice kernel (same order as above)
__global__ __launch_bounds__(kThreads) void pack_tokens_kernel(const float *__restrict__ out_token,
                                                               uint16_t *__restrict__ tokp, int S) {
  const int64_t bh = blockIdx.x;
  const int NCH = S / 16;
  for (int i = threadIdx.x; i < S * 32; i += kThreads) {
    const int s = i >> 5, e = i & 31;
    const int cq = s >> 4, ss = s & 15, gq = (ss >> 2) & 1, j = 4 * (ss >> 3) + (ss & 3);
    tokp[(((bh * NCH + cq) * 64 + 32 * gq + e) * 8) + j] = f32_to_bf16_bits(out_token[bh * S * 32 + i]);
  }
}

int pack_tokens(const pa_shape &s, const float *out_token, void *tokp, hipStream_t st) {
  hipLaunchKernelGGL(pack_tokens_kernel, dim3((unsigned)(s.B * s.H)), dim3(kThreads), 0, st, out_token,
                     static_cast<uint16_t *>(tokp), (int)s.S);
  return launch_status();
}

size_t lds_bytes(const pa_shape &s, int64_t Sc, int64_t Dc) {
  return (size_t)(2 * s.S * (s.D + 1) + Sc * (Dc + 1) + 2 * Sc * (s.D + 1) + (kThreads / 64) * Sc +
                  s.D * (s.D + 1) + 2 * s.D * (Dc + 1) + s.D * (2 * s.D + 1)) * 4;
}

int slice_cross_mix(const pa_shape &s, const pa_gale_params &gp, int64_t Sc, int64_t Dc, const float *slice_token,
                    const float *self_token, const float *context, float *out_token, void *tokp, hipStream_t st) {
  // heads of 32 channels, context rows of whole pairs of float4, up to 128 context tokens (a lane's scores: 64 registers)
  bool mfma = s.D == 32 && Dc % 8 == 0 && Sc <= 128;
  for (const void *p : {(const void *)slice_token, (const void *)self_token, (const void *)context, (const void *)out_token,
                        (const void *)gp.cross_q_weight, (const void *)gp.cross_k_weight, (const void *)gp.cross_v_weight,
                        (const void *)gp.concat_project_weight})
    mfma = mfma && aligned16(p);
  if (mfma) {
    auto launch = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3((unsigned)(s.B * s.H)), dim3(kThreads), 0, st, slice_token, self_token, context, gp,
                         out_token, static_cast<uint16_t *>(tokp), (int)s.S, (int)Sc, (int)Dc);
      return launch_status();
    };
    return Sc <= 32   ? launch(slice_cross_mix_mfma_kernel<1>)
           : Sc <= 64 ? launch(slice_cross_mix_mfma_kernel<2>)
                      : launch(slice_cross_mix_mfma_kernel<4>);
  }
  const size_t lds = lds_bytes(s, Sc, Dc);
  int rc = allow_dynamic_lds(slice_cross_mix_kernel, lds);
  if (rc) return rc;
  hipLaunchKernelGGL(slice_cross_mix_kernel, dim3((unsigned)(s.B * s.H), (unsigned)((s.S + kQueryBlock - 1) / kQueryBlock)),
                     dim3(kThreads), lds, st, slice_token,
                     self_token, context, gp, out_token, static_cast<uint16_t *>(tokp), (int)s.S, (int)s.D, (int)Sc,
                     (int)Dc);
  return launch_status();
}

}  // namespace gale
}  // namespace pa
