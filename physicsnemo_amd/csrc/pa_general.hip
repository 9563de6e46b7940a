// General PhysicsAttention kernels: any (C, H, D, S) within the library limits, fp32 or bf16 storage,
// fp32 arithmetic on the vector ALUs, natural tensor layouts.  They serve fp32 runs (rtol 1e-4 class),
// the structured-2D (Conv2d) projections and every shape the MFMA kernels do not cover.
//
// Stage map (reference lines in include/physattn.h):
//   rows_gemm_kernel          in_project_x / in_project_fx (Linear or k x k Conv2d as implicit GEMM), out_linear
//   rows GEMM + softmax_rows  in_project_slice, then clamp(temperature) + softmax over S in place (pa_flare.hip)
//   slice_partial_kernel      per-chunk sums  sum_n w[n,s] * [fx_mid[n,:], 1]
//   slice_combine_attn_kernel fixed-order combine, / (norm + 1e-2), qkv, softmax(q k^T / sqrt D) v   (LDS resident)
//   deslice_kernel            out_x[n,h,:] = sum_s w[n,h,s] * tok'[h,s,:]
//   residual_ln_kernel        fx_new = y + residual; ln_out = LayerNorm(fx_new)
#include <type_traits>

#include "pa_common.h"
#include "pa_host.h"

namespace pa {
namespace general {

// ------------------------------------------------------------------------------------------------
// rows_gemm_kernel: out[m, o] = bias[o] + sum_k A(m, k) * W[o, k]
//   linear: A(m, k) = in[m*K + k]
//   conv  : K = taps*C, k = tap*C + c; 2-D: taps = ks^2, tap = u*ks + v, A(m,k) = in[b, (i+u-p)*gw + (j+v-p), c];
//           3-D: taps = ks^3, tap = (u*ks + v)*ks + z, A(m,k) = in[b, ((i+u-p)*gw + (j+v-p))*gd + (l+z-p), c];
//           0 outside the grid; the PyTorch weight element is W[o, c, u, v(, z)] = W[o*K + c*taps + tap].
// 64x64 output tile per 256-thread workgroup, 4x4 outputs per thread, K staged 16 at a time through LDS.
// blockIdx.z selects one of two (W, bias, out) sets that share the same input (x_mid and fx_mid).
// ------------------------------------------------------------------------------------------------
// four consecutive elements with one 8- or 16-byte access
template <typename T>
__device__ __forceinline__ void load4(const T *p, float (&v)[4]) {
  if constexpr (sizeof(T) == 2) {
    const uint2 r = *reinterpret_cast<const uint2 *>(p);
    const T *e = reinterpret_cast<const T *>(&r);
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = load_as_f32(e + j);
  } else {
    const float4 r = *reinterpret_cast<const float4 *>(p);
    v[0] = r.x, v[1] = r.y, v[2] = r.z, v[3] = r.w;
  }
}
template <typename T>
__device__ __forceinline__ void store4(T *p, const float (&v)[4]) {
  if constexpr (sizeof(T) == 2) {
    alignas(8) T o[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) store_from_f32(o + j, v[j]);
    *reinterpret_cast<uint2 *>(p) = *reinterpret_cast<const uint2 *>(o);
  } else {
    *reinterpret_cast<float4 *>(p) = float4{v[0], v[1], v[2], v[3]};
  }
}

template <typename TA, typename TW>
__global__ __launch_bounds__(256) void rows_gemm_kernel(GemmArgs a) {
  __shared__ float As[16][64 + 4];
  __shared__ float Ws[16][64 + 4];
  const int z = blockIdx.z;
  const TA *in = static_cast<const TA *>(a.in);
  const TW *W = static_cast<const TW *>(a.w[z]);
  const float *bias = a.bias[z];
  TA *out = static_cast<TA *>(a.out[z]);
  const int t = threadIdx.x;
  const int tx = t & 15, ty = t >> 4;
  const int64_t m0 = (int64_t)blockIdx.x * 64;
  const int o0 = blockIdx.y * 64;
  const int lr = t >> 2;         // tile row / tile out column this thread stages
  const int lk = (t & 3) * 4;    // first of 4 consecutive k it stages
  const int pad = a.ks / 2;
  const int gd = a.gd > 0 ? a.gd : 1;          // a 2-D grid is a 3-D grid of depth 1 with a single depth tap
  const int ksd = a.gd > 0 ? a.ks : 1;
  const int taps = a.ks * a.ks * ksd;

  // decode the staged row once
  const int64_t m_ld = m0 + lr;
  const bool m_ok = m_ld < a.M;
  int64_t b_ld = 0;
  int i_ld = 0, j_ld = 0, l_ld = 0;
  if (a.ks > 0 && m_ok) {
    b_ld = m_ld / a.N;
    int n = (int)(m_ld - b_ld * a.N);
    l_ld = n % gd;
    n /= gd;
    i_ld = n / a.gw;
    j_ld = n - i_ld * a.gw;
  }
  const int o_ld = o0 + lr;

  float acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;

  // a Linear whose rows are whole numbers of four elements is staged with 8- / 16-byte loads
  const bool vec = a.ks == 0 && a.K % 4 == 0 && reinterpret_cast<uintptr_t>(in) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(W) % 16 == 0;
  const bool vec_out = a.O % 4 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0;
  for (int k0 = 0; k0 < a.K; k0 += 16) {
    if (vec) {
      float av4[4] = {0.f, 0.f, 0.f, 0.f}, wv4[4] = {0.f, 0.f, 0.f, 0.f};
      if (k0 + lk < a.K) {
        if (m_ok) load4(in + m_ld * a.K + k0 + lk, av4);
        if (o_ld < a.O) load4(W + (int64_t)o_ld * a.K + k0 + lk, wv4);
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        As[lk + q][lr] = av4[q];
        Ws[lk + q][lr] = wv4[q];
      }
    } else if (a.ks == 0) {  // all eight loads together, from the last element where there is none: a choice each is a trip each
      float av[4], wv[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int k = k0 + lk + q < a.K ? k0 + lk + q : a.K - 1;
        av[q] = load_as_f32(in + (m_ok ? m_ld : a.M - 1) * a.K + k);
        wv[q] = load_as_f32(W + (int64_t)(o_ld < a.O ? o_ld : a.O - 1) * a.K + k);
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const bool k_ok = k0 + lk + q < a.K;
        As[lk + q][lr] = k_ok && m_ok ? av[q] : 0.f;
        Ws[lk + q][lr] = k_ok && o_ld < a.O ? wv[q] : 0.f;
      }
    } else
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int k = k0 + lk + q;
      float av = 0.f, wv = 0.f;
      if (k < a.K) {
        const int tap = k / a.C, c = k - tap * a.C;
        const int uv = tap / ksd, z = tap - uv * ksd;
        const int u = uv / a.ks, v = uv - u * a.ks;
        const int ii = i_ld + u - pad, jj = j_ld + v - pad, ll = l_ld + (a.gd > 0 ? z - pad : 0);
        if (m_ok && ii >= 0 && ii < a.gh && jj >= 0 && jj < a.gw && ll >= 0 && ll < gd)
          av = load_as_f32(in + ((b_ld * a.N + ((int64_t)ii * a.gw + jj) * gd + ll) * a.C + c));
        if (o_ld < a.O)
          wv = load_as_f32(W + (int64_t)o_ld * a.K + (a.w_tap_major ? (int64_t)k : (int64_t)c * taps + tap));
      }
      As[lk + q][lr] = av;
      Ws[lk + q][lr] = wv;
    }
    __syncthreads();
    auto step = [&](int kk) {
      float av[4], wv[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) av[i] = As[kk][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) wv[j] = Ws[kk][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(av[i], wv[j], acc[i][j]);
    };
    if (a.K - k0 >= 16) {
#pragma unroll
      for (int kk = 0; kk < 16; ++kk) step(kk);
    } else {  // few inputs: 49 380 x 5 -> 128 14.6 us with whole blocks and a trip per load, 12.1 here
      for (int kk = 0; kk < a.K - k0; ++kk) step(kk);
    }
    __syncthreads();
  }
  float bv[4] = {0.f, 0.f, 0.f, 0.f};
  if (bias) {
#pragma unroll
    for (int j = 0; j < 4; ++j) bv[j] = bias[o0 + tx * 4 + j < a.O ? o0 + tx * 4 + j : a.O - 1];
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t m = m0 + ty * 4 + i;
    if (m >= a.M) continue;
    if (vec_out && o0 + tx * 4 < a.O) {
      float v4[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float v = acc[i][j] + bv[j];
        v4[j] = a.act == 1 ? gelu_erf(v) : v;
      }
      store4(out + m * a.O + o0 + tx * 4, v4);
      continue;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int o = o0 + tx * 4 + j;
      if (o < a.O) {
        const float v = acc[i][j] + bv[j];
        store_from_f32(out + m * a.O + o, a.act == 1 ? gelu_erf(v) : v);
      }
    }
  }
}

// ------------------------------------------------------------------------------------------------
// slice_softmax_plus_kernel: the Transolver++ form of slice_softmax_kernel (PA.py:166-170, gumbel_softmax.py:49-57).
//   temp[r,h]  = max(temperature[h] + gelu(b2 + sum_s w2[s] gelu(b1[s] + x_mid[r,h,:] . w1[s,:])), 0.01)
//   w[r,h,:]   = softmax_s((logits[r,h,s] - log(-log(u[r,h,s] + 1e-8) + 1e-8)) / temp[r,h])
// `uniform` holds the caller's U[0,1) samples in the activation type (what torch.rand_like(logits) draws).
// ------------------------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void slice_softmax_plus_kernel(
    const T *__restrict__ x_mid, const T *__restrict__ uniform, const float *__restrict__ w_slice,
    const float *__restrict__ b_slice, const float *__restrict__ temperature, const float *__restrict__ pt_w1,
    const float *__restrict__ pt_b1, const float *__restrict__ pt_w2, const float *__restrict__ pt_b2,
    T *__restrict__ w_out, int64_t M, int H, int D, int S, int R) {
  extern __shared__ float lds[];
  float *xs = lds;                       // R * H * (D+1)
  float *wsl = xs + R * H * (D + 1);     // S * D
  float *bsl = wsl + S * D;              // S
  float *w1 = bsl + S;                   // S * D
  float *b1 = w1 + S * D;                // S
  float *w2 = b1 + S;                    // S
  float *lg = w2 + S;                    // R * H * (S+1)
  const int t = threadIdx.x;
  const int64_t m0 = (int64_t)blockIdx.x * R;
  const int rows = (int)min((int64_t)R, M - m0);
  const int HD = H * D, HS = H * S;
  for (int i = t; i < rows * HD; i += 256) {
    const int r = i / HD, c = i - r * HD;
    const int h = c / D, d = c - h * D;
    xs[(r * H + h) * (D + 1) + d] = load_as_f32(x_mid + (m0 + r) * HD + c);
  }
  for (int i = t; i < S * D; i += 256) {
    wsl[i] = w_slice[i];
    w1[i] = pt_w1[i];
  }
  for (int i = t; i < S; i += 256) {
    bsl[i] = b_slice[i];
    b1[i] = pt_b1[i];
    w2[i] = pt_w2[i];
  }
  for (int i = t; i < rows * HS; i += 256) {
    const int pair = i / S, s = i - pair * S;
    lg[pair * (S + 1) + s] = load_as_f32(uniform + m0 * HS + i);
  }
  __syncthreads();
  for (int pair = t; pair < rows * H; pair += 256) {
    const int h = pair % H;
    const float *xr = xs + pair * (D + 1);
    float *lrow = lg + pair * (S + 1);
    float tacc = pt_b2[0];
    for (int s = 0; s < S; ++s) {
      float acc = b1[s];
      const float *wr = w1 + s * D;
      for (int d = 0; d < D; ++d) acc = fmaf(xr[d], wr[d], acc);
      tacc = fmaf(w2[s], gelu_erf(acc), tacc);
    }
    const float temp = round_to(w_out, fmaxf(temperature[h] + gelu_erf(tacc), 0.01f));
    float mx = -INFINITY;
    for (int s = 0; s < S; ++s) {
      float acc = 0.f;
      const float *wr = wsl + s * D;
      for (int d = 0; d < D; ++d) acc = fmaf(xr[d], wr[d], acc);
      const float noise = -logf(-logf(lrow[s] + 1e-8f) + 1e-8f);
      const float z = (round_to(w_out, acc + bsl[s]) + noise) / temp;
      lrow[s] = z;
      mx = fmaxf(mx, z);
    }
    float sum = 0.f;
    for (int s = 0; s < S; ++s) {
      const float e = expf(lrow[s] - mx);
      lrow[s] = e;
      sum += e;
    }
    const float inv = 1.f / sum;
    for (int s = 0; s < S; ++s) lrow[s] *= inv;
  }
  __syncthreads();
  for (int i = t; i < rows * HS; i += 256) {
    const int pair = i / S, s = i - pair * S;
    store_from_f32(w_out + m0 * HS + i, lg[pair * (S + 1) + s]);
  }
}

// ------------------------------------------------------------------------------------------------
// softmax_rows_plus_kernel: the row stage of the Transolver++ slice weights when the two Linears over the
// (point, head) rows -- the slice logits and the hidden layer gelu(b1 + W1 x_mid) of proj_temperature -- were formed by
// the row GEMM kernels (logits in `w`, hidden in `hidden`, both (rows, S)).  L lanes share a row:
//   temp = max(temperature[h] + gelu(b2 + sum_s w2[s] hidden[s]), 0.01);  w <- softmax_s((w + noise(u)) / temp) in place
// ------------------------------------------------------------------------------------------------
template <typename T, int L>
__global__ __launch_bounds__(256) void softmax_rows_plus_kernel(T *__restrict__ w, const T *__restrict__ hidden,
                                                                const T *__restrict__ uniform,
                                                                const float *__restrict__ temperature,
                                                                const float *__restrict__ pt_w2,
                                                                const float *__restrict__ pt_b2, int64_t rows, int S,
                                                                int H) {
  const int per_wg = 256 / L;
  const int sub = threadIdx.x / L, l = threadIdx.x % L;
  for (int64_t row = (int64_t)blockIdx.x * per_wg + sub; row < rows; row += (int64_t)gridDim.x * per_wg) {
    T *p = w + row * S;
    const T *hp = hidden + row * S, *up = uniform + row * S;
    float tacc = 0.f;
    for (int s = l; s < S; s += L) tacc = fmaf(pt_w2[s], load_as_f32(hp + s), tacc);
#pragma unroll
    for (int off = L >> 1; off > 0; off >>= 1) tacc += __shfl_xor(tacc, off, 64);
    const float temp = round_to(w, fmaxf(temperature[row % H] + gelu_erf(tacc + pt_b2[0]), 0.01f));
    const float inv_t = 1.f / temp;
    auto arg = [&](int s) {
      return (load_as_f32(p + s) - logf(-logf(load_as_f32(up + s) + 1e-8f) + 1e-8f)) * inv_t;
    };
    float mx = -INFINITY;
    for (int s = l; s < S; s += L) mx = fmaxf(mx, arg(s));
#pragma unroll
    for (int off = L >> 1; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
    float sum = 0.f;
    for (int s = l; s < S; s += L) sum += expf(arg(s) - mx);
#pragma unroll
    for (int off = L >> 1; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
    const float inv = 1.f / sum;
    for (int s = l; s < S; s += L) store_from_f32(p + s, expf(arg(s) - mx) * inv);
  }
}

// The same with 16-byte accesses, for rows that are a whole number of 16-byte units: LR lanes share a row (a power of
// two >= S / unit), a lane keeps its unit of softmax arguments in registers, so every element is read once and its
// Gumbel noise (two logarithms) is formed once.
template <typename T, int LR>
__global__ __launch_bounds__(256) void softmax_rows_plus_vec_kernel(T *__restrict__ w, const T *__restrict__ hidden,
                                                                    const T *__restrict__ uniform,
                                                                    const float *__restrict__ temperature,
                                                                    const float *__restrict__ pt_w2,
                                                                    const float *__restrict__ pt_b2, int64_t rows, int S,
                                                                    int H) {
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  constexpr int UE = 16 / sizeof(T);
  constexpr int per_wg = 256 / LR;
  const int sub = threadIdx.x / LR, l = threadIdx.x % LR;
  const bool mine = l * UE < S;
  float w2[UE];
#pragma unroll
  for (int j = 0; j < UE; ++j) w2[j] = mine ? pt_w2[l * UE + j] : 0.f;
  const float b2 = pt_b2[0];
  for (int64_t row = (int64_t)blockIdx.x * per_wg + sub; row < rows; row += (int64_t)gridDim.x * per_wg) {
    const int64_t off0 = row * S + l * UE;
    float v[UE];
    float tacc = 0.f;
    if (mine) {
      const u32x4 rw = *reinterpret_cast<const u32x4 *>(w + off0);
      const u32x4 rh = *reinterpret_cast<const u32x4 *>(hidden + off0);
      const u32x4 ru = *reinterpret_cast<const u32x4 *>(uniform + off0);
      const T *ew = reinterpret_cast<const T *>(&rw), *eh = reinterpret_cast<const T *>(&rh),
              *eu = reinterpret_cast<const T *>(&ru);
#pragma unroll
      for (int j = 0; j < UE; ++j) {
        tacc = fmaf(w2[j], load_as_f32(eh + j), tacc);
        v[j] = load_as_f32(ew + j) - logf(-logf(load_as_f32(eu + j) + 1e-8f) + 1e-8f);
      }
    }
#pragma unroll
    for (int off = LR >> 1; off > 0; off >>= 1) tacc += __shfl_xor(tacc, off, 64);
    const float temp = round_to(w, fmaxf(temperature[row % H] + gelu_erf(tacc + b2), 0.01f));
    const float inv_t = 1.f / temp;
    float mx = -INFINITY;
    if (mine) {
#pragma unroll
      for (int j = 0; j < UE; ++j) {
        v[j] *= inv_t;
        mx = fmaxf(mx, v[j]);
      }
    }
#pragma unroll
    for (int off = LR >> 1; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
    float sum = 0.f;
    if (mine) {
#pragma unroll
      for (int j = 0; j < UE; ++j) {
        v[j] = expf(v[j] - mx);
        sum += v[j];
      }
    }
#pragma unroll
    for (int off = LR >> 1; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
    if (mine) {
      const float inv = 1.f / sum;
      alignas(16) T o[UE];
#pragma unroll
      for (int j = 0; j < UE; ++j) store_from_f32(o + j, v[j] * inv);
      *reinterpret_cast<u32x4 *>(w + off0) = *reinterpret_cast<const u32x4 *>(o);
    }
  }
}

// ------------------------------------------------------------------------------------------------
// slice_partial_kernel: grid (G chunks, B*H, output slabs).  For its chunk of points of one (b, h):
//   partial[s, d] = sum_n w[n, s] * fx_mid[n, d]   (d < D),   partial[s, D] = sum_n w[n, s]
// The (S x D+1) output is cut into 4 x 4 register tiles; a thread owns NS of them (tile t + 256 i of its slab of
// 256 NS tiles) and walks the chunk 64 points at a time through LDS: per point and tile two 16-byte LDS reads
// (4 slice weights, 4 features) feed 16 FMAs.  Up to 256 tiles several groups of threads take every so many points, their
// sums added up through LDS: S = 32, D = 16 has 40 tiles, 4 x 7 225 points of 8 heads 18 us in six groups, 36 with 216 of
// 256 threads waiting; S = 64, D = 32 (144 tiles, 65 536 points in bf16) 37 us in three groups of 512 threads, 41 before.
// LDS rows are padded to multiples of four (zeros; column D of the
// feature rows holds 1 for the count).  Sums run in a fixed order, so the result is bit-reproducible.
// ------------------------------------------------------------------------------------------------
constexpr int kAttnThreads = 1024;  // slice_combine_attn_kernel: 16 waves, one query row per wave at a time
constexpr int kPartialTile = 64;
constexpr int kPartialMaxNS = 4;

// threads of a workgroup and the groups of them that share a chunk's points (up to 256 tiles)
__host__ __device__ inline int partial_threads(int n_tiles) { return n_tiles > 128 ? 512 : 256; }
__host__ __device__ inline int partial_groups(int n_tiles) {
  const int g = partial_threads(n_tiles) / n_tiles;
  return g > 32 ? 32 : g;
}

template <typename T, int NS>
__global__ __launch_bounds__(NS == 1 ? 512 : 256) void slice_partial_kernel(const T *__restrict__ w, const T *__restrict__ fx_mid,
                                                            float *__restrict__ partials, int B, int64_t N, int H, int D,
                                                            int S, int64_t chunk) {
  extern __shared__ float4 lds4[];
  const int D1 = D + 1, SB = (S + 3) / 4, DB = (D1 + 3) / 4;  // tiles along the slices / the features
  float4 *wl = lds4;                      // kPartialTile * SB
  float4 *fl = wl + kPartialTile * SB;    // kPartialTile * DB
  float *wlf = reinterpret_cast<float *>(wl), *flf = reinterpret_cast<float *>(fl);
  const int t = threadIdx.x;
  const int g = blockIdx.x;
  const int b = blockIdx.y / H, h = blockIdx.y % H;
  const int n_tiles = SB * DB;
  const int slab0 = blockIdx.z * 256 * NS;
  const int threads = NS == 1 ? blockDim.x : 256;
  const int groups = NS == 1 ? partial_groups(n_tiles) : 1, tile0 = NS == 1 ? t % n_tiles : t, group = NS == 1 ? t / n_tiles : 0;
  int sb[NS], db[NS];
  float acc[NS][4][4];
#pragma unroll
  for (int i = 0; i < NS; ++i) {
    const int tile = slab0 + tile0 + 256 * i;
    const bool ok = tile < n_tiles;
    sb[i] = ok ? tile % SB : 0;
    db[i] = ok ? tile / SB : 0;
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[i][u][v] = 0.f;
  }
  const int64_t n_begin = (int64_t)g * chunk;
  const int64_t n_end = min(N, n_begin + chunk);
  const int HS = H * S, HD = H * D;
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  constexpr int UE = 16 / sizeof(T);
  const bool vec_w = S % UE == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0;
  const bool vec_f = D % UE == 0 && reinterpret_cast<uintptr_t>(fx_mid) % 16 == 0;
  for (int64_t n0 = n_begin; n0 < n_end; n0 += kPartialTile) {
    const int pts = (int)min((int64_t)kPartialTile, n_end - n0);
    if (vec_w) {  // 16-byte loads: the rows are whole numbers of 16-byte units
      const int units = S / UE;
      for (int i = t; i < kPartialTile * units; i += threads) {
        const int p = i / units, u = i - p * units;
        u32x4 raw = {0u, 0u, 0u, 0u};
        if (p < pts) raw = *reinterpret_cast<const u32x4 *>(w + ((int64_t)b * N + n0 + p) * HS + h * S + u * UE);
        const T *e = reinterpret_cast<const T *>(&raw);
#pragma unroll
        for (int j = 0; j < UE; ++j) wlf[p * (SB * 4) + u * UE + j] = load_as_f32(e + j);
      }
    } else {
      for (int i = t; i < kPartialTile * SB * 4; i += threads) {
        const int p = i / (SB * 4), s = i - p * (SB * 4);
        wlf[i] = (p < pts && s < S) ? load_as_f32(w + ((int64_t)b * N + n0 + p) * HS + h * S + s) : 0.f;
      }
    }
    if (vec_f) {
      const int units = D / UE;
      for (int i = t; i < kPartialTile * units; i += threads) {
        const int p = i / units, u = i - p * units;
        u32x4 raw = {0u, 0u, 0u, 0u};
        if (p < pts) raw = *reinterpret_cast<const u32x4 *>(fx_mid + ((int64_t)b * N + n0 + p) * HD + h * D + u * UE);
        const T *e = reinterpret_cast<const T *>(&raw);
#pragma unroll
        for (int j = 0; j < UE; ++j) flf[p * (DB * 4) + u * UE + j] = load_as_f32(e + j);
      }
      for (int i = t; i < kPartialTile * (DB * 4 - D); i += threads) {  // the count column and the padding behind it
        const int p = i / (DB * 4 - D), d = D + i - p * (DB * 4 - D);
        flf[p * (DB * 4) + d] = (p < pts && d == D) ? 1.f : 0.f;
      }
    } else {
      for (int i = t; i < kPartialTile * DB * 4; i += threads) {
        const int p = i / (DB * 4), d = i - p * (DB * 4);
        float v = 0.f;
        if (p < pts && d < D) v = load_as_f32(fx_mid + ((int64_t)b * N + n0 + p) * HD + h * D + d);
        if (p < pts && d == D) v = 1.f;
        flf[i] = v;
      }
    }
    __syncthreads();
#pragma unroll 2
    for (int p = group; p < kPartialTile; p += groups) {
#pragma unroll
      for (int i = 0; i < NS; ++i) {
        const float4 wv = wl[p * SB + sb[i]];
        const float4 fv = fl[p * DB + db[i]];
        const float ws[4] = {wv.x, wv.y, wv.z, wv.w}, fs[4] = {fv.x, fv.y, fv.z, fv.w};
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int v = 0; v < 4; ++v) acc[i][u][v] = fmaf(ws[u], fs[v], acc[i][u][v]);
      }
    }
    __syncthreads();
  }
  if (groups > 1) {  // the groups' sums added up in order
    float4 *part = lds4 + ((group - 1) * n_tiles + tile0) * 4;
    if (group > 0 && group < groups) {
#pragma unroll
      for (int u = 0; u < 4; ++u) part[u] = float4{acc[0][u][0], acc[0][u][1], acc[0][u][2], acc[0][u][3]};
    }
    __syncthreads();
    if (group > 0) return;
    for (int q = 1; q < groups; ++q) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float4 v = lds4[((q - 1) * n_tiles + tile0) * 4 + u];
        acc[0][u][0] += v.x, acc[0][u][1] += v.y, acc[0][u][2] += v.z, acc[0][u][3] += v.w;
      }
    }
  }
  float *dst = partials + (((int64_t)g * B + b) * H + h) * (S * D1);
#pragma unroll
  for (int i = 0; i < NS; ++i) {
    if (slab0 + tile0 + 256 * i >= n_tiles) continue;
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int s = 4 * sb[i] + u, d = 4 * db[i] + v;
        if (s < S && d < D1) dst[s * D1 + d] = acc[i][u][v];
      }
  }
}

// ------------------------------------------------------------------------------------------------
// combine_partials_kernel: second pass of the reduction, parallel over outputs.  grid (ceil(n_out/64), B*H);
// 64 outputs x 4 quarter-ranges of the G partials per workgroup; each thread adds its quarter in SUMS sums, every SUMS-th
// partial in index order, (a0 + a1) + (a2 + a3); the four quarter sums are then added in a fixed order
// ((q0 + q1) + q2) + q3: bit-reproducible, no atomics.
// Bound by the latency of the partials, which other XCDs wrote: 16 of a thread's loads are in flight at once.  256 partials
// of 8 x 2 112 floats 5.1 us; one load at a time 17.5.
// ------------------------------------------------------------------------------------------------
template <int SUMS>
__global__ __launch_bounds__(256) void combine_partials_kernel(const float *__restrict__ partials, int G,
                                                               int64_t partial_stride, float *__restrict__ combined,
                                                               int n_out) {
  constexpr int kAhead = 16;
  __shared__ float quarter[4][64];
  const int t = threadIdx.x, q = t >> 6, l = t & 63;
  const int o = blockIdx.x * 64 + l;
  const int bh = blockIdx.y;
  const int per = (G + 3) / 4;
  const int g0 = q * per, g1 = min(G, g0 + per);
  float acc[SUMS] = {};
  if (o < n_out) {
    const float *src = partials + (int64_t)bh * n_out + o;
    for (int g = g0; g < g1; g += kAhead) {  // kAhead loads in flight
      float v[kAhead];
#pragma unroll
      for (int u = 0; u < kAhead; ++u) v[u] = src[(int64_t)min(g + u, g1 - 1) * partial_stride];
#pragma unroll
      for (int u = 0; u < kAhead; ++u) acc[u % SUMS] += g + u < g1 ? v[u] : 0.f;
    }
  }
  if constexpr (SUMS == 4) quarter[q][l] = (acc[0] + acc[1]) + (acc[2] + acc[3]);
  else quarter[q][l] = acc[0];
  __syncthreads();
  if (q == 0 && o < n_out)
    combined[(int64_t)bh * n_out + o] = ((quarter[0][l] + quarter[1][l]) + quarter[2][l]) + quarter[3][l];
}

// ------------------------------------------------------------------------------------------------
// slice_combine_attn_kernel: one workgroup per (b, h), everything after the load stays in LDS.
//   1. num[s, :], cnt[s] = sum over the G partials in index order
//   2. tok = num / (cnt + 1e-2)            -> slice_token, slice_norm (optional outputs)
//   3. q|k|v = tok Wqkv^T                  (rows of Wqkv: [0,D) q, [D,2D) k, [2D,3D) v)
//   4. out[s, :] = softmax_t(q[s].k[t] / sqrt(D)) v[t, :], one wave per query row
// `partial_stride` = elements between consecutive partials of the same (b, h).  G == 0: `partials` holds
// finished tokens (steps 1-2 skipped); out_token == nullptr: stop after step 2.
// ------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(kAttnThreads) void slice_combine_attn_kernel(const float *__restrict__ partials, int G,
                                                                 int64_t partial_stride, const float *__restrict__ w_qkv,
                                                                 float *__restrict__ slice_token,
                                                                 float *__restrict__ slice_norm,
                                                                 float *__restrict__ out_token, int D, int S,
                                                                 int stage_w) {
  extern __shared__ float lds[];
  const int D1 = D + 1;
  float *tok = lds;              // S * D1 (column D holds the count, then the norm)
  float *q = tok + S * D1;       // S * D1
  float *k = q + S * D1;
  float *v = k + S * D1;
  float *prow = v + S * D1;      // one row of S per wave
  float *wq = prow + (kAttnThreads / 64) * S;      // 3D * D1 (only when stage_w)
  const int t = threadIdx.x;
  const int bh = blockIdx.x;
  const int n_out = S * D1;
  if (G > 0) {
    const float *src = partials + (int64_t)bh * n_out;
    for (int o = t; o < n_out; o += kAttnThreads) {
      float acc = 0.f;
      for (int g = 0; g < G; ++g) acc += src[(int64_t)g * partial_stride + o];
      tok[o] = acc;
    }
    __syncthreads();
    for (int s = t; s < S; s += kAttnThreads) tok[s * D1 + D] += kSliceNormEps;
    __syncthreads();
    for (int i = t; i < S * D; i += kAttnThreads) {
      const int s = i / D, d = i - s * D;
      const float val = tok[s * D1 + d] / tok[s * D1 + D];
      tok[s * D1 + d] = val;
      if (slice_token) slice_token[(int64_t)bh * S * D + i] = val;
    }
    if (slice_norm)
      for (int s = t; s < S; s += kAttnThreads) slice_norm[(int64_t)bh * S + s] = tok[s * D1 + D];
  } else {
    // G == 0: `partials` already holds finished slice tokens (B, H, S, D)
    for (int i = t; i < S * D; i += kAttnThreads) tok[(i / D) * D1 + (i % D)] = partials[(int64_t)bh * S * D + i];
  }
  if (!out_token) return;  // reduction-only call (uniform across the workgroup)
  if (stage_w)
    for (int i = t; i < 3 * D * D; i += kAttnThreads) wq[(i / D) * D1 + (i % D)] = w_qkv[i];
  __syncthreads();
  for (int i = t; i < S * 3 * D; i += kAttnThreads) {
    const int s = i / (3 * D), e = i - s * 3 * D;
    const float *wr = stage_w ? wq + e * D1 : w_qkv + (int64_t)e * D;
    const float *tr = tok + s * D1;
    float acc = 0.f;
#pragma unroll 8
    for (int d = 0; d < D; ++d) acc = fmaf(tr[d], wr[d], acc);
    float *dst = e < D ? q : (e < 2 * D ? k : v);
    dst[s * D1 + (e % D)] = acc;
  }
  __syncthreads();
  const int wave = t >> 6, lane = t & 63;
  const float scale = rsqrtf((float)D);
  float *pr = prow + wave * S;
  for (int s = wave; s < S; s += kAttnThreads / 64) {
    const float *qs = q + s * D1;
    float mx = -INFINITY;
    for (int u = lane; u < S; u += 64) {
      const float *ku = k + u * D1;
      float acc = 0.f;
#pragma unroll 8
      for (int e = 0; e < D; ++e) acc = fmaf(qs[e], ku[e], acc);
      acc *= scale;
      pr[u] = acc;
      mx = fmaxf(mx, acc);
    }
    mx = wave_max(mx);
    float sum = 0.f;
    for (int u = lane; u < S; u += 64) {
      const float e = expf(pr[u] - mx);
      pr[u] = e;
      sum += e;
    }
    sum = wave_sum(sum);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const float inv = 1.f / sum;
    for (int e = lane; e < D; e += 64) {
      float acc = 0.f;
#pragma unroll 8
      for (int u = 0; u < S; ++u) acc = fmaf(pr[u], v[u * D1 + e], acc);
      out_token[((int64_t)bh * S + s) * D + e] = acc * inv;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

// ------------------------------------------------------------------------------------------------
// narrow_combine_attn_kernel<D>: combine_partials_kernel and slice_combine_attn_kernel in one launch for narrow heads, with
// their sums in their order, bit for bit: 32 threads per slice, everything of a (b, h) in registers and LDS, sizes known to
// the compiler.  Bound by latency: one trip for partials and weights, four barriers.  D = 16, S = 32 (us, the two launches before ->
// now): 16 workgroups of 97 partials 4.5 + 11.0 -> 7.5, of 63 partials 5.9 (with one sum at a time instead of four neighbouring ones
// 9.5 and 6.5).
// ------------------------------------------------------------------------------------------------
constexpr int kNarrowSlices = 32;

template <int D>
__global__ __launch_bounds__(32 * kNarrowSlices) void narrow_combine_attn_kernel(const float *__restrict__ partials, int G,
                                                                    int64_t partial_stride, const float *__restrict__ w_qkv,
                                                                    float *__restrict__ slice_token,
                                                                    float *__restrict__ slice_norm,
                                                                    float *__restrict__ out_token) {
  constexpr int S = kNarrowSlices, T = 32 * S, D1 = D + 1, LD = D + 4, NOUT = S * D1, NQ = NOUT / 4, kParts = 4, kAhead = 16;
  static_assert(S == 2 * 16 && D % 4 == 0, "16 threads per slice in the softmax, two keys each; whole float4 rows");
  __shared__ __align__(16) float part[kParts][NOUT];
  __shared__ __align__(16) float tok[S * LD], wq[3 * D * LD], qkv[3][S * LD], prob[S * (S + 1)];
  const int t = threadIdx.x, bh = blockIdx.x;
  float w[(3 * D * D + T - 1) / T];
#pragma unroll
  for (int k = 0; k < (3 * D * D + T - 1) / T; ++k) w[k] = k * T + t < 3 * D * D ? w_qkv[k * T + t] : 0.f;
  // a thread adds up four neighbouring sums of a quarter of the partials in index order, kAhead of them in flight: one trip for 64
  const int per = (G + kParts - 1) / kParts, pt = t / NQ, o4 = t - pt * NQ, g0 = pt * per, g1 = min(G, g0 + per);
  if (pt < kParts) {
    const float4 *src = reinterpret_cast<const float4 *>(partials + (int64_t)bh * NOUT) + o4;  // NOUT and the stride: whole float4
    float4 acc{0.f, 0.f, 0.f, 0.f};
    for (int g = g0; g < g1; g += kAhead) {
      float4 v[kAhead];
#pragma unroll
      for (int u = 0; u < kAhead; ++u) v[u] = src[(int64_t)min(g + u, g1 - 1) * (partial_stride / 4)];
#pragma unroll
      for (int u = 0; u < kAhead; ++u)
        if (g + u < g1) acc.x += v[u].x, acc.y += v[u].y, acc.z += v[u].z, acc.w += v[u].w;
    }
    reinterpret_cast<float4 *>(part[pt])[o4] = acc;
  }
#pragma unroll
  for (int k = 0; k < (3 * D * D + T - 1) / T; ++k) {
    const int i = k * T + t;
    if (i < 3 * D * D) wq[(i / D) * LD + i % D] = w[k];
  }
  __syncthreads();
  auto total = [&](int o) { return ((part[0][o] + part[1][o]) + part[2][o]) + part[3][o]; };
  for (int i = t; i < S * D; i += T) {
    const int s = i / D, d = i % D;
    const float cnt = total(s * D1 + D) + kSliceNormEps, val = total(s * D1 + d) / cnt;
    tok[s * LD + d] = val;
    if (slice_token) slice_token[(int64_t)bh * S * D + i] = val;
    if (slice_norm && d == 0) slice_norm[(int64_t)bh * S + s] = cnt;
  }
  __syncthreads();
  auto dot = [](const float *a, const float *b) {  // in index order
    float acc = 0.f;
#pragma unroll
    for (int k = 0; k < D; k += 4) {
      const float4 x = *reinterpret_cast<const float4 *>(a + k), y = *reinterpret_cast<const float4 *>(b + k);
      acc = fmaf(x.w, y.w, fmaf(x.z, y.z, fmaf(x.y, y.y, fmaf(x.x, y.x, acc))));
    }
    return acc;
  };
#pragma unroll
  for (int i = t; i < S * 3 * D; i += T) {
    const int s = i % S, e = i / S;
    qkv[e / D][s * LD + e % D] = dot(tok + s * LD, wq + e * LD);
  }
  __syncthreads();
  // The first half of the workgroup: slice s = t / 16, keys t % 16 and t % 16 + 16.  A sum over a slice's keys pairs them as a sum over the
  // 64 lanes of a wave does.
  const int s = t >> 4, l = t & 15;
  float inv = 0.f;
  if (s < S) {
    const float scale = rsqrtf((float)D);
    float e[2], mx = -INFINITY;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      e[j] = dot(qkv[0] + s * LD, qkv[1] + (l + 16 * j) * LD) * scale;
      asm("" : "+v"(e[j]));  // rounded, as the kernel that stores it has it: no fused multiply-subtract below
      mx = fmaxf(mx, e[j]);
    }
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      e[j] = expf(e[j] - mx);
      prob[s * (S + 1) + l + 16 * j] = e[j];
    }
    float sum = e[0] + e[1];
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
    inv = 1.f / sum;
  }
  __syncthreads();
  if (s < S) {
    for (int d = l; d < D; d += 16) {
      float acc = 0.f;
#pragma unroll
      for (int u = 0; u < S; ++u) acc = fmaf(prob[s * (S + 1) + u], qkv[2][u * LD + d], acc);
      out_token[((int64_t)bh * S + s) * D + d] = acc * inv;
    }
  }
}

// ------------------------------------------------------------------------------------------------
// deslice_kernel: grid (row tiles of R, B-independent; H).  out_x[m, h*D + d] = sum_s w[m, h, s] * tok'[b, h, s, d]
// A row tile never straddles two batches (the host picks tiles per batch).
// ------------------------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void deslice_kernel(const T *__restrict__ w, const float *__restrict__ out_token,
                                                      T *__restrict__ out_x, int64_t N, int H, int D, int S, int R,
                                                      int tiles_per_batch) {
  extern __shared__ float lds[];
  float *tk = lds;            // S * D
  float *wl = tk + S * D;     // R * (S+1)
  const int t = threadIdx.x;
  const int h = blockIdx.y;
  const int b = blockIdx.x / tiles_per_batch;
  const int64_t n0 = (int64_t)(blockIdx.x % tiles_per_batch) * R;
  const int rows = (int)min((int64_t)R, N - n0);
  const int64_t m0 = (int64_t)b * N + n0;
  for (int i = t; i < S * D; i += 256) tk[i] = out_token[((int64_t)b * H + h) * S * D + i];
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
  constexpr int UE = 16 / sizeof(T);
  if (S % UE == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0) {  // 16-byte loads of the slice weights
    const int units = S / UE;
    for (int i = t; i < R * units; i += 256) {  // rows past the end of the batch: zeros
      const int r = i / units, u = i - r * units;
      u32x4 raw = {0u, 0u, 0u, 0u};
      if (r < rows) raw = *reinterpret_cast<const u32x4 *>(w + (m0 + r) * H * S + h * S + u * UE);
      const T *e = reinterpret_cast<const T *>(&raw);
#pragma unroll
      for (int j = 0; j < UE; ++j) wl[r * (S + 1) + u * UE + j] = load_as_f32(e + j);
    }
  } else {
    for (int i = t; i < R * S; i += 256) {
      const int r = i / S, s = i - r * S;
      wl[r * (S + 1) + s] = r < rows ? load_as_f32(w + (m0 + r) * H * S + h * S + s) : 0.f;
    }
  }
  __syncthreads();
  if (D % 4 == 0 && reinterpret_cast<uintptr_t>(out_x) % 16 == 0) {
    // a thread owns 4 rows x 4 adjacent features: one 16-byte and four 4-byte LDS reads per 16 multiply-adds, and the
    // results leave as 8- or 16-byte stores
    const int DQ4 = D >> 2, S1 = S + 1;
    for (int tile = t; tile < (R >> 2) * DQ4; tile += 256) {
      const int rq = tile / DQ4, dq = tile - rq * DQ4, r0 = 4 * rq;
      if (r0 >= rows) continue;
      const float *w0 = wl + r0 * S1;
      float acc[4][4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int k = 0; k < 4; ++k) acc[j][k] = 0.f;
      for (int sl = 0; sl < S; ++sl) {
        const float4 tv = *reinterpret_cast<const float4 *>(tk + sl * D + 4 * dq);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float wv = w0[j * S1 + sl];
          acc[j][0] = fmaf(wv, tv.x, acc[j][0]);
          acc[j][1] = fmaf(wv, tv.y, acc[j][1]);
          acc[j][2] = fmaf(wv, tv.z, acc[j][2]);
          acc[j][3] = fmaf(wv, tv.w, acc[j][3]);
        }
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (r0 + j >= rows) continue;
        alignas(16) T o4[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) store_from_f32(o4 + k, acc[j][k]);
        T *dst = out_x + (m0 + r0 + j) * H * D + h * D + 4 * dq;
        if constexpr (sizeof(T) == 2) *reinterpret_cast<u32x2 *>(dst) = *reinterpret_cast<const u32x2 *>(o4);
        else *reinterpret_cast<u32x4 *>(dst) = *reinterpret_cast<const u32x4 *>(o4);
      }
    }
    return;
  }
  // a thread owns 4 rows x 2 features (features dq and dq + DQ): 6 LDS reads per 8 multiply-adds
  const int DQ = (D + 1) >> 1, S1 = S + 1;
  for (int tile = t; tile < (R >> 2) * DQ; tile += 256) {
    const int rq = tile / DQ, dq = tile - rq * DQ, r0 = 4 * rq;
    if (r0 >= rows) continue;
    const int d1 = min(dq + DQ, D - 1);
    const float *w0 = wl + r0 * S1;
    float acc[4][2] = {{0.f, 0.f}, {0.f, 0.f}, {0.f, 0.f}, {0.f, 0.f}};
    for (int sl = 0; sl < S; ++sl) {
      const float t0 = tk[sl * D + dq], t1 = tk[sl * D + d1];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float wv = w0[j * S1 + sl];
        acc[j][0] = fmaf(wv, t0, acc[j][0]);
        acc[j][1] = fmaf(wv, t1, acc[j][1]);
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (r0 + j >= rows) continue;
      T *o = out_x + (m0 + r0 + j) * H * D + h * D;
      store_from_f32(o + dq, acc[j][0]);
      if (dq + DQ < D) store_from_f32(o + dq + DQ, acc[j][1]);
    }
  }
}

// ------------------------------------------------------------------------------------------------
// residual_ln_kernel: one wave per row.  y <- y + residual (rounded to the storage type);
// ln_out = (y - mean) / sqrt(var + eps) * gamma + beta with the biased variance, all statistics in fp32.
// ------------------------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void residual_ln_kernel(T *__restrict__ y, const T *__restrict__ residual,
                                                          const float *__restrict__ gamma, const float *__restrict__ beta,
                                                          float eps, T *__restrict__ ln_out, int64_t M, int C) {
  const int lane = threadIdx.x & 63;
  const int64_t m = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (m >= M) return;
  T *yr = y + m * C;
  float sum = 0.f;
  for (int c = lane; c < C; c += 64) {
    float v = load_as_f32(yr + c);
    if (residual) {
      v = round_to(yr, v + load_as_f32(residual + m * C + c));
      store_from_f32(yr + c, v);
    }
    sum += v;
  }
  if (!ln_out) return;
  const float mean = wave_sum(sum) / (float)C;
  float sq = 0.f;
  for (int c = lane; c < C; c += 64) {
    const float dlt = load_as_f32(yr + c) - mean;
    sq = fmaf(dlt, dlt, sq);
  }
  const float rstd = rsqrtf(wave_sum(sq) / (float)C + eps);
  for (int c = lane; c < C; c += 64) {
    const float v = (load_as_f32(yr + c) - mean) * rstd;
    store_from_f32(ln_out + m * C + c, v * gamma[c] + beta[c]);
  }
}

// Rows of whole 16-byte units (C % UE == 0): LPR lanes share a row, the smallest power of two that gives every unit a lane
// (all 64 with UPL units each for rows beyond 64 units), so a wave works on 64 / LPR rows at once, every lane of an access
// carries data, and the row sums are exchanges inside the group.  The next rows are fetched while these are worked on.
template <int LPR>
__device__ __forceinline__ float group_sum(float v) {
#pragma unroll
  for (int off = LPR / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

template <typename T>
struct RowUnit {
  static constexpr int UE = 16 / sizeof(T);
  typedef uint32_t vec __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ void unpack(vec v, float (&f)[UE]) {
    if constexpr (sizeof(T) == 4) {
#pragma unroll
      for (int e = 0; e < UE; ++e) {
        const uint32_t w = v[e];
        f[e] = __uint_as_float(w);
      }
    } else {
#pragma unroll
      for (int e = 0; e < UE; ++e) {
        const uint32_t w = v[e >> 1];
        f[e] = __uint_as_float((e & 1) ? (w & 0xffff0000u) : (w << 16));
      }
    }
  }
  static __device__ __forceinline__ vec pack(const float (&f)[UE]) {
    vec v;
    if constexpr (sizeof(T) == 4) {
#pragma unroll
      for (int e = 0; e < UE; ++e) v[e] = __float_as_uint(f[e]);
    } else {
#pragma unroll
      for (int w = 0; w < 4; ++w)
        v[w] = (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)f[2 * w]) |
               ((uint32_t)__builtin_bit_cast(uint16_t, (__bf16)f[2 * w + 1]) << 16);
    }
    return v;
  }
};

// residual_ln_rows_kernel: y <- y + residual (if given), ln_out = LayerNorm(y) (if given).  Bound by HBM: 262 144 bf16
// rows of 256 channels without a residual 56 us = 4.8 TB/s (one row per wave with half of its lanes idle: 88 us).
template <typename T, int LPR, int UPL>
__global__ __launch_bounds__(256) void residual_ln_rows_kernel(T *__restrict__ y, const T *__restrict__ residual,
                                                               const float *__restrict__ gamma,
                                                               const float *__restrict__ beta, float eps,
                                                               T *__restrict__ ln_out, int64_t M, int C) {
  using U = RowUnit<T>;
  using vec = typename U::vec;
  constexpr int UE = U::UE, RPW = 64 / LPR;
  const int lane = threadIdx.x & 63, l = lane % LPR, sub = lane / LPR, units = C / UE;
  float gam[UPL][UE], bet[UPL][UE];
#pragma unroll
  for (int k = 0; k < UPL; ++k)
#pragma unroll
    for (int e = 0; e < UE; ++e) {
      const int c = (l + LPR * k) * UE + e;
      gam[k][e] = (ln_out && c < C) ? gamma[c] : 1.f;
      bet[k][e] = (ln_out && c < C) ? beta[c] : 0.f;
    }
  const float inv_c = 1.f / (float)C;
  const int64_t step = (int64_t)gridDim.x * 4 * RPW;
  int64_t mw = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * RPW;  // the wave's first row
  auto fetch = [&](int64_t m, vec(&a)[UPL], vec(&r)[UPL]) {
#pragma unroll
    for (int k = 0; k < UPL; ++k) {
      a[k] = r[k] = vec{0, 0, 0, 0};
      if (m < M && l + LPR * k < units) {
        a[k] = *reinterpret_cast<const vec *>(y + m * C + (l + LPR * k) * UE);
        if (residual) r[k] = *reinterpret_cast<const vec *>(residual + m * C + (l + LPR * k) * UE);
      }
    }
  };
  vec a[UPL], r[UPL];
  if (mw < M) fetch(mw + sub, a, r);
  for (; mw < M; mw += step) {
    const int64_t m = mw + sub;
    vec an[UPL], rn[UPL];
    fetch(m + step, an, rn);
    float v[UPL][UE], sum = 0.f;
#pragma unroll
    for (int k = 0; k < UPL; ++k) {
      U::unpack(a[k], v[k]);
      if (residual) {
        float rv[UE];
        U::unpack(r[k], rv);
#pragma unroll
        for (int e = 0; e < UE; ++e) v[k][e] += rv[e];
        const vec o = U::pack(v[k]);
        U::unpack(o, v[k]);  // the sum as it is stored
        if (m < M && l + LPR * k < units) *reinterpret_cast<vec *>(y + m * C + (l + LPR * k) * UE) = o;
      }
#pragma unroll
      for (int e = 0; e < UE; ++e) sum += v[k][e];
    }
    if (ln_out) {
      const float mean = group_sum<LPR>(sum) * inv_c;
      float sq = 0.f;
#pragma unroll
      for (int k = 0; k < UPL; ++k)
        if (l + LPR * k < units) {
#pragma unroll
          for (int e = 0; e < UE; ++e) {
            const float d = v[k][e] - mean;
            sq = fmaf(d, d, sq);
          }
        }
      const float rstd = rsqrtf(group_sum<LPR>(sq) * inv_c + eps);
#pragma unroll
      for (int k = 0; k < UPL; ++k) {
#pragma unroll
        for (int e = 0; e < UE; ++e) v[k][e] = (v[k][e] - mean) * rstd * gam[k][e] + bet[k][e];
        if (m < M && l + LPR * k < units) *reinterpret_cast<vec *>(ln_out + m * C + (l + LPR * k) * UE) = U::pack(v[k]);
      }
    }
#pragma unroll
    for (int k = 0; k < UPL; ++k) {
      a[k] = an[k];
      r[k] = rn[k];
    }
  }
}

// layernorm_backward_rows_kernel: backward of y = (x - mean) rstd gamma + beta.
//   xh = (x - mean) rstd;  g = dy gamma;  dx = [add +] rstd (g - mean_c(g) - xh mean_c(g xh));  d gamma = sum_rows dy xh;
//   d beta = sum_rows dy (statistics recomputed from x; `add`: the gradient that reaches x past the LayerNorm).
// Every lane sums d gamma / d beta of its columns over the rows it walks, the groups and waves of a workgroup add up in
// order through LDS, each workgroup leaves one partial [2][C].  Bound by HBM: 262 144 bf16 rows of 256 channels 73 us =
// 5.5 TB/s (one row per wave: 128 us).
template <typename T, int LPR, int UPL>
__global__ __launch_bounds__(256) void layernorm_backward_rows_kernel(const T *__restrict__ x, const T *__restrict__ dy,
                                                                      const T *__restrict__ add,
                                                                      const float *__restrict__ gamma, float eps,
                                                                      T *__restrict__ dx, float *__restrict__ partials,
                                                                      int64_t M, int C) {
  using U = RowUnit<T>;
  using vec = typename U::vec;
  constexpr int UE = U::UE, RPW = 64 / LPR;
  extern __shared__ float red[];  // [4 waves][2][C]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l = lane % LPR, sub = lane / LPR, units = C / UE;
  float gam[UPL][UE], dg[UPL][UE], db[UPL][UE];
#pragma unroll
  for (int k = 0; k < UPL; ++k)
#pragma unroll
    for (int e = 0; e < UE; ++e) {
      const int c = (l + LPR * k) * UE + e;
      gam[k][e] = c < C ? gamma[c] : 0.f;
      dg[k][e] = db[k][e] = 0.f;
    }
  const float inv_c = 1.f / (float)C;
  const int64_t step = (int64_t)gridDim.x * 4 * RPW;
  int64_t mw = ((int64_t)blockIdx.x * 4 + wave) * RPW;
  auto fetch = [&](int64_t m, vec(&a)[UPL], vec(&d)[UPL], vec(&p)[UPL]) {
#pragma unroll
    for (int k = 0; k < UPL; ++k) {
      a[k] = d[k] = p[k] = vec{0, 0, 0, 0};
      if (m < M && l + LPR * k < units) {
        const int64_t at = m * C + (l + LPR * k) * UE;
        a[k] = *reinterpret_cast<const vec *>(x + at);
        d[k] = *reinterpret_cast<const vec *>(dy + at);
        if (add) p[k] = *reinterpret_cast<const vec *>(add + at);
      }
    }
  };
  vec a[UPL], d[UPL], p[UPL];
  if (mw < M) fetch(mw + sub, a, d, p);
  for (; mw < M; mw += step) {
    const int64_t m = mw + sub;
    vec an[UPL], dn[UPL], pn[UPL];
    fetch(m + step, an, dn, pn);
    float xv[UPL][UE], gv[UPL][UE], sum = 0.f;
#pragma unroll
    for (int k = 0; k < UPL; ++k) {
      U::unpack(a[k], xv[k]);
      U::unpack(d[k], gv[k]);
#pragma unroll
      for (int e = 0; e < UE; ++e) sum += xv[k][e];
    }
    const float mean = group_sum<LPR>(sum) * inv_c;
    float sq = 0.f;
#pragma unroll
    for (int k = 0; k < UPL; ++k)
      if (l + LPR * k < units) {
#pragma unroll
        for (int e = 0; e < UE; ++e) {
          const float dlt = xv[k][e] - mean;
          sq = fmaf(dlt, dlt, sq);
        }
      }
    // rows beyond M hold zeros throughout; with eps = 0 their statistics alone would be infinite
    const float rstd = m < M ? rsqrtf(group_sum<LPR>(sq) * inv_c + eps) : 0.f;
    float s1 = 0.f, s2 = 0.f;
#pragma unroll
    for (int k = 0; k < UPL; ++k)
#pragma unroll
      for (int e = 0; e < UE; ++e) {  // lanes without a unit and rows beyond M hold dy = 0
        const float xh = (xv[k][e] - mean) * rstd, dyv = gv[k][e], gg = dyv * gam[k][e];
        dg[k][e] = fmaf(dyv, xh, dg[k][e]);
        db[k][e] += dyv;
        xv[k][e] = xh;
        gv[k][e] = gg;
        s1 += gg;
        s2 = fmaf(gg, xh, s2);
      }
    s1 = group_sum<LPR>(s1) * inv_c;
    s2 = group_sum<LPR>(s2) * inv_c;
#pragma unroll
    for (int k = 0; k < UPL; ++k) {
      float o[UE], pv[UE];
      U::unpack(p[k], pv);
#pragma unroll
      for (int e = 0; e < UE; ++e) o[e] = fmaf(rstd, gv[k][e] - s1 - xv[k][e] * s2, pv[e]);
      if (m < M && l + LPR * k < units) *reinterpret_cast<vec *>(dx + m * C + (l + LPR * k) * UE) = U::pack(o);
      a[k] = an[k];
      d[k] = dn[k];
      p[k] = pn[k];
    }
  }
#pragma unroll
  for (int k = 0; k < UPL; ++k)
#pragma unroll
    for (int e = 0; e < UE; ++e) {
      float vg = dg[k][e], vb = db[k][e];
#pragma unroll
      for (int off = 32; off >= LPR; off >>= 1) {  // the wave's groups
        vg += __shfl_xor(vg, off, 64);
        vb += __shfl_xor(vb, off, 64);
      }
      const int c = (l + LPR * k) * UE + e;
      if (sub == 0 && c < C) {
        red[(wave * 2 + 0) * C + c] = vg;
        red[(wave * 2 + 1) * C + c] = vb;
      }
    }
  __syncthreads();
  for (int i = threadIdx.x; i < 2 * C; i += 256)
    partials[(int64_t)blockIdx.x * 2 * C + i] = ((red[i] + red[2 * C + i]) + red[4 * C + i]) + red[6 * C + i];
}

// ------------------------------------------------------------------------------------------------
// dequant_e4m3_kernel: out[o, k] = bf16(scale[o] * decode_e4m3fn(in[o, k])), for the shapes whose kernels read the
// large weights in natural layout (the repacking kernels of the MFMA paths read the e4m3 bytes themselves).
// ------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void dequant_e4m3_kernel(const uint8_t *__restrict__ in, const float *__restrict__ scale,
                                                           bf16 *__restrict__ out, int64_t rows, int64_t cols) {
  const int64_t n = rows * cols;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
    store_from_f32(out + i, scale[i / cols] * decode_e4m3fn(in[i]));
}

// ================================================================================================
// host launchers
// ================================================================================================
template <typename TA, typename TW>
static int launch_gemm(const GemmArgs &a, int nsets, hipStream_t st) {
  if constexpr (sizeof(TA) == sizeof(TW))  // the MFMA kernels take both operands in one type
    if (gemm::serves(a, nsets, sizeof(TA))) return gemm::launch(a, nsets, sizeof(TA) == 4 ? PA_F32 : PA_BF16, st);
  dim3 grid((unsigned)((a.M + 63) / 64), (unsigned)((a.O + 63) / 64), (unsigned)nsets);
  hipLaunchKernelGGL((rows_gemm_kernel<TA, TW>), grid, dim3(256), 0, st, a);
  return launch_status();
}

int dequant_e4m3(const void *in, const float *scale, void *out, int64_t rows, int64_t cols, hipStream_t st) {
  int64_t blocks = (rows * cols + 255) / 256;
  if (blocks > 1024) blocks = 1024;
  hipLaunchKernelGGL(dequant_e4m3_kernel, dim3((unsigned)blocks), dim3(256), 0, st, static_cast<const uint8_t *>(in),
                     scale, static_cast<bf16 *>(out), rows, cols);
  return launch_status();
}

int project_inputs(int dtype, const pa_shape &s, const pa_params &p, const void *x, void *x_mid, void *fx_mid,
                   hipStream_t st) {
  GemmArgs a{};
  a.in = x;
  a.w[0] = p.in_project_x_weight;
  a.w[1] = p.in_project_fx_weight;
  a.bias[0] = p.in_project_x_bias;
  a.bias[1] = p.in_project_fx_bias;
  a.out[0] = x_mid;
  a.out[1] = fx_mid;
  a.M = s.B * s.N;
  a.O = (int)(s.H * s.D);
  a.C = (int)s.C;
  a.N = (int)s.N;
  a.gh = (int)s.grid_h;
  a.gw = (int)s.grid_w;
  a.ks = (int)s.conv_k;
  a.gd = (int)s.grid_d;
  a.w_tap_major = (int)s.conv_tap_major;
  a.K = s.conv_k > 0 ? (int)(s.conv_k * s.conv_k * (s.grid_d > 0 ? s.conv_k : 1) * s.C) : (int)s.C;
  const int nsets = fx_mid ? 2 : 1;  // Transolver++ has a single projection
  return dtype == PA_F32 ? launch_gemm<float, float>(a, nsets, st) : launch_gemm<bf16, bf16>(a, nsets, st);
}

// out[m, o] = bias[o] + sum_k A(m, k) weight[o, k] for any (c_in, c_out): a Linear over the rows when grid.conv_k == 0,
// else the k x k (x k) convolution over grid's point grid with weight (c_out, c_in, k, k(, k)).
int rows_gemm(int dtype, const pa_shape &grid, int64_t c_in, int64_t c_out, const void *in, const void *weight,
              const float *bias, int act, void *out, hipStream_t st) {
  GemmArgs a{};
  a.act = act;
  a.in = in;
  a.w[0] = weight;
  a.bias[0] = bias;
  a.out[0] = out;
  a.M = grid.B * grid.N;
  a.O = (int)c_out;
  a.C = (int)c_in;
  a.N = (int)grid.N;
  a.gh = (int)grid.grid_h;
  a.gw = (int)grid.grid_w;
  a.ks = (int)grid.conv_k;
  a.gd = (int)grid.grid_d;
  a.w_tap_major = (int)grid.conv_tap_major;
  a.K = grid.conv_k > 0 ? (int)(grid.conv_k * grid.conv_k * (grid.grid_d > 0 ? grid.conv_k : 1) * c_in) : (int)c_in;
  return dtype == PA_F32 ? launch_gemm<float, float>(a, 1, st) : launch_gemm<bf16, bf16>(a, 1, st);
}

// bf16 Linear over the rows with the result in natural layout (`out`, may be NULL) and in the packed operand layout of
// the MFMA slice kernels (`out_pack`, (B * tiles * H * 2) KiB as fx_pack); c_out = H * 32.
int rows_gemm_packed(const pa_shape &s, int64_t c_in, const void *in, const void *weight, const float *bias, void *out,
                     void *out_pack, hipStream_t st) {
  GemmArgs a{};
  a.in = in;
  a.w[0] = weight;
  a.bias[0] = bias;
  a.out[0] = out;
  a.out_pack[0] = out_pack;
  a.M = s.B * s.N;
  a.N = (int)s.N;
  a.K = (int)c_in;
  a.O = (int)(s.H * 32);
  a.C = (int)c_in;
  a.pack_tpb = (int)((s.N + 31) / 32);
  a.pack_heads = (int)s.H;
  if (c_in % 8 != 0 || !gemm::serves(a, 1, 2)) return PA_ERR_UNSUPPORTED;
  return gemm::launch(a, 1, PA_BF16, st);
}

int out_linear(int dtype, const pa_shape &s, const pa_params &p, const void *out_x, void *y, hipStream_t st) {
  GemmArgs a{};
  a.in = out_x;
  a.w[0] = p.out_linear_weight;
  a.bias[0] = p.out_linear_bias;
  a.out[0] = y;
  a.M = s.B * s.N;
  a.K = (int)(s.H * s.D);
  a.O = (int)s.C;
  a.ks = 0;
  return dtype == PA_F32 ? launch_gemm<float, float>(a, 1, st) : launch_gemm<bf16, bf16>(a, 1, st);
}

// Slice weights (PA.py:537, :172-181): the logits are a Linear over the (point, head) rows -- D inputs, S outputs,
// one weight for all heads -- so they come from the row GEMM kernels (MFMA for float32; the float32 weight against
// bf16 rows takes the FMA kernel), written in the storage type as the reference's Linear output is; the softmax with
// the head's clamped temperature then runs in place over each row of S.
template <typename T>
static int slice_softmax_t(const pa_shape &s, const pa_params &p, const void *x_mid, void *w, hipStream_t st) {
  GemmArgs a{};
  a.in = x_mid;
  a.w[0] = p.in_project_slice_weight;
  a.bias[0] = p.in_project_slice_bias;
  a.out[0] = w;
  a.M = s.B * s.N * s.H;
  a.K = (int)s.D;
  a.O = (int)s.S;
  int rc = launch_gemm<T, float>(a, 1, st);
  if (rc) return rc;
  return flare::softmax_rows(sizeof(T) == 4 ? PA_F32 : PA_BF16, s, w, p.temperature, st);
}

int slice_softmax(int dtype, const pa_shape &s, const pa_params &p, const void *x_mid, void *w, hipStream_t st) {
  return dtype == PA_F32 ? slice_softmax_t<float>(s, p, x_mid, w, st) : slice_softmax_t<bf16>(s, p, x_mid, w, st);
}

template <typename T, int L>
static int softmax_rows_plus_l(const pa_shape &s, const pa_params &p, const pa_plus_params &pp, void *w,
                               const void *hidden, const void *uniform, hipStream_t st) {
  const int64_t rows = s.B * s.N * s.H;
  int64_t blocks = (rows + (256 / L) - 1) / (256 / L);
  if (blocks > 16384) blocks = 16384;
  hipLaunchKernelGGL((softmax_rows_plus_kernel<T, L>), dim3((unsigned)blocks), dim3(256), 0, st, static_cast<T *>(w),
                     static_cast<const T *>(hidden), static_cast<const T *>(uniform), p.temperature,
                     pp.proj_temperature_2_weight, pp.proj_temperature_2_bias, rows, (int)s.S, (int)s.H);
  return launch_status();
}

template <typename T, int LR>
static int softmax_rows_plus_vec(const pa_shape &s, const pa_params &p, const pa_plus_params &pp, void *w,
                                 const void *hidden, const void *uniform, hipStream_t st) {
  const int64_t rows = s.B * s.N * s.H;
  int64_t blocks = (rows + (256 / LR) - 1) / (256 / LR);
  if (blocks > 16384) blocks = 16384;
  hipLaunchKernelGGL((softmax_rows_plus_vec_kernel<T, LR>), dim3((unsigned)blocks), dim3(256), 0, st,
                     static_cast<T *>(w), static_cast<const T *>(hidden), static_cast<const T *>(uniform), p.temperature,
                     pp.proj_temperature_2_weight, pp.proj_temperature_2_bias, rows, (int)s.S, (int)s.H);
  return launch_status();
}

// With a scratch buffer of B*N*H*S elements the two Linears run on the row GEMM kernels (several times faster than the
// single kernel below, which forms them per point on the vector ALUs).
template <typename T>
static int slice_softmax_plus_staged(const pa_shape &s, const pa_params &p, const pa_plus_params &pp, const void *x_mid,
                                     const void *uniform, void *w, void *scratch, hipStream_t st) {
  GemmArgs a{};
  a.in = x_mid;
  a.M = s.B * s.N * s.H;
  a.K = (int)s.D;
  a.O = (int)s.S;
  a.w[0] = p.in_project_slice_weight;
  a.bias[0] = p.in_project_slice_bias;
  a.out[0] = w;
  int rc = launch_gemm<T, float>(a, 1, st);
  if (rc) return rc;
  a.w[0] = pp.proj_temperature_0_weight;
  a.bias[0] = pp.proj_temperature_0_bias;
  a.out[0] = scratch;
  a.act = 1;
  if ((rc = launch_gemm<T, float>(a, 1, st))) return rc;
  constexpr int UE = 16 / sizeof(T);
  if (s.S % UE == 0 && s.S / UE <= 64 && (reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(scratch) |
                                          reinterpret_cast<uintptr_t>(uniform)) % 16 == 0) {
    const int64_t units = s.S / UE;
    if (units <= 1) return softmax_rows_plus_vec<T, 1>(s, p, pp, w, scratch, uniform, st);
    if (units <= 2) return softmax_rows_plus_vec<T, 2>(s, p, pp, w, scratch, uniform, st);
    if (units <= 4) return softmax_rows_plus_vec<T, 4>(s, p, pp, w, scratch, uniform, st);
    if (units <= 8) return softmax_rows_plus_vec<T, 8>(s, p, pp, w, scratch, uniform, st);
    if (units <= 16) return softmax_rows_plus_vec<T, 16>(s, p, pp, w, scratch, uniform, st);
    if (units <= 32) return softmax_rows_plus_vec<T, 32>(s, p, pp, w, scratch, uniform, st);
    return softmax_rows_plus_vec<T, 64>(s, p, pp, w, scratch, uniform, st);
  }
  if (s.S <= 8) return softmax_rows_plus_l<T, 8>(s, p, pp, w, scratch, uniform, st);
  if (s.S <= 16) return softmax_rows_plus_l<T, 16>(s, p, pp, w, scratch, uniform, st);
  if (s.S <= 32) return softmax_rows_plus_l<T, 32>(s, p, pp, w, scratch, uniform, st);
  return softmax_rows_plus_l<T, 64>(s, p, pp, w, scratch, uniform, st);
}

template <typename T>
static int slice_softmax_plus_t(const pa_shape &s, const pa_params &p, const pa_plus_params &pp, const void *x_mid,
                                const void *uniform, void *w, void *scratch, hipStream_t st) {
  if (scratch) return slice_softmax_plus_staged<T>(s, p, pp, x_mid, uniform, w, scratch, st);
  const int H = (int)s.H, D = (int)s.D, S = (int)s.S;
  const size_t fixed = (size_t)(2 * S * D + 3 * S) * 4;
  const size_t per_row = (size_t)(H * (D + 1) + H * (S + 1)) * 4;
  if (fixed + per_row > 60 * 1024) return PA_ERR_UNSUPPORTED;
  int R = (int)((60 * 1024 - fixed) / per_row);
  if (R > 8) R = 8;
  const size_t lds = fixed + per_row * R;
  int rc = allow_dynamic_lds(slice_softmax_plus_kernel<T>, lds);
  if (rc) return rc;
  const int64_t M = s.B * s.N;
  hipLaunchKernelGGL((slice_softmax_plus_kernel<T>), dim3((unsigned)((M + R - 1) / R)), dim3(256), lds, st,
                     static_cast<const T *>(x_mid), static_cast<const T *>(uniform), p.in_project_slice_weight,
                     p.in_project_slice_bias, p.temperature, pp.proj_temperature_0_weight, pp.proj_temperature_0_bias,
                     pp.proj_temperature_2_weight, pp.proj_temperature_2_bias, static_cast<T *>(w), M, H, D, S, R);
  return launch_status();
}

int slice_softmax_plus(int dtype, const pa_shape &s, const pa_params &p, const pa_plus_params &pp, const void *x_mid,
                       const void *uniform, void *w, void *scratch, hipStream_t st) {
  return dtype == PA_F32 ? slice_softmax_plus_t<float>(s, p, pp, x_mid, uniform, w, scratch, st)
                         : slice_softmax_plus_t<bf16>(s, p, pp, x_mid, uniform, w, scratch, st);
}

// Number of point chunks of the first reduction pass: enough workgroups to fill 256 CUs several times
// over, at least 256 points per chunk.  Depends on the shape only, so results are reproducible.
int64_t partial_count(const pa_shape &s) {
  int64_t by_size = (s.N + 255) / 256;
  int64_t by_grid = (4096 + s.B * s.H - 1) / (s.B * s.H);
  int64_t g = by_size < by_grid ? by_size : by_grid;
  return g < 1 ? 1 : g;
}

size_t combine_attn_lds_bytes(const pa_shape &s) {
  return (size_t)(4 * s.S * (s.D + 1) + (kAttnThreads / 64) * s.S) * 4;
}

template <typename T>
static int slice_partial_t(const pa_shape &s, const void *w, const void *fx_mid, float *partials, hipStream_t st) {
  const int64_t G = partial_count(s);
  const int64_t chunk = (s.N + G - 1) / G;
  const int SB = (int)((s.S + 3) / 4), DB = (int)((s.D + 1 + 3) / 4);
  const int n_tiles = SB * DB;
  const size_t rows = (size_t)kPartialTile * (SB + DB) * 16, sums = n_tiles <= 256 ? (size_t)(partial_groups(n_tiles) - 1) * n_tiles * 64 : 0;
  const size_t lds = rows > sums ? rows : sums;
  const int per_thread = (n_tiles + 255) / 256;
  const int ns = per_thread <= 1 ? 1 : (per_thread <= 2 ? 2 : kPartialMaxNS);
  dim3 grid((unsigned)G, (unsigned)(s.B * s.H), (unsigned)((n_tiles + 256 * ns - 1) / (256 * ns)));
  auto launch = [&](auto kernel) {
    int rc = allow_dynamic_lds(kernel, lds);
    if (rc) return rc;
    hipLaunchKernelGGL(kernel, grid, dim3(ns == 1 ? partial_threads(n_tiles) : 256), lds, st, static_cast<const T *>(w),
                       static_cast<const T *>(fx_mid), partials, (int)s.B, s.N, (int)s.H, (int)s.D, (int)s.S, chunk);
    return launch_status();
  };
  if (ns == 1) return launch(slice_partial_kernel<T, 1>);
  if (ns == 2) return launch(slice_partial_kernel<T, 2>);
  return launch(slice_partial_kernel<T, kPartialMaxNS>);
}

// `partials` holds G partial sums followed by one spare slot (index G) that receives their fixed-order total.
// G == 0: `partials` holds finished slice tokens (attention only).
// Fixed-order total of the G partial sums [G][B][H][S][D+1]; the total goes to slot G of the same buffer.  Returns
// where the totals are (the partials themselves when G == 1).
int combine_partials(const pa_shape &s, const float *partials, int64_t G, const float **combined, hipStream_t st) {
  const int64_t stride = s.B * s.H * s.S * (s.D + 1);
  *combined = partials;
  if (G <= 1) return PA_OK;
  float *total = const_cast<float *>(partials) + G * stride;
  const int n_out = (int)(s.S * (s.D + 1));
  // Four sums where one would be a chain of more than 64 roundings: slice tokens of 131 072 points in 512 partials 2.7e-7 -> 2.0e-7 off
  // float64, of 1 048 576 points in 4 096 6.0e-7 -> 3.3e-7.
  auto kernel = G > 256 ? combine_partials_kernel<4> : combine_partials_kernel<1>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)((n_out + 63) / 64), (unsigned)(s.B * s.H)), dim3(256), 0, st,
                     partials, (int)G, stride, total, n_out);
  *combined = total;
  return launch_status();
}

// Partials of a (b, h) that one workgroup sums itself: 256 of 32 x 17 floats take 3.6 us at the 64 bytes a clock that a CU gets
// from L2, about what the launch that spreads them over the chip costs with its start.
constexpr int64_t kFewPartials = 256;

template <int D>
static int narrow_combine_attention(const pa_shape &s, const pa_params &p, const float *partials, int64_t G, float *slice_token,
                                    float *slice_norm, float *out_token, hipStream_t st) {
  hipLaunchKernelGGL(narrow_combine_attn_kernel<D>, dim3((unsigned)(s.B * s.H)), dim3(32 * kNarrowSlices), 0, st, partials, (int)G,
                     s.B * s.H * s.S * (s.D + 1), p.qkv_project_weight, slice_token, slice_norm, out_token);
  return launch_status();
}

int combine_attention(const pa_shape &s, const pa_params &p, const float *partials, int64_t G, float *slice_token,
                      float *slice_norm, float *out_token, hipStream_t st) {
  if (s.S == kNarrowSlices && out_token && G > 8 && G <= kFewPartials) {
    if (s.D == 8) return narrow_combine_attention<8>(s, p, partials, G, slice_token, slice_norm, out_token, st);
    if (s.D == 16) return narrow_combine_attention<16>(s, p, partials, G, slice_token, slice_norm, out_token, st);
  }
  size_t lds = combine_attn_lds_bytes(s);
  const size_t wq_bytes = (size_t)3 * s.D * (s.D + 1) * 4;
  const int stage_w = lds + wq_bytes <= 96 * 1024 ? 1 : 0;  // qkv weight rows in LDS when they fit comfortably
  if (stage_w) lds += wq_bytes;
  int rc = allow_dynamic_lds(slice_combine_attn_kernel, lds);
  if (rc) return rc;
  const int64_t stride = s.B * s.H * s.S * (s.D + 1);
  const float *src = partials;
  int g_in = (int)G;  // a few partials are summed by the attention kernel itself, in index order
  if (G > 8) {
    if ((rc = combine_partials(s, partials, G, &src, st))) return rc;
    g_in = 1;
  }
  hipLaunchKernelGGL(slice_combine_attn_kernel, dim3((unsigned)(s.B * s.H)), dim3(kAttnThreads), lds, st, src, g_in, stride,
                     p.qkv_project_weight, slice_token, slice_norm, out_token, (int)s.D, (int)s.S, stage_w);
  return launch_status();
}

int slice_partial(int dtype, const pa_shape &s, const void *w, const void *fx_mid, float *partials, hipStream_t st) {
  return dtype == PA_F32 ? slice_partial_t<float>(s, w, fx_mid, partials, st)
                         : slice_partial_t<bf16>(s, w, fx_mid, partials, st);
}

template <typename T>
static int deslice_t(const pa_shape &s, const void *w, const float *out_token, void *out_x, hipStream_t st) {
  int R = 128;  // rows per workgroup: the head's token table (S x D floats) is loaded once per tile
  while (R > 8 && (size_t)(s.S * s.D + R * (s.S + 1)) * 4 > 48 * 1024) R >>= 1;
  size_t lds = (size_t)(s.S * s.D + R * (s.S + 1)) * 4;
  int rc = allow_dynamic_lds(deslice_kernel<T>, lds);
  if (rc) return rc;
  const int tiles = (int)((s.N + R - 1) / R);
  dim3 grid((unsigned)(tiles * s.B), (unsigned)s.H);
  hipLaunchKernelGGL((deslice_kernel<T>), grid, dim3(256), lds, st, static_cast<const T *>(w), out_token,
                     static_cast<T *>(out_x), s.N, (int)s.H, (int)s.D, (int)s.S, R, tiles);
  return launch_status();
}

int deslice(int dtype, const pa_shape &s, const void *w, const float *out_token, void *out_x, hipStream_t st) {
  return dtype == PA_F32 ? deslice_t<float>(s, w, out_token, out_x, st) : deslice_t<bf16>(s, w, out_token, out_x, st);
}

// f(integral constants LPR, UPL) for rows of `units` 16-byte units; false: longer than the kernels' 256 units
template <class F>
static bool for_row_units(int units, F &&f) {
  using std::integral_constant;
  const auto one = integral_constant<int, 1>{};
  if (units <= 4) f(integral_constant<int, 4>{}, one);
  else if (units <= 8) f(integral_constant<int, 8>{}, one);
  else if (units <= 16) f(integral_constant<int, 16>{}, one);
  else if (units <= 32) f(integral_constant<int, 32>{}, one);
  else if (units <= 64) f(integral_constant<int, 64>{}, one);
  else if (units <= 128) f(integral_constant<int, 64>{}, integral_constant<int, 2>{});
  else if (units <= 256) f(integral_constant<int, 64>{}, integral_constant<int, 4>{});
  else return false;
  return true;
}

template <typename T>
static int residual_ln_t(const pa_shape &s, void *y, const pa_block_tail &tail, hipStream_t st) {
  const int64_t M = s.B * s.N;
  const int C = (int)s.C;
  constexpr int UE = 16 / sizeof(T);
  T *yp = static_cast<T *>(y), *lo = static_cast<T *>(tail.ln_out);
  const T *res = static_cast<const T *>(tail.residual);
  const bool vec = C % UE == 0 && aligned16(y) && aligned16(tail.residual) && aligned16(tail.ln_out);
  if (vec && for_row_units(C / UE, [&](auto lpr, auto upl) {
        constexpr int LPR = decltype(lpr)::value, UPL = decltype(upl)::value, RPB = 4 * (64 / LPR);
        const dim3 grid((unsigned)std::min<int64_t>((M + RPB - 1) / RPB, 256 * 8));
        hipLaunchKernelGGL((residual_ln_rows_kernel<T, LPR, UPL>), grid, dim3(256), 0, st, yp, res, tail.ln_gamma,
                           tail.ln_beta, tail.ln_eps, lo, M, C);
      }))
    return launch_status();
  hipLaunchKernelGGL((residual_ln_kernel<T>), dim3((unsigned)((M + 3) / 4)), dim3(256), 0, st, yp, res, tail.ln_gamma,
                     tail.ln_beta, tail.ln_eps, lo, M, C);
  return launch_status();
}

// workgroups (partial sums): every wave walks several rows, so that the partials stay few next to the rows
int64_t layernorm_backward_groups(int64_t rows) { return std::min<int64_t>((rows + 15) / 16, 256 * 4); }

template <typename T>
static int layernorm_backward_t(int64_t rows, int C, const void *x, const void *dy, const void *add, const float *gamma,
                                float eps, void *dx, float *partials, hipStream_t st) {
  constexpr int UE = 16 / sizeof(T);
  if (C % UE != 0) return PA_ERR_UNSUPPORTED;
  const dim3 grid((unsigned)layernorm_backward_groups(rows));
  const size_t lds = (size_t)8 * C * 4;
  const bool ok = for_row_units(C / UE, [&](auto lpr, auto upl) {
    constexpr int LPR = decltype(lpr)::value, UPL = decltype(upl)::value;
    hipLaunchKernelGGL((layernorm_backward_rows_kernel<T, LPR, UPL>), grid, dim3(256), lds, st, static_cast<const T *>(x),
                       static_cast<const T *>(dy), static_cast<const T *>(add), gamma, eps, static_cast<T *>(dx), partials,
                       rows, C);
  });
  return ok ? launch_status() : PA_ERR_UNSUPPORTED;
}

// partials: layernorm_backward_groups(rows) * 2 C floats; grads (2, C): their sums d gamma, d beta, or NULL (the caller adds
// them up); add may be NULL
int layernorm_backward(int dtype, int64_t rows, int64_t C, const void *x, const void *dy, const void *add, const float *gamma,
                       float eps, void *dx, float *partials, float *grads, hipStream_t st) {
  const int rc = dtype == PA_F32 ? layernorm_backward_t<float>(rows, (int)C, x, dy, add, gamma, eps, dx, partials, st)
                                 : layernorm_backward_t<bf16>(rows, (int)C, x, dy, add, gamma, eps, dx, partials, st);
  return rc || !grads ? rc : wgrad::sum_rows(partials, layernorm_backward_groups(rows), 2 * C, grads, st);
}

int residual_ln(int dtype, const pa_shape &s, void *y, const pa_block_tail &tail, hipStream_t st) {
  return dtype == PA_F32 ? residual_ln_t<float>(s, y, tail, st) : residual_ln_t<bf16>(s, y, tail, st);
}

}  // namespace general
}  // namespace pa
