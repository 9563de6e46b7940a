// Float32 blocks of narrow models on an irregular mesh (C = 32 or 64 channels, heads of 8 or 16, 32 slices), two launches
// per block around the slice attention:
//   front_kernel   both projections, slice softmax, per-workgroup sums of the slice tokens (PA.py:106-170, :606-627)
//   tail_kernel    hand-back, out_linear, + residual, LayerNorm, MLP, + residual, next LayerNorm, output head (TR.py:300-307)
// A row is 128 or 256 bytes, so as separate products, softmax, reduction and LayerNorm launches (12 per block) every step
// is a trip through the caches with little work in it; here a point's intermediates stay in registers.
//
// Products are v_mfma_f32_32x32x2_f32 on tiles of 32 points, a wave to a tile.  Rows are held transposed: lane (i, g) <->
// point i, register r of tile c <-> channel 32 c + rowmap(r, g), four consecutive channels per register quad.  That is an
// accumulator's layout and at the same time, one register per step, the B (or A) operand of a product whose reduction index
// runs over the channels in the order (rowmap(r, 0), rowmap(r, 1)); the other operand is then a float4 per quad of the
// row-major weight, which lies in LDS as it is (rows four floats apart in the banks).
#include "pa_host.h"
#include "pa_mfma_ops.h"

namespace pa {
namespace narrow {

using mfma::f32x16;
using mfma::half_max;
using mfma::half_sum;
using mfma::rowmap;

constexpr int kS = 32, kWaves = 4;

__device__ __forceinline__ f32x16 mma32(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}
// keeps the LDS reads of a later section from being hoisted into registers here
__device__ __forceinline__ void section() { asm volatile("" ::: "memory"); }
__device__ __forceinline__ float4 quad(const float *p) { return *reinterpret_cast<const float4 *>(p); }
__device__ __forceinline__ float at(const float4 &v, int j) { return j == 0 ? v.x : j == 1 ? v.y : j == 2 ? v.z : v.w; }

// a row-major (rows, cols) matrix, cols a multiple of 4, into LDS rows of cols + 4 floats; several loads in flight at once
__device__ __forceinline__ void stage_matrix(const float *__restrict__ src, int rows, int cols, float *dst) {
  constexpr int NT = 64 * kWaves, AHEAD = 4;
  const int per = cols / 4, total = rows * per;
  if (reinterpret_cast<uintptr_t>(src) & 15u) {  // a weight that is a view off a 16-byte boundary
    for (int k = threadIdx.x; k < rows * cols; k += NT) dst[k / cols * (cols + 4) + k % cols] = src[k];
    return;
  }
  for (int k0 = threadIdx.x; k0 < total; k0 += AHEAD * NT) {
    float4 v[AHEAD];
#pragma unroll
    for (int e = 0; e < AHEAD; ++e) v[e] = reinterpret_cast<const float4 *>(src)[min(k0 + e * NT, total - 1)];
#pragma unroll
    for (int e = 0; e < AHEAD; ++e) {
      const int k = k0 + e * NT, r = k / per;
      if (k < total) *reinterpret_cast<float4 *>(dst + r * (cols + 4) + 4 * (k - r * per)) = v[e];
    }
  }
}
// M vectors of n <= 256 floats, all loads before the first store (NULL: `fill`)
template <int M>
__device__ __forceinline__ void stage_vectors(const float *const (&src)[M], const float (&fill)[M], float *const (&dst)[M], int n) {
  const int k = threadIdx.x;
  float v[M];
#pragma unroll
  for (int m = 0; m < M; ++m) v[m] = src[m] && k < n ? src[m][k] : fill[m];
#pragma unroll
  for (int m = 0; m < M; ++m)
    if (k < n) dst[m][k] = v[m];
}

// row-major (., C) row -> transposed tiles
template <int C>
__device__ __forceinline__ void load_row(const float *row, int g, f32x16 (&v)[C / 32]) {
#pragma unroll
  for (int c = 0; c < C / 32; ++c)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float4 e = quad(row + 32 * c + 8 * q + 4 * g);
      v[c][4 * q] = e.x, v[c][4 * q + 1] = e.y, v[c][4 * q + 2] = e.z, v[c][4 * q + 3] = e.w;
    }
}
template <int C>
__device__ __forceinline__ void store_row(float *row, int g, const f32x16 (&v)[C / 32]) {
#pragma unroll
  for (int c = 0; c < C / 32; ++c)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *reinterpret_cast<float4 *>(row + 32 * c + 8 * q + 4 * g) =
          float4{v[c][4 * q], v[c][4 * q + 1], v[c][4 * q + 2], v[c][4 * q + 3]};
}
// acc += W rows (lane i: row `wrow`, starting at the reduction index of v's first channel) . v^T
template <int T>
__device__ __forceinline__ void product(const float *wrow, int g, const f32x16 (&v)[T], f32x16 &acc) {
#pragma unroll
  for (int c = 0; c < T; ++c)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float4 w = quad(wrow + 32 * c + 8 * q + 4 * g);
#pragma unroll
      for (int j = 0; j < 4; ++j) acc = mma32(at(w, j), v[c][4 * q + j], acc);
    }
}
// the same un-transposed: rows of v^T (points) as A, W's rows as B columns -> lane i <-> W row, registers <-> points
template <int T>
__device__ __forceinline__ void product_rows(const float *wrow, int g, const f32x16 (&v)[T], f32x16 &acc) {
#pragma unroll
  for (int c = 0; c < T; ++c)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float4 w = quad(wrow + 32 * c + 8 * q + 4 * g);
#pragma unroll
      for (int j = 0; j < 4; ++j) acc = mma32(v[c][4 * q + j], at(w, j), acc);
    }
}
__device__ __forceinline__ void fill_from(const float *vec, int g, f32x16 &v) {  // channel vector in LDS
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float4 e = quad(vec + 8 * q + 4 * g);
    v[4 * q] = e.x, v[4 * q + 1] = e.y, v[4 * q + 2] = e.z, v[4 * q + 3] = e.w;
  }
}

template <int C, int D>
struct Front {
  static constexpr int H = C / D, kMat = C * (C + 4), kSliceW = kS * (D + 4);
  static constexpr int kTile = kS * (kS + 1);          // a wave's weights of one head, turned around
  static constexpr int kTok = H * kS * (D + 1);        // token sums of a wave
  static constexpr int kMain = 2 * kMat + kSliceW + 2 * C + kS + kWaves * kTile;
  static constexpr int kFloats = kMain > kWaves * kTok ? kMain : kWaves * kTok;
};

// grid: (groups, B); the waves of a group walk the batch's tiles 4 group + wave, + 4 groups, ...
// Bound by matrix issue and latency (a tile is 14 k cycles of one SIMD, every operand in the caches): 4 x 12 345 points of
// 64 channels 29 us, tail_kernel 31 us; the twelve launches they replace took 195 us.
template <int C, int D>
__global__ __launch_bounds__(64 * kWaves, C == 64 && D == 8 ? 1 : 2) void front_kernel(const float *__restrict__ x, const float *__restrict__ w_x,
                                                            const float *__restrict__ b_x, const float *__restrict__ w_fx,
                                                            const float *__restrict__ b_fx, const float *__restrict__ w_s,
                                                            const float *__restrict__ b_s,
                                                            const float *__restrict__ temperature, float *__restrict__ w,
                                                            float *__restrict__ partials, int64_t N) {
  using K = Front<C, D>;
  constexpr int H = K::H, T = C / 32, HPT = 32 / D;
  extern __shared__ float4 lds4[];
  float *lds = reinterpret_cast<float *>(lds4);
  float *wx = lds, *wf = wx + K::kMat, *ws = wf + K::kMat, *bx = ws + K::kSliceW, *bf = bx + C, *bs = bf + C, *turn = bs + kS;
  const int tid = threadIdx.x, lane = tid & 63, i = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = blockIdx.y, B = gridDim.y;
  stage_matrix(w_x, C, C, wx), stage_matrix(w_fx, C, C, wf), stage_matrix(w_s, kS, D, ws);
  stage_vectors<2>({b_x, b_fx}, {0.f, 0.f}, {bx, bf}, C);
  stage_vectors<1>({b_s}, {0.f}, {bs}, kS);
  float inv_t[H];
#pragma unroll
  for (int h = 0; h < H; ++h) inv_t[h] = 1.f / clamp_temperature(temperature[h]);
  turn += wave * K::kTile;
  f32x16 tok[H];
  float nrm[H];
#pragma unroll
  for (int h = 0; h < H; ++h) {
    nrm[h] = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) tok[h][r] = 0.f;
  }
  __syncthreads();
  const int64_t tiles = (N + 31) / 32;
  for (int64_t t = (int64_t)blockIdx.x * kWaves + wave; t < tiles; t += (int64_t)gridDim.x * kWaves) {
    const int64_t n = t * 32 + i;
    const bool ok = n < N;
    const int64_t row = (int64_t)b * N + (ok ? n : N - 1);
    f32x16 xt[T];
    load_row<C>(x + row * C, g, xt);
#pragma unroll
    for (int c = 0; c < T; ++c) {
      f32x16 xm, fx;
      fill_from(bx + 32 * c, g, xm);
      const float bfi = bf[32 * c + i];
#pragma unroll
      for (int r = 0; r < 16; ++r) fx[r] = bfi;
      product<T>(wx + (32 * c + i) * (C + 4), g, xt, xm);
      product_rows<T>(wf + (32 * c + i) * (C + 4), g, xt, fx);
#pragma unroll
      for (int hh = 0; hh < HPT; ++hh) {
        constexpr int QPH = D / 8;  // register quads of a head
        const int h = HPT * c + hh;
        f32x16 lg;
        fill_from(bs, g, lg);
#pragma unroll
        for (int q = 0; q < QPH; ++q) {
          const float4 a = quad(ws + i * (D + 4) + 8 * q + 4 * g);
#pragma unroll
          for (int j = 0; j < 4; ++j) lg = mma32(at(a, j), xm[4 * (QPH * hh + q) + j], lg);
        }
        float mx = -INFINITY, sum = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          lg[r] *= inv_t[h];
          mx = fmaxf(mx, lg[r]);
        }
        mx = half_max(mx);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          lg[r] = expf(lg[r] - mx);
          sum += lg[r];
        }
        const float inv = 1.f / half_sum(sum);
        // the weights leave, and turn around in LDS: lane (point) x register (slice) -> lane (slice) x step (point)
#pragma unroll
        for (int r = 0; r < 16; ++r) lg[r] *= inv;
        if (ok) {
          f32x16 one[1] = {lg};
          store_row<32>(w + (row * H + h) * kS, g, one);
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) turn[i * (kS + 1) + rowmap(r, g)] = ok ? lg[r] : 0.f;
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float a = turn[rowmap(r, g) * (kS + 1) + i];
          nrm[h] += a;
          tok[h] = mma32(a, fx[r], tok[h]);
        }
        __builtin_amdgcn_wave_barrier();  // read before the next head overwrites them
      }
    }
  }
  // tok[h]: lane i <-> channel i of the head's tile (only its own D count), registers <-> slices; nrm[h]: lane i <-> slice i
  __syncthreads();  // the weights in LDS are done with
  float *mine = lds + wave * K::kTok;
#pragma unroll
  for (int h = 0; h < H; ++h) {
    const float total = half_sum(nrm[h]);
    if (g == 0) mine[(h * kS + i) * (D + 1) + D] = total;
    if (i / D == h % HPT) {
#pragma unroll
      for (int r = 0; r < 16; ++r) mine[(h * kS + rowmap(r, g)) * (D + 1) + i % D] = tok[h][r];
    }
  }
  __syncthreads();
  float *dst = partials + ((int64_t)blockIdx.x * B + b) * K::kTok;
  for (int k = tid; k < K::kTok; k += 64 * kWaves)
    dst[k] = ((lds[k] + lds[K::kTok + k]) + lds[2 * K::kTok + k]) + lds[3 * K::kTok + k];
}

struct TailArgs {
  const float *w, *out_token, *w_out, *b_out, *fx_in, *ln2_gamma, *ln2_beta, *w1, *b1, *w2, *b2;
  float ln2_eps, next_eps;
  float *fx_out, *ln_out;  // ln_out: NULL: not stored
  const float *next_gamma, *next_beta, *head_w, *head_b;
  float *head_out;
  int O, F;
  int64_t N;
};

template <int C, int D>
struct Tail {
  static constexpr int H = C / D, kTok = C * (kS + 4);
  static constexpr int floats(int F) { return C * (C + 4) + F * (C + 4) + C * (F + 4) + kTok + 6 * C + F + 4 * C; }
};

template <int C>
__device__ __forceinline__ void layer_norm(const f32x16 (&v)[C / 32], const float *gamma, const float *beta, float eps, int g,
                                           f32x16 (&out)[C / 32]) {
  float sum = 0.f, sq = 0.f;
#pragma unroll
  for (int c = 0; c < C / 32; ++c)
#pragma unroll
    for (int r = 0; r < 16; ++r) sum += v[c][r];
  const float mean = half_sum(sum) * (1.f / C);
#pragma unroll
  for (int c = 0; c < C / 32; ++c)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float d = v[c][r] - mean;
      sq = fmaf(d, d, sq);
    }
  const float rstd = 1.f / sqrtf(half_sum(sq) * (1.f / C) + eps);
#pragma unroll
  for (int c = 0; c < C / 32; ++c)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float4 ga = quad(gamma + 32 * c + 8 * q + 4 * g), be = quad(beta + 32 * c + 8 * q + 4 * g);
#pragma unroll
      for (int j = 0; j < 4; ++j) out[c][4 * q + j] = (v[c][4 * q + j] - mean) * rstd * at(ga, j) + at(be, j);
    }
}

// grid: (groups, B), tiles as above
template <int C, int D>
__global__ __launch_bounds__(64 * kWaves, C == 64 && D == 8 ? 1 : 2) void tail_kernel(TailArgs a) {
  using K = Tail<C, D>;
  constexpr int H = K::H, T = C / 32, HPT = 32 / D;
  const int F = a.F;
  extern __shared__ float4 lds4[];
  float *lds = reinterpret_cast<float *>(lds4);
  float *wo = lds, *w1 = wo + C * (C + 4), *w2 = w1 + F * (C + 4), *tokt = w2 + C * (F + 4), *bo = tokt + K::kTok, *g2 = bo + C,
        *be2 = g2 + C, *gn = be2 + C, *ben = gn + C, *b2 = ben + C, *b1 = b2 + C, *hw = b1 + F;
  const int tid = threadIdx.x, lane = tid & 63, i = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = blockIdx.y;
  stage_matrix(a.w_out, C, C, wo), stage_matrix(a.w1, F, C, w1), stage_matrix(a.w2, C, F, w2);
  // the batch's attended tokens (H, 32, D) turned: row h D + d, the slices along it
  constexpr int TPT = H * kS * D / (64 * kWaves);  // tokens per thread
  float tv[TPT];
#pragma unroll
  for (int e = 0; e < TPT; ++e) tv[e] = a.out_token[(int64_t)b * H * kS * D + e * 64 * kWaves + tid];
#pragma unroll
  for (int e = 0; e < TPT; ++e) {
    const int k = e * 64 * kWaves + tid, d = k % D, s = k / D % kS, h = k / (D * kS);
    tokt[(h * D + d) * (kS + 4) + s] = tv[e];
  }
  stage_vectors<6>({a.b_out, a.ln2_gamma, a.ln2_beta, a.next_gamma, a.next_beta, a.b2}, {0.f, 1.f, 0.f, 1.f, 0.f, 0.f},
                   {bo, g2, be2, gn, ben, b2}, C);
  stage_vectors<1>({a.head_w}, {0.f}, {hw}, a.O * C);
  for (int k = tid; k < F; k += 64 * kWaves) b1[k] = a.b1[k];
  __syncthreads();
  const int64_t tiles = (a.N + 31) / 32;
  for (int64_t t = (int64_t)blockIdx.x * kWaves + wave; t < tiles; t += (int64_t)gridDim.x * kWaves) {
    const int64_t n = t * 32 + i;
    const bool ok = n < a.N;
    const int64_t row = (int64_t)b * a.N + (ok ? n : a.N - 1);
    f32x16 fx[T];  // residual row
    load_row<C>(a.fx_in + row * C, g, fx);
    // out_x^T: tile c's rows are the channels of HPT heads; every head's product counts for its own D rows only
    f32x16 ox[T];
#pragma unroll
    for (int c = 0; c < T; ++c) {
#pragma unroll
      for (int r = 0; r < 16; ++r) ox[c][r] = 0.f;
      f32x16 wt[HPT];  // the point's slice weights of the tile's heads
      load_row<HPT * kS>(a.w + (row * H + HPT * c) * kS, g, wt);
#pragma unroll
      for (int hh = 0; hh < HPT; ++hh)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float4 e = quad(tokt + (32 * c + i) * (kS + 4) + 8 * q + 4 * g);
          const bool own = i / D == hh;
#pragma unroll
          for (int j = 0; j < 4; ++j) ox[c] = mma32(own ? at(e, j) : 0.f, wt[hh][4 * q + j], ox[c]);
        }
    }
    // fx1 = out_x W_out^T + b_out + fx_in
#pragma unroll
    for (int c = 0; c < T; ++c) {
      f32x16 y;
      fill_from(bo + 32 * c, g, y);
      section();
      product<T>(wo + (32 * c + i) * (C + 4), g, ox, y);
#pragma unroll
      for (int r = 0; r < 16; ++r) fx[c][r] += y[r];
    }
    f32x16 nt[T], y[T];
    layer_norm<C>(fx, g2, be2, a.ln2_eps, g, nt);
#pragma unroll
    for (int c = 0; c < T; ++c) fill_from(b2 + 32 * c, g, y[c]);
    for (int f = 0; f < F; f += 32) {
      f32x16 h[1];
      fill_from(b1 + f, g, h[0]);
      section();
      product<T>(w1 + (f + i) * (C + 4), g, nt, h[0]);
#pragma unroll
      for (int r = 0; r < 16; ++r) h[0][r] = gelu_erf(h[0][r]);
#pragma unroll
      for (int c = 0; c < T; ++c) {
        section();
        product<1>(w2 + (32 * c + i) * (F + 4) + f, g, h, y[c]);
      }
    }
#pragma unroll
    for (int c = 0; c < T; ++c)
#pragma unroll
      for (int r = 0; r < 16; ++r) y[c][r] += fx[c][r];
    if (ok) store_row<C>(a.fx_out + row * C, g, y);
    if (!a.ln_out && a.O == 0) continue;
    layer_norm<C>(y, gn, ben, a.next_eps, g, nt);
    if (ok && a.ln_out) store_row<C>(a.ln_out + row * C, g, nt);
    for (int o = 0; o < a.O; ++o) {
      float acc = 0.f;
#pragma unroll
      for (int c = 0; c < T; ++c)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float4 e = quad(hw + o * C + 32 * c + 8 * q + 4 * g);
#pragma unroll
          for (int j = 0; j < 4; ++j) acc = fmaf(nt[c][4 * q + j], at(e, j), acc);
        }
      acc = half_sum(acc) + (a.head_b ? a.head_b[o] : 0.f);
      if (ok && g == 0) a.head_out[row * a.O + o] = acc;
    }
  }
}

bool block_supported(int dtype, const pa_shape &s, int64_t F) {
  if (dtype != PA_F32 || s.conv_k != 0 || s.S != kS || (s.C != 32 && s.C != 64) || (s.D != 8 && s.D != 16) || s.H * s.D != s.C)
    return false;
  if (F < 32 || F % 32 != 0 || s.B > 65535) return false;
  const int64_t floats = s.C == 32 ? Tail<32, 8>::floats((int)F) : Tail<64, 8>::floats((int)F);  // the same for both D
  return F <= 1024 && floats * 4 <= 160 * 1024;
}

// workgroups per batch element: one tile per wave while two workgroups per CU can take them all
int64_t groups(const pa_shape &s, int num_cu) {
  const int64_t all = ((s.N + 31) / 32 + kWaves - 1) / kWaves, most = (2 * num_cu + s.B - 1) / s.B;
  return all < most ? all : most;
}

template <int C, int D>
static int front_t(const pa_shape &s, const pa_params &p, const void *x, float *w, float *partials, int64_t G, hipStream_t st) {
  const size_t lds = (size_t)Front<C, D>::kFloats * 4;
  if (int rc = allow_dynamic_lds(front_kernel<C, D>, lds)) return rc;
  hipLaunchKernelGGL((front_kernel<C, D>), dim3((unsigned)G, (unsigned)s.B), dim3(64 * kWaves), lds, st,
                     static_cast<const float *>(x), static_cast<const float *>(p.in_project_x_weight), p.in_project_x_bias,
                     static_cast<const float *>(p.in_project_fx_weight), p.in_project_fx_bias,
                     static_cast<const float *>(p.in_project_slice_weight), p.in_project_slice_bias, p.temperature, w, partials,
                     s.N);
  return launch_status();
}

template <int C, int D>
static int tail_t(const pa_shape &s, const TailArgs &a, int64_t G, hipStream_t st) {
  const size_t lds = (size_t)Tail<C, D>::floats(a.F) * 4;
  if (int rc = allow_dynamic_lds(tail_kernel<C, D>, lds)) return rc;
  hipLaunchKernelGGL((tail_kernel<C, D>), dim3((unsigned)G, (unsigned)s.B), dim3(64 * kWaves), lds, st, a);
  return launch_status();
}

int front(const pa_shape &s, const pa_params &p, const void *x, float *w, float *partials, int num_cu, hipStream_t st) {
  const int64_t G = groups(s, num_cu);
  if (s.C == 32) return s.D == 8 ? front_t<32, 8>(s, p, x, w, partials, G, st) : front_t<32, 16>(s, p, x, w, partials, G, st);
  return s.D == 8 ? front_t<64, 8>(s, p, x, w, partials, G, st) : front_t<64, 16>(s, p, x, w, partials, G, st);
}

int block_tail(const pa_shape &s, const pa_params &p, const pa_block_mlp &m, const float *w, const float *out_token,
               const void *fx_in, void *fx_out, const pa_block_tail *next, const pa_block_head *head, int num_cu,
               hipStream_t st) {
  TailArgs a{};
  a.w = w, a.out_token = out_token;
  a.w_out = static_cast<const float *>(p.out_linear_weight), a.b_out = p.out_linear_bias;
  a.fx_in = static_cast<const float *>(fx_in), a.fx_out = static_cast<float *>(fx_out);
  a.ln2_gamma = m.ln_gamma, a.ln2_beta = m.ln_beta, a.ln2_eps = m.ln_eps;
  a.w1 = static_cast<const float *>(m.w1), a.b1 = m.b1, a.w2 = static_cast<const float *>(m.w2), a.b2 = m.b2;
  a.F = (int)m.F, a.N = s.N;
  if (next) {
    a.ln_out = static_cast<float *>(next->ln_out);
    a.next_gamma = next->ln_gamma, a.next_beta = next->ln_beta, a.next_eps = next->ln_eps;
  }
  if (head) {
    a.head_w = static_cast<const float *>(head->weight), a.head_b = head->bias;
    a.head_out = static_cast<float *>(head->out), a.O = (int)head->O;
  }
  const int64_t G = groups(s, num_cu);
  if (s.C == 32) return s.D == 8 ? tail_t<32, 8>(s, a, G, st) : tail_t<32, 16>(s, a, G, st);
  return s.D == 8 ? tail_t<64, 8>(s, a, G, st) : tail_t<64, 16>(s, a, G, st);
}

}  // namespace narrow
}  // namespace pa
