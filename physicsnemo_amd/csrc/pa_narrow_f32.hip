// Float32 blocks of narrow models on an irregular mesh (C = 32 or 64 channels, heads of 8 or 16, 32 slices), two launches
// per block around the slice attention:
//   front_kernel   both projections, slice softmax, per-workgroup sums of the slice tokens (PA.py:106-170, :606-627)
//   tail_kernel    hand-back, out_linear, + residual, LayerNorm, MLP, + residual, next LayerNorm, output head (TR.py:300-307)
// A row is 128 or 256 bytes, so as separate products, softmax, reduction and LayerNorm launches (12 per block) every step
// is a trip through the caches with little work in it; here a point's intermediates stay in registers.
//
// Products are v_mfma_f32_16x16x4_f32 on tiles of 16 points, a wave to a tile (a head of 16 channels fills a tile of columns, where
// tiles of 32 multiplied zeros for half or three quarters of them, and a wave is small enough for four on a SIMD).  Rows are held
// transposed: lane (i, g) = 16 g + i <-> point i, register r of tile c <-> channel 16 c + 4 g + r.  That is an accumulator's layout and
// at the same time, one register per step, the B (or A) operand of a product whose reduction index runs over the channels in the
// order 4 g + r, g = 0 .. 3; the other operand is then a float4 per tile of the row-major weight, which lies in LDS as it is
// (rows four floats apart in the banks).
#include "pa_host.h"
#include "pa_narrow_ops.h"

namespace pa {
namespace narrow {

__device__ __forceinline__ float4 quad(const float *p) { return *reinterpret_cast<const float4 *>(p); }
__device__ __forceinline__ float at(const float4 &v, int j) { return j == 0 ? v.x : j == 1 ? v.y : j == 2 ? v.z : v.w; }

// three row-major (rows, cols) matrices, cols a multiple of 4, into LDS rows of cols + 4 floats; loads of all of them in flight at once
struct Matrix {
  const float *src;
  int rows, cols;
  float *dst;
  __device__ __forceinline__ bool whole() const { return (reinterpret_cast<uintptr_t>(src) & 15u) == 0; }
  __device__ __forceinline__ int units() const { return whole() ? rows * (cols / 4) : 0; }
  __device__ __forceinline__ float4 load(int k) const { return reinterpret_cast<const float4 *>(src)[min(k, units() - 1)]; }
  __device__ __forceinline__ void store(int k, float4 v) const {
    const int per = cols / 4, r = k / per;
    if (k < units()) *reinterpret_cast<float4 *>(dst + r * (cols + 4) + 4 * (k - r * per)) = v;
  }
  __device__ __forceinline__ void by_element() const {  // a weight that is a view off a 16-byte boundary
    for (int k = threadIdx.x; k < rows * cols; k += blockDim.x) dst[k / cols * (cols + 4) + k % cols] = src[k];
  }
};
__device__ __forceinline__ void stage_matrices(Matrix a, Matrix b, Matrix c) {
  if (!(a.whole() && b.whole() && c.whole())) {
    a.by_element(), b.by_element(), c.by_element();
    return;
  }
  const int NT = blockDim.x, most = max(a.units(), max(b.units(), c.units()));
  for (int k = threadIdx.x; k < most; k += 2 * NT) {
    const float4 a0 = a.load(k), a1 = a.load(k + NT), b0 = b.load(k), b1 = b.load(k + NT), c0 = c.load(k), c1 = c.load(k + NT);
    a.store(k, a0), a.store(k + NT, a1), b.store(k, b0), b.store(k + NT, b1), c.store(k, c0), c.store(k + NT, c1);
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
__device__ __forceinline__ void load_row(const float *row, int g, f32x4 (&v)[C / 16]) {
#pragma unroll
  for (int c = 0; c < C / 16; ++c) v[c] = *reinterpret_cast<const f32x4 *>(row + 16 * c + 4 * g);
}
template <int C>
__device__ __forceinline__ void store_row(float *row, int g, const f32x4 (&v)[C / 16]) {
#pragma unroll
  for (int c = 0; c < C / 16; ++c) *reinterpret_cast<f32x4 *>(row + 16 * c + 4 * g) = v[c];
}
// acc += W rows (lane i: row `wrow`, starting at the reduction index of v's first channel) . v^T
template <int T>
__device__ __forceinline__ void product(const float *wrow, int g, const f32x4 (&v)[T], f32x4 &acc) {
#pragma unroll
  for (int c = 0; c < T; ++c) {
    const float4 w = quad(wrow + 16 * c + 4 * g);
#pragma unroll
    for (int j = 0; j < 4; ++j) acc = mma16(at(w, j), v[c][j], acc);
  }
}
// the same un-transposed: rows of v^T (points) as A, W's rows as B columns -> lane i <-> W row, registers <-> points
template <int T>
__device__ __forceinline__ void product_rows(const float *wrow, int g, const f32x4 (&v)[T], f32x4 &acc) {
#pragma unroll
  for (int c = 0; c < T; ++c) {
    const float4 w = quad(wrow + 16 * c + 4 * g);
#pragma unroll
    for (int j = 0; j < 4; ++j) acc = mma16(v[c][j], at(w, j), acc);
  }
}
__device__ __forceinline__ f32x4 fill_from(const float *vec, int g) { return *reinterpret_cast<const f32x4 *>(vec + 4 * g); }  // channel vector in LDS

template <int C, int D, int W>
struct Front {
  static constexpr int H = C / D, kMat = C * (C + 4), kSliceW = kS * (D + 4);
  static constexpr int kTurn = kTilePts * (kS + 4);    // a wave's weights of one head, turned around
  static constexpr int kTok = H * kS * (D + 1);        // token sums of a wave
  static constexpr int kMain = 2 * kMat + kSliceW + 2 * C + kS + W * kTurn;
  static constexpr int kFloats = kMain > W * kTok ? kMain : W * kTok;
};

// grid: (groups, B), W waves; the waves of a group walk the batch's tiles W group + wave, + W groups, ...
// Bound by matrix issue (6 144 cycles of one SIMD per tile of 16 points at D = 16) and the vector work of the softmax beside it; one
// tile per wave and four waves per SIMD at most cover each other's waits.  The two do not overlap: v_mfma_f32_* runs on the vector
// unit's lanes (eight fma and one 32 x 32 x 2: 42.7 ns, the fma alone 14.8, the MFMA alone 27.7).  Four clouds of 12 345 points, 64
// channels, 16-wide heads: 26.5 us, tail_kernel 26.5; on tiles of 32 points (v_mfma_f32_32x32x2_f32) 30.4 and 30.8.  2 x 8 000 points
// 13 and 12 against 19 and 19, 500 points 10.5 and 10 against 15.8 and 15; the twelve launches they replaced took 195 us a block.
template <int C, int D, int W>
__global__ __launch_bounds__(64 * W, C == 64 && D == 8 ? 2 : 4) void front_kernel(const float *__restrict__ x, const float *__restrict__ w_x,
                                                          const float *__restrict__ b_x, const float *__restrict__ w_fx,
                                                          const float *__restrict__ b_fx, const float *__restrict__ w_s,
                                                          const float *__restrict__ b_s,
                                                          const float *__restrict__ temperature, float *__restrict__ w,
                                                          float *__restrict__ partials, int64_t N) {
  using K = Front<C, D, W>;
  constexpr int H = K::H, T = C / 16, HPT = 16 / D;  // heads per tile of channels
  extern __shared__ float4 lds4[];
  float *lds = reinterpret_cast<float *>(lds4);
  float *wx = lds, *wf = wx + K::kMat, *ws = wf + K::kMat, *bx = ws + K::kSliceW, *bf = bx + C, *bs = bf + C, *turn = bs + kS;
  const int tid = threadIdx.x, lane = tid & 63, i = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = blockIdx.y, B = gridDim.y;
  const int64_t tiles = (N + kTilePts - 1) / kTilePts, t0 = (int64_t)blockIdx.x * W + wave, step = (int64_t)gridDim.x * W;
  auto row_of = [&](int64_t t) {  // the last row again beyond N
    const int64_t n = t * kTilePts + i;
    return (int64_t)b * N + (n < N ? n : N - 1);
  };
  f32x4 xt[T];
  if (t0 < tiles) load_row<C>(x + row_of(t0) * C, g, xt);  // on its way while the weights are
  stage_matrices({w_x, C, C, wx}, {w_fx, C, C, wf}, {w_s, kS, D, ws});
  stage_vectors<2>({b_x, b_fx}, {0.f, 0.f}, {bx, bf}, C);
  stage_vectors<1>({b_s}, {0.f}, {bs}, kS);
  float sc[H], sc_low[H];
#pragma unroll
  for (int h = 0; h < H; ++h) {
    exponent_scale(clamp_temperature(temperature[h]), sc[h], sc_low[h]);
  }
  turn += wave * K::kTurn;
  f32x4 tok[H][2];  // lane i <-> channel i of the head's tile, registers <-> slices 16 st + 4 g + r
  float nrm[H][2];  // lane i <-> slice 16 st + i
#pragma unroll
  for (int h = 0; h < H; ++h)
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      nrm[h][st] = 0.f;
      tok[h][st] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  __syncthreads();
  for (int64_t t = t0; t < tiles; t += step) {
    const bool ok = t * kTilePts + i < N;
    const int64_t row = row_of(t);
#pragma unroll
    for (int c = 0; c < T; ++c) {
      section();
      f32x4 xm = fill_from(bx + 16 * c, g), fx;
      const float bfi = bf[16 * c + i];
#pragma unroll
      for (int r = 0; r < 4; ++r) fx[r] = bfi;
      product<T>(wx + (16 * c + i) * (C + 4), g, xt, xm);
      product_rows<T>(wf + (16 * c + i) * (C + 4), g, xt, fx);
#pragma unroll
      for (int hh = 0; hh < HPT; ++hh) {
        const int h = HPT * c + hh;
        f32x4 lg[2];
        float mx = -INFINITY, sum = 0.f;
#pragma unroll
        for (int st = 0; st < 2; ++st) {
          lg[st] = fill_from(bs + 16 * st, g);
          // D = 8: the tile's channels 4 g + r belong to head g / 2, the other head's lanes bring zeros
          const float4 a = quad(ws + (16 * st + i) * (D + 4) + 4 * (D == 16 ? g : g & 1));
          const bool own = D == 16 || (g >> 1) == hh;
#pragma unroll
          for (int j = 0; j < 4; ++j) lg[st] = mma16(own ? at(a, j) : 0.f, xm[j], lg[st]);
#pragma unroll
          for (int r = 0; r < 4; ++r) mx = fmaxf(mx, lg[st][r]);
        }
        mx = group_max(mx);
#pragma unroll
        for (int st = 0; st < 2; ++st)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            lg[st][r] = exponential(lg[st][r] - mx, sc[h], sc_low[h]);
            sum += lg[st][r];
          }
        const float inv = 1.f / group_sum(sum);
        // the weights leave, and turn around in LDS: lane (point) x register (slice) -> lane (slice) x step (point)
#pragma unroll
        for (int st = 0; st < 2; ++st) lg[st] *= inv;
        if (ok) store_row<kS>(w + (row * H + h) * kS, g, lg);
#pragma unroll
        for (int st = 0; st < 2; ++st) *reinterpret_cast<f32x4 *>(turn + i * (kS + 4) + 16 * st + 4 * g) = ok ? lg[st] : f32x4{0.f, 0.f, 0.f, 0.f};
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int st = 0; st < 2; ++st)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float a = turn[(4 * g + r) * (kS + 4) + 16 * st + i];
            nrm[h][st] += a;
            tok[h][st] = mma16(a, fx[r], tok[h][st]);
          }
        __builtin_amdgcn_wave_barrier();  // read before the next head overwrites them
      }
    }
    if (t + step < tiles) load_row<C>(x + row_of(t + step) * C, g, xt);
  }
  __syncthreads();  // the weights in LDS are done with
  float *mine = lds + wave * K::kTok;
#pragma unroll
  for (int h = 0; h < H; ++h)
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      const float total = group_sum(nrm[h][st]);
      if (g == 0) mine[(h * kS + 16 * st + i) * (D + 1) + D] = total;
      if (i / D == h % HPT) {  // D = 8: a head's own half of the columns
#pragma unroll
        for (int r = 0; r < 4; ++r) mine[(h * kS + 16 * st + 4 * g + r) * (D + 1) + i % D] = tok[h][st][r];
      }
    }
  __syncthreads();
  float *dst = partials + ((int64_t)blockIdx.x * B + b) * K::kTok;
  for (int k = tid; k < K::kTok; k += 64 * W) {
    float v = lds[k];
#pragma unroll
    for (int u = 1; u < W; ++u) v += lds[u * K::kTok + k];
    dst[k] = v;
  }
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
__device__ __forceinline__ void layer_norm(const f32x4 (&v)[C / 16], const float *gamma, const float *beta, float eps, int g,
                                           f32x4 (&out)[C / 16]) {
  float sum = 0.f, sq = 0.f;
#pragma unroll
  for (int c = 0; c < C / 16; ++c)
#pragma unroll
    for (int r = 0; r < 4; ++r) sum += v[c][r];
  const float mean = group_sum(sum) * (1.f / C);
#pragma unroll
  for (int c = 0; c < C / 16; ++c)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float d = v[c][r] - mean;
      sq = fmaf(d, d, sq);
    }
  const float rstd = 1.f / sqrtf(group_sum(sq) * (1.f / C) + eps);
#pragma unroll
  for (int c = 0; c < C / 16; ++c) {
    const float4 ga = quad(gamma + 16 * c + 4 * g), be = quad(beta + 16 * c + 4 * g);
#pragma unroll
    for (int j = 0; j < 4; ++j) out[c][j] = (v[c][j] - mean) * rstd * at(ga, j) + at(be, j);
  }
}

// grid: (groups, B), tiles as above.  7 168 cycles of matrix issue per tile at F = 64, and erff beside them.
template <int C, int D, int W>
__global__ __launch_bounds__(64 * W, 4) void tail_kernel(TailArgs a) {
  using K = Tail<C, D>;
  constexpr int H = K::H, T = C / 16, HPT = 16 / D;
  const int F = a.F;
  extern __shared__ float4 lds4[];
  float *lds = reinterpret_cast<float *>(lds4);
  float *wo = lds, *w1 = wo + C * (C + 4), *w2 = w1 + F * (C + 4), *tokt = w2 + C * (F + 4), *bo = tokt + K::kTok, *g2 = bo + C,
        *be2 = g2 + C, *gn = be2 + C, *ben = gn + C, *b2 = ben + C, *b1 = b2 + C, *hw = b1 + F;
  const int tid = threadIdx.x, lane = tid & 63, i = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = blockIdx.y;
  const int64_t tiles = (a.N + kTilePts - 1) / kTilePts, t0 = (int64_t)blockIdx.x * W + wave, step = (int64_t)gridDim.x * W;
  auto row_of = [&](int64_t t) {  // the last row again beyond N
    const int64_t n = t * kTilePts + i;
    return (int64_t)b * a.N + (n < a.N ? n : a.N - 1);
  };
  f32x4 fx[T];  // residual row
  if (t0 < tiles) load_row<C>(a.fx_in + row_of(t0) * C, g, fx);  // on its way while the weights are
  stage_matrices({a.w_out, C, C, wo}, {a.w1, F, C, w1}, {a.w2, C, F, w2});
  // the batch's attended tokens (H, 32, D) turned: row h D + d, the slices along it
  constexpr int TPT = H * kS * D / (64 * W);  // tokens per thread
  float tv[TPT];
#pragma unroll
  for (int e = 0; e < TPT; ++e) tv[e] = a.out_token[(int64_t)b * H * kS * D + e * 64 * W + tid];
#pragma unroll
  for (int e = 0; e < TPT; ++e) {
    const int k = e * 64 * W + tid, d = k % D, s = k / D % kS, h = k / (D * kS);
    tokt[(h * D + d) * (kS + 4) + s] = tv[e];
  }
  stage_vectors<6>({a.b_out, a.ln2_gamma, a.ln2_beta, a.next_gamma, a.next_beta, a.b2}, {0.f, 1.f, 0.f, 1.f, 0.f, 0.f},
                   {bo, g2, be2, gn, ben, b2}, C);
  stage_vectors<1>({a.head_w}, {0.f}, {hw}, a.O * C);
  for (int k = tid; k < F; k += 64 * W) b1[k] = a.b1[k];
  __syncthreads();
  for (int64_t t = t0; t < tiles; t += step) {
    const bool ok = t * kTilePts + i < a.N;
    const int64_t row = row_of(t);
    // out_x^T: tile c's rows are the channels of HPT heads; every head's product counts for its own D rows only
    f32x4 ox[T];
#pragma unroll
    for (int c = 0; c < T; ++c) {
      ox[c] = f32x4{0.f, 0.f, 0.f, 0.f};
      f32x4 wt[2 * HPT];  // the point's slice weights of the tile's heads
      load_row<HPT * kS>(a.w + (row * H + HPT * c) * kS, g, wt);
#pragma unroll
      for (int q = 0; q < 2 * HPT; ++q) {  // 16 slices of head q / 2
        const float4 e = quad(tokt + (16 * c + i) * (kS + 4) + 16 * (q & 1) + 4 * g);
        const bool own = i / D == q / 2;
#pragma unroll
        for (int j = 0; j < 4; ++j) ox[c] = mma16(own ? at(e, j) : 0.f, wt[q][j], ox[c]);
      }
    }
    // fx1 = out_x W_out^T + b_out + fx_in
#pragma unroll
    for (int c = 0; c < T; ++c) {
      section();
      f32x4 y = fill_from(bo + 16 * c, g);
      product<T>(wo + (16 * c + i) * (C + 4), g, ox, y);
      fx[c] += y;
    }
    f32x4 nt[T], y[T];
    layer_norm<C>(fx, g2, be2, a.ln2_eps, g, nt);
#pragma unroll
    for (int c = 0; c < T; ++c) y[c] = fill_from(b2 + 16 * c, g);
#pragma unroll 2
    for (int f = 0; f < F; f += 16) {
      section();
      f32x4 h[1] = {fill_from(b1 + f, g)};
      product<T>(w1 + (f + i) * (C + 4), g, nt, h[0]);
#pragma unroll
      for (int r = 0; r < 4; ++r) h[0][r] = gelu_erf(h[0][r]);
#pragma unroll
      for (int c = 0; c < T; ++c) product<1>(w2 + (16 * c + i) * (F + 4) + f, g, h, y[c]);
    }
#pragma unroll
    for (int c = 0; c < T; ++c) y[c] += fx[c];
    if (t + step < tiles) load_row<C>(a.fx_in + row_of(t + step) * C, g, fx);
    if (ok) store_row<C>(a.fx_out + row * C, g, y);
    if (!a.ln_out && a.O == 0) continue;
    layer_norm<C>(y, gn, ben, a.next_eps, g, nt);
    if (ok && a.ln_out) store_row<C>(a.ln_out + row * C, g, nt);
    for (int o = 0; o < a.O; ++o) {
      float acc = 0.f;
#pragma unroll
      for (int c = 0; c < T; ++c) {
        const float4 e = quad(hw + o * C + 16 * c + 4 * g);
#pragma unroll
        for (int j = 0; j < 4; ++j) acc = fmaf(nt[c][j], at(e, j), acc);
      }
      acc = group_sum(acc) + (a.head_b ? a.head_b[o] : 0.f);
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

// Waves per workgroup: eight share a staging of the weights, four where a workgroup per CU takes all tiles.
static int waves(const pa_shape &s, int num_cu) { return s.B * ((s.N + 4 * kTilePts - 1) / (4 * kTilePts)) <= num_cu ? 4 : 8; }

// workgroups per batch element: one tile per wave while two workgroups per CU can take them all
int64_t groups(const pa_shape &s, int num_cu) {
  const int64_t per = waves(s, num_cu) * kTilePts, all = (s.N + per - 1) / per, most = (2 * num_cu + s.B - 1) / s.B;
  return all < most ? all : most;
}

template <int C, int D, int W>
static int front_t(const pa_shape &s, const pa_params &p, const void *x, float *w, float *partials, int64_t G, hipStream_t st) {
  const size_t lds = (size_t)Front<C, D, W>::kFloats * 4;
  if (int rc = allow_dynamic_lds(front_kernel<C, D, W>, lds)) return rc;
  hipLaunchKernelGGL((front_kernel<C, D, W>), dim3((unsigned)G, (unsigned)s.B), dim3(64 * W), lds, st,
                     static_cast<const float *>(x), static_cast<const float *>(p.in_project_x_weight), p.in_project_x_bias,
                     static_cast<const float *>(p.in_project_fx_weight), p.in_project_fx_bias,
                     static_cast<const float *>(p.in_project_slice_weight), p.in_project_slice_bias, p.temperature, w, partials,
                     s.N);
  return launch_status();
}

template <int C, int D, int W>
static int tail_t(const pa_shape &s, const TailArgs &a, int64_t G, hipStream_t st) {
  const size_t lds = (size_t)Tail<C, D>::floats(a.F) * 4;
  if (int rc = allow_dynamic_lds(tail_kernel<C, D, W>, lds)) return rc;
  hipLaunchKernelGGL((tail_kernel<C, D, W>), dim3((unsigned)G, (unsigned)s.B), dim3(64 * W), lds, st, a);
  return launch_status();
}

#define PA_NARROW(CALL)                                                                \
  if (waves(s, num_cu) == 4) {                                                         \
    if (s.C == 32) return s.D == 8 ? CALL(32, 8, 4) : CALL(32, 16, 4);                 \
    return s.D == 8 ? CALL(64, 8, 4) : CALL(64, 16, 4);                                \
  }                                                                                    \
  if (s.C == 32) return s.D == 8 ? CALL(32, 8, 8) : CALL(32, 16, 8);                   \
  return s.D == 8 ? CALL(64, 8, 8) : CALL(64, 16, 8)

int front(const pa_shape &s, const pa_params &p, const void *x, float *w, float *partials, int num_cu, hipStream_t st) {
  const int64_t G = groups(s, num_cu);
#define PA_FRONT(CC, DD, WW) front_t<CC, DD, WW>(s, p, x, w, partials, G, st)
  PA_NARROW(PA_FRONT);
#undef PA_FRONT
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
#define PA_TAIL(CC, DD, WW) tail_t<CC, DD, WW>(s, a, G, st)
  PA_NARROW(PA_TAIL);
#undef PA_TAIL
#undef PA_NARROW
}

}  // namespace narrow
}  // namespace pa
