// Per-point stages of a float32 training step with heads of 16 channels and 32 slices (PA.py:106-203, :501-558), a wave to a head
// and tiles of 16 points, operands and intermediates in registers (layouts: pa_narrow_ops.h):
//   point_sums_kernel      slice softmax and token sums; or the sums alone, of given weights and values
//   point_backward_kernel  the adjoints of slice softmax, aggregation and hand-back, with d W_slice, d b_slice, d temperature
// The formulas are those of the general kernels (pa_backward.hip), which serve every other shape.
#include "pa_host.h"
#include "pa_narrow_ops.h"

namespace pa {
namespace narrow {

constexpr int kD = 16;

// Rows of a batch element's 16 points from a base, `rows` of them present: reads past the last row give 0, writes are dropped.
// (A row is `ld` floats; `width` of them from the base on are reached.)
struct Rows {
  __amdgpu_buffer_rsrc_t rsrc;
  __device__ __forceinline__ Rows(const float *base, int rows, int ld, int width) {
    const uint64_t at = reinterpret_cast<uint64_t>(base);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)at), hi = __builtin_amdgcn_readfirstlane((uint32_t)(at >> 32));
    rsrc = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void *>(((uint64_t)hi << 32) | lo), 0,
                                             __builtin_amdgcn_readfirstlane(((rows - 1) * ld + width) * 4), 0x00027000);
  }
  __device__ __forceinline__ f32x4 load4(int at) const {
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, at * 4, 0, 0));
  }
  __device__ __forceinline__ float load(int at) const {
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsrc, at * 4, 0, 0));
  }
  __device__ __forceinline__ void store4(int at, f32x4 v) const {
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(mfma::u32x4, v), rsrc, at * 4, 0, 0);
  }
};

__device__ __forceinline__ f32x4 zero4() { return f32x4{0.f, 0.f, 0.f, 0.f}; }
__device__ __forceinline__ f32x4 quad4(const float *p) { return *reinterpret_cast<const f32x4 *>(p); }

struct SumsArgs {
  const float *x_mid, *v;  // (B, N, H 16) rows: logits' input, values
  const float *w_s, *b_s, *temperature;
  float *w;                // (B, N, H, 32): written, or read (GIVEN)
  float *partials;         // [workgroup][B][H][32][17]
  int64_t N;
  int H;
};

// grid (groups, B, head groups), a wave per head of the group; a wave keeps its head's sums in registers over the tiles
// blockIdx.x, + gridDim.x, ...  Bound by memory (x_mid and v read, w written: 256 bytes a point and head).
// 4 x 7 225 points of eight heads 15.8 us, where a product, a softmax over rows and the general sums took 22 + 12 + 18; with the
// weights given 11.4 against 18.
template <bool GIVEN>
__global__ __launch_bounds__(512, 4) void point_sums_kernel(SumsArgs a) {
  constexpr int LD = kS + 4;
  extern __shared__ float4 lds4[];
  const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int H = a.H, h = blockIdx.z * (blockDim.x >> 6) + wave, b = blockIdx.y, HD = H * kD, HS = H * kS;
  float *turn = reinterpret_cast<float *>(lds4) + wave * kTilePts * LD;
  const int tiles = (int)((a.N + kTilePts - 1) / kTilePts);
  f32x4 ws[2], bias[2];
  float sc = 0.f, sc_low = 0.f;
  if constexpr (!GIVEN) {
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      ws[st] = quad4(a.w_s + (16 * st + i) * kD + 4 * g);
      bias[st] = quad4(a.b_s + 16 * st + 4 * g);
    }
    exponent_scale(clamp_temperature(a.temperature[h]), sc, sc_low);
  }
  f32x4 tok[2] = {zero4(), zero4()};  // lane i <-> channel, registers <-> slices 16 st + 4 g + r
  float nrm[2] = {0.f, 0.f};          // lane i <-> slice 16 st + i, this g's points
  f32x4 x, v, wt[2];                  // v[r], wt[st][r]: point 4 g + r of channel i, of slice 16 st + i
  auto fetch = [&](int t) {
    const int rows = (int)(a.N - (int64_t)t * kTilePts < kTilePts ? a.N - (int64_t)t * kTilePts : kTilePts);
    const int64_t row0 = (int64_t)b * a.N + (int64_t)t * kTilePts;
    const Rows values(a.v + row0 * HD + h * kD, rows, HD, kD);
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = values.load((4 * g + r) * HD + i);
    if constexpr (GIVEN) {
      const Rows weights(a.w + row0 * HS + h * kS, rows, HS, kS);
#pragma unroll
      for (int st = 0; st < 2; ++st)
#pragma unroll
        for (int r = 0; r < 4; ++r) wt[st][r] = weights.load((4 * g + r) * HS + 16 * st + i);
    } else {
      x = Rows(a.x_mid + row0 * HD + h * kD, rows, HD, kD).load4(i * HD + 4 * g);
    }
  };
  fetch(blockIdx.x);  // the grid is no larger than the number of tiles
  for (int t = blockIdx.x; t < tiles; t += gridDim.x) {
    f32x4 now = v, lg[2];
    if constexpr (!GIVEN) {
      float mx = -INFINITY, sum = 0.f;
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        lg[st] = bias[st];
#pragma unroll
        for (int j = 0; j < 4; ++j) lg[st] = mma16(ws[st][j], x[j], lg[st]);
#pragma unroll
        for (int r = 0; r < 4; ++r) mx = fmaxf(mx, lg[st][r]);
      }
      if (t + (int)gridDim.x < tiles) fetch(t + gridDim.x);
      mx = group_max(mx);
#pragma unroll
      for (int st = 0; st < 2; ++st)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          lg[st][r] = exponential(lg[st][r] - mx, sc, sc_low);
          sum += lg[st][r];
        }
      const float inv = 1.f / group_sum(sum);
      const int rows = (int)(a.N - (int64_t)t * kTilePts < kTilePts ? a.N - (int64_t)t * kTilePts : kTilePts);
      const Rows weights(a.w + ((int64_t)b * a.N + (int64_t)t * kTilePts) * HS + h * kS, rows, HS, kS);
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        lg[st] *= inv;
        weights.store4(i * HS + 16 * st + 4 * g, lg[st]);
        *reinterpret_cast<f32x4 *>(turn + i * LD + 16 * st + 4 * g) = i < rows ? lg[st] : zero4();
      }
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int st = 0; st < 2; ++st)
#pragma unroll
        for (int r = 0; r < 4; ++r) lg[st][r] = turn[(4 * g + r) * LD + 16 * st + i];
      __builtin_amdgcn_wave_barrier();  // read before the next tile overwrites them
    } else {
      lg[0] = wt[0], lg[1] = wt[1];
      if (t + (int)gridDim.x < tiles) fetch(t + gridDim.x);
    }
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        nrm[st] += lg[st][r];
        tok[st] = mma16(lg[st][r], now[r], tok[st]);
      }
  }
  float *dst = a.partials + (((int64_t)blockIdx.x * gridDim.y + b) * H + h) * kS * (kD + 1);
#pragma unroll
  for (int st = 0; st < 2; ++st) {
    const float total = group_sum(nrm[st]);
    if (g == 0) dst[(16 * st + i) * (kD + 1) + kD] = total;
#pragma unroll
    for (int r = 0; r < 4; ++r) dst[(16 * st + 4 * g + r) * (kD + 1) + i] = tok[st][r];
  }
}

struct PointBackwardArgs {
  const float *x_mid, *fx_mid, *g;                      // (B, N, H 16) rows; g = d out_x
  const float *out_token, *d_num, *d_norm;              // (B, H, 32, 16), the same, (B, H, 32)
  const float *w_s, *b_s, *temperature;
  float *d_proj;                                        // (B, N, 2 H 16): d x_mid, d fx_mid
  float *partials;                                      // [workgroup] d W_slice (32, 16), d b_slice (32), d temperature (H)
  int64_t N;
  int H;
};

// grid as above.  The products of a tile (A . B, the tile's points as columns unless noted):
//   z^T = W_s x^T + b,  d w^T = tok' g^T + d num fx^T + d nrm,  d fx^T = d num^T w^T,  d x^T = W_s^T d z^T,
//   d W_s (slices x channels, reduction over the points) = d z^T x, both turned around in LDS
// Bound by matrix and vector issue in equal parts, which do not overlap for float32, and the memory time of 320 bytes a point and
// head close behind.  4 x 7 225 points of eight heads 27 us; the general kernel, which also reads w and writes d z, 81, and the product
// over the points that formed d W_slice from them 31 more.
__global__ __launch_bounds__(512, 4) void point_backward_kernel(PointBackwardArgs a) {
  constexpr int LD = kTilePts + 4, OUT = kS * kD + kS;
  static_assert(kD == kTilePts && OUT + 1 <= (kS + kTilePts) * LD, "rows of LD floats; a wave's results fit its tiles' place");
  extern __shared__ float4 lds4[];
  float *lds = reinterpret_cast<float *>(lds4);
  const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
  const int H = a.H, h = blockIdx.z * waves + wave, b = blockIdx.y, HD = H * kD;
  float *turn_z = lds + wave * (kS + kTilePts) * LD, *turn_x = turn_z + kS * LD;  // [slice][point], [point][channel]
  const int tiles = (int)((a.N + kTilePts - 1) / kTilePts);
  const int64_t bh = (int64_t)b * H + h;
  // W_s rows and b in LDS, the other tables of the head in registers
  float *ws = lds + waves * (kS + kTilePts) * LD, *bs = ws + kS * LD;
  for (int e = threadIdx.x; e < kS * kD; e += blockDim.x) ws[e / kD * LD + e % kD] = a.w_s[e];
  if (threadIdx.x < kS) bs[threadIdx.x] = a.b_s[threadIdx.x];
  f32x4 wst[2], to[2], dn[2], dnt[2], dnr[2];
#pragma unroll
  for (int st = 0; st < 2; ++st) {
    const int s = 16 * st + i, s4 = 16 * st + 4 * g;
    to[st] = quad4(a.out_token + (bh * kS + s) * kD + 4 * g);
    dn[st] = quad4(a.d_num + (bh * kS + s) * kD + 4 * g);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      wst[st][r] = a.w_s[(s4 + r) * kD + i];
      dnt[st][r] = a.d_num[(bh * kS + s4 + r) * kD + i];
    }
    dnr[st] = quad4(a.d_norm + bh * kS + s4);
  }
  const float raw = a.temperature[h], inv_temp = uniform(1.f / clamp_temperature(raw));
  float sc, sc_low;
  exponent_scale(clamp_temperature(raw), sc, sc_low);
  f32x4 dws[2] = {zero4(), zero4()}, dbs[2] = {zero4(), zero4()};
  float dt = 0.f;
  f32x4 x, f, go;
  auto fetch = [&](int t) {
    const int rows = (int)(a.N - (int64_t)t * kTilePts < kTilePts ? a.N - (int64_t)t * kTilePts : kTilePts);
    const int64_t at = ((int64_t)b * a.N + (int64_t)t * kTilePts) * HD + h * kD;
    x = Rows(a.x_mid + at, rows, HD, kD).load4(i * HD + 4 * g);
    f = Rows(a.fx_mid + at, rows, HD, kD).load4(i * HD + 4 * g);
    go = Rows(a.g + at, rows, HD, kD).load4(i * HD + 4 * g);
  };
  fetch(blockIdx.x);  // the grid is no larger than the number of tiles
  __syncthreads();
  for (int t = blockIdx.x; t < tiles; t += gridDim.x) {
    const int rows = (int)(a.N - (int64_t)t * kTilePts < kTilePts ? a.N - (int64_t)t * kTilePts : kTilePts);
    f32x4 w[2], dw[2];
    float mx = -INFINITY, sum = 0.f, dot = 0.f, mean = 0.f;
    section();
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      const f32x4 wrow = quad4(ws + (16 * st + i) * LD + 4 * g);
      f32x4 part = zero4();  // sums of their own: shorter chains of roundings
      w[st] = quad4(bs + 16 * st + 4 * g);
      dw[st] = dnr[st];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        w[st] = mma16(wrow[j], x[j], w[st]);
        dw[st] = mma16(to[st][j], go[j], dw[st]);
        part = mma16(dn[st][j], f[j], part);
      }
      dw[st] += part;
#pragma unroll
      for (int r = 0; r < 4; ++r) mx = fmaxf(mx, w[st][r]);
    }
    *reinterpret_cast<f32x4 *>(turn_x + i * LD + 4 * g) = x;
    if (t + (int)gridDim.x < tiles) fetch(t + gridDim.x);
    mx = group_max(mx);
    f32x4 z[2];  // z - max z; d temperature takes it from its weighted mean, as in the general kernel
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float arg = w[st][r] - mx;
        w[st][r] = exponential(arg, sc, sc_low);
        z[st][r] = fmaxf(arg, -FLT_MAX);  // 0 z is 0 for a slice of no weight; a NaN is in w
        sum += w[st][r];
        dot = fmaf(w[st][r], dw[st][r], dot);
        mean = fmaf(w[st][r], z[st][r], mean);
      }
    const float inv = 1.f / group_sum(sum);
    dot = group_sum(dot) * inv;
    mean = group_sum(mean) * inv;
    f32x4 dx[2] = {zero4(), zero4()}, df[2] = {zero4(), zero4()};
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        w[st][r] *= inv;
        df[st] = mma16(dnt[st][r], w[st][r], df[st]);
        const float dl = i < rows ? w[st][r] * (dw[st][r] - dot) : 0.f;
        dt = fmaf(dl, z[st][r] - mean, dt);
        const float dz = dl * inv_temp;
        dbs[st][r] += dz;
        dx[st] = mma16(wst[st][r], dz, dx[st]);
        turn_z[(16 * st + 4 * g + r) * LD + i] = dz;
      }
    const Rows out(a.d_proj + (((int64_t)b * a.N + (int64_t)t * kTilePts) * 2 * H + h) * kD, rows, 2 * HD, HD + kD);
    out.store4(i * 2 * HD + 4 * g, dx[0] + dx[1]);
    out.store4(i * 2 * HD + HD + 4 * g, df[0] + df[1]);
    __builtin_amdgcn_wave_barrier();
    f32x4 xt;
#pragma unroll
    for (int r = 0; r < 4; ++r) xt[r] = turn_x[(4 * g + r) * LD + i];
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      const f32x4 zt = quad4(turn_z + (16 * st + i) * LD + 4 * g);
#pragma unroll
      for (int r = 0; r < 4; ++r) dws[st] = mma16(zt[r], xt[r], dws[st]);
    }
    __builtin_amdgcn_wave_barrier();  // read before the next tile overwrites them
  }
  // over the 16 lanes of a row of lanes
  auto row_sum = [](float v) {
    auto step = [](float y, auto ctrl) {
      return y + __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(y), decltype(ctrl)::value, 0xf, 0xf, true));
    };
    v = step(v, std::integral_constant<int, 0xB1>{});   // quad_perm [1,0,3,2]
    v = step(v, std::integral_constant<int, 0x4E>{});   // quad_perm [2,3,0,1]
    v = step(v, std::integral_constant<int, 0x141>{});  // row_half_mirror
    return step(v, std::integral_constant<int, 0x140>{});  // row_mirror
  };
  __syncthreads();  // the tiles in LDS are done with
  float *mine = lds + wave * (OUT + 1);
#pragma unroll
  for (int st = 0; st < 2; ++st)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int s = 16 * st + 4 * g + r;
      mine[s * kD + i] = dws[st][r];
      const float v = row_sum(dbs[st][r]);
      if (i == 0) mine[kS * kD + s] = v;
    }
  const float total = group_sum(row_sum(dt));
  if (lane == 0) mine[OUT] = raw >= kTempMin && raw <= kTempMax ? -total * inv_temp * inv_temp : 0.f;
  __syncthreads();
  float *dst = a.partials + (((int64_t)blockIdx.z * gridDim.y + b) * gridDim.x + blockIdx.x) * (OUT + H);
  for (int e = threadIdx.x; e < OUT + H; e += blockDim.x) {
    float v = 0.f;
    if (e < OUT) {
      for (int u = 0; u < waves; ++u) v += lds[u * (OUT + 1) + e];
    } else {
      const int u = e - OUT - (int)blockIdx.z * waves;  // the group's heads; the others are other workgroups'
      if (u >= 0 && u < waves) v = lds[u * (OUT + 1) + OUT];
    }
    dst[e] = v;
  }
}

bool points_supported(const pa_shape &s) { return s.S == kS && s.D == kD && (s.H <= 8 || s.H % 8 == 0) && s.B <= 65535; }

// Workgroups (of up to eight heads) per batch element: four waves per SIMD, no more than there are tiles.
static void points_grid(const pa_shape &s, int num_cu, dim3 *grid, dim3 *block) {
  const int waves = (int)(s.H < 8 ? s.H : 8);
  const int64_t sets = s.H / waves, tiles = (s.N + kTilePts - 1) / kTilePts;
  int64_t gx = ((int64_t)num_cu * (16 / waves) + s.B * sets - 1) / (s.B * sets);
  if (gx > tiles) gx = tiles;
  *grid = dim3((unsigned)gx, (unsigned)s.B, (unsigned)sets);
  *block = dim3((unsigned)(64 * waves));
}

int64_t point_groups(const pa_shape &s, int num_cu) {
  dim3 grid, block;
  points_grid(s, num_cu, &grid, &block);
  return grid.x;
}
int64_t point_backward_rows(const pa_shape &s, int num_cu) {
  dim3 grid, block;
  points_grid(s, num_cu, &grid, &block);
  return (int64_t)grid.x * grid.y * grid.z;
}

int point_sums(const pa_shape &s, const pa_params *p, const float *x_mid, const float *v, float *w, float *partials, int num_cu,
               hipStream_t st) {
  SumsArgs a{};
  a.x_mid = x_mid, a.v = v, a.w = w, a.partials = partials, a.N = s.N, a.H = (int)s.H;
  dim3 grid, block;
  points_grid(s, num_cu, &grid, &block);
  if (!p) {
    hipLaunchKernelGGL((point_sums_kernel<true>), grid, block, 0, st, a);
    return launch_status();
  }
  a.w_s = static_cast<const float *>(p->in_project_slice_weight), a.b_s = p->in_project_slice_bias, a.temperature = p->temperature;
  hipLaunchKernelGGL((point_sums_kernel<false>), grid, block, block.x / 64 * kTilePts * (kS + 4) * 4, st, a);
  return launch_status();
}

int point_backward(const pa_shape &s, const pa_params &p, const float *x_mid, const float *fx_mid, const float *g,
                   const float *out_token, const float *d_num, const float *d_norm, float *d_proj, float *partials, int num_cu,
                   hipStream_t st) {
  const PointBackwardArgs a{x_mid, fx_mid, g, out_token, d_num, d_norm, static_cast<const float *>(p.in_project_slice_weight),
                            p.in_project_slice_bias, p.temperature, d_proj, partials, s.N, (int)s.H};
  dim3 grid, block;
  points_grid(s, num_cu, &grid, &block);
  const size_t lds = (block.x / 64 * (kS + kTilePts) * (kTilePts + 4) + kS * (kTilePts + 4) + kS) * 4;
  hipLaunchKernelGGL(point_backward_kernel, grid, block, lds, st, a);
  return launch_status();
}

}  // namespace narrow
}  // namespace pa
