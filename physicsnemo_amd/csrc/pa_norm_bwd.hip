// Input gradient of a Linear that follows a LayerNorm, and the LayerNorm's backward, in one pass over the rows (gfx950 MFMA,
// bf16 rows of 256 channels): for n = LayerNorm(x) gamma + beta, h = W n + .. and dh given,
//   g = dh W   (the gradient of n, rounded to bf16 as the separate product leaves it)
//   dx = add + rstd (g gamma - mean_c(g gamma) - xh mean_c(g gamma xh)),  d gamma = sum_rows g xh,  d beta = sum_rows g
// so that g is neither written nor read back (2 x 512 bytes per row).
#include "pa_host.h"
#include "pa_mfma_ops.h"

namespace pa {
namespace norm {

using mfma::f32x16;
using mfma::half_wave_sum;
using mfma::load_unit_to_lds;
using mfma::mma;
using mfma::pack2;
using mfma::static_for;
using mfma::u32x2;
using mfma::u32x4;

struct Args {
  const uint16_t *dh, *wt, *x, *add;  // (M, K), (256, K): W^T, (M, 256), (M, 256)
  const float *gamma;
  uint16_t *dx;
  float *partials;  // [workgroup][2][256]
  float eps;
  int64_t M, nblocks;
  int K;
};

// ---------------------------------------------------------------------------------------------------------------
// rows_ln_backward_kernel.  Workgroup = 8 waves, two workgroups per CU, so that one's LayerNorm rows run beside the other's
// product; a block is ROWS rows x 256 outputs, a wave's tile 64 x (ROWS / 2) of them.  Steps of 32 reduction indices of dh and
// of W^T (rows of 64 bytes) form a ring of three stages in LDS, filled two steps ahead by direct global -> LDS loads, one
// barrier per step.  Position p of row r holds the row's 16-byte unit p ^ (r / 4 % 4): the lanes of an access phase fall on all
// banks.  g leaves the accumulators through LDS in bf16; half a wave then finishes a row as layernorm_backward_rows_kernel does.
// Bound by the reach of the ring (24 KB a step and workgroup, W^T two thirds of it) at K = 1 024, by HBM below (2 K + 1 536 bytes
// per row).  262 144 rows (us), the product and layernorm_backward_rows_kernel -> this: K = 1 024 149 + 99 -> 231, K = 512 96 +
// 102 -> 149 (the best of 15 launches each), K = 256 94 less in all.  dh as register operands straight from memory instead: 280 at
// K = 1 024, its 16-byte pieces of rows coming from L2 four times.
// ---------------------------------------------------------------------------------------------------------------
template <int ROWS>
struct Tile {
  static constexpr int RT = 2, OT = ROWS / 64, STAGE = (ROWS + 256) * 64, STAGES = 3, LD = 256 + 8;
  static constexpr int BYTES = STAGES * STAGE > ROWS * LD * 2 ? STAGES * STAGE : ROWS * LD * 2;
};

template <int ROWS>
__global__ __launch_bounds__(512, 4) void rows_ln_backward_kernel(Args a) {
  using Q = Tile<ROWS>;
  constexpr int C = 256, RT = Q::RT, OT = Q::OT, LD = Q::LD, RPW = ROWS / 8;  // RPW: rows a wave finishes
  extern __shared__ u32x4 smem[];
  uint16_t *stage = reinterpret_cast<uint16_t *>(smem);  // behind the steps of a block: its rows of g
  float *gammas = reinterpret_cast<float *>(reinterpret_cast<char *>(smem) + Q::BYTES);
  const int tid = threadIdx.x, lane = tid & 63, i = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = ROWS == 128 ? (wave & 1) * 64 : 0, wc = ROWS == 128 ? (wave >> 1) * 64 : wave * 32;
  const int K = a.K, nkb = K / 32;
  // a wave fetches 16 rows of dh (ROWS = 64: two waves the same ones) and 32 of W^T per step, a lane unit lane % 4 of its row
  const int frow = lane >> 2, unit = 8 * ((lane & 3) ^ ((frow >> 2) & 3)), arow = 16 * (ROWS == 128 ? wave : wave & 3);
  const uint16_t *wsrc = a.wt + (int64_t)(32 * wave + frow) * K + unit;
  if (tid < C) gammas[tid] = a.gamma[tid];  // read behind the first block's barriers
  float dg[8], db[8];                       // of channels 8 i .. + 7
#pragma unroll
  for (int e = 0; e < 8; ++e) dg[e] = db[e] = 0.f;

  for (int64_t mb = blockIdx.x; mb < a.nblocks; mb += gridDim.x) {
    const int64_t row0 = mb * ROWS;
    const int have = (int)(a.M - row0 < ROWS ? a.M - row0 : ROWS);
    const uint16_t *asrc = a.dh + (row0 + (arow + frow < have ? arow + frow : have - 1)) * K + unit;  // past the last row: that one
    auto fetch = [&](int kb) {  // past the last step: that one again, so that every step counts three loads
      const int k = 32 * (kb < nkb ? kb : nkb - 1);
      const unsigned dst = (unsigned)(uintptr_t)smem + (unsigned)(kb % Q::STAGES) * Q::STAGE;
      load_unit_to_lds(asrc + k, dst + arow * 64);
      load_unit_to_lds(wsrc + k, dst + ROWS * 64 + 32 * wave * 64);
      load_unit_to_lds(wsrc + (int64_t)16 * K + k, dst + ROWS * 64 + (32 * wave + 16) * 64);
    };
    f32x16 acc[OT][RT];
#pragma unroll
    for (int u = 0; u < OT; ++u)
#pragma unroll
      for (int v = 0; v < RT; ++v)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[u][v][r] = 0.f;
    __syncthreads();  // the rows of the block before are finished
    fetch(0);
    fetch(1);
    const int swz = (i >> 2) & 3;
#pragma clang loop unroll(disable)
    for (int kb = 0; kb < nkb; ++kb) {
      asm volatile("s_waitcnt vmcnt(3)" ::: "memory");  // this wave's share of the step; the next one stays in flight
      __syncthreads();
      fetch(kb + 2);  // into the stage multiplied one step ago, which every wave is past
      const u32x4 *xs = smem + (kb % Q::STAGES) * (Q::STAGE / 16) + (wr + i) * 4;
      const u32x4 *ws = smem + (kb % Q::STAGES) * (Q::STAGE / 16) + (ROWS + wc + i) * 4;
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const int at = (2 * ks + g) ^ swz;
        u32x4 w[OT], x[RT];
#pragma unroll
        for (int u = 0; u < OT; ++u) w[u] = ws[32 * 4 * u + at];
#pragma unroll
        for (int v = 0; v < RT; ++v) x[v] = xs[32 * 4 * v + at];
#pragma unroll
        for (int u = 0; u < OT; ++u)
#pragma unroll
          for (int v = 0; v < RT; ++v) acc[u][v] = mma(w[u], x[v], acc[u][v]);
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing is landing in the ring any more
    __syncthreads();

    // ---- g to bf16 rows in LDS, then the LayerNorm's backward: half a wave per row, eight channels per lane ----
    int il = i, hl = g;  // taken afresh: nothing derived from them is kept across the steps
    asm volatile("" : "+v"(il), "+v"(hl));
#pragma unroll
    for (int u = 0; u < OT; ++u)
#pragma unroll
      for (int v = 0; v < RT; ++v)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *reinterpret_cast<u32x2 *>(stage + (wr + 32 * v + il) * LD + wc + 32 * u + 8 * q + 4 * hl) =
              u32x2{pack2(acc[u][v][4 * q], acc[u][v][4 * q + 1]), pack2(acc[u][v][4 * q + 2], acc[u][v][4 * q + 3])};
    // buffer accesses end at the last row by themselves
    auto rows_of = [&](const uint16_t *p) {
      return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(p) + row0 * C, 0, have * C * 2, 0x00027000);
    };
    constexpr int STREAM = 2, NIT = RPW / 2, PF = NIT < 4 ? NIT : 4;  // STREAM: the non-temporal hint
    u32x4 xv[NIT], av[NIT];
    auto load = [&](auto it_) {
      constexpr int it = decltype(it_)::value;
      const int at = ((wave * RPW + 2 * it + hl) * C + 8 * il) * 2;
      xv[it] = __builtin_amdgcn_raw_buffer_load_b128(rows_of(a.x), at, 0, STREAM);
      av[it] = __builtin_amdgcn_raw_buffer_load_b128(rows_of(a.add), at, 0, STREAM);
    };
    static_for<PF>(load);
    __syncthreads();
    static_for<NIT>([&](auto it_) {
      constexpr int it = decltype(it_)::value;
      if constexpr (it + PF < NIT) load(std::integral_constant<int, it + PF>{});
      const int rw = wave * RPW + 2 * it + hl;
      const bool ok = rw < have;
      const u32x4 gs = *reinterpret_cast<const u32x4 *>(stage + rw * LD + 8 * il);
      float xf[8], gf[8], sum = 0.f;
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        xf[2 * w] = __uint_as_float(xv[it][w] << 16), xf[2 * w + 1] = __uint_as_float(xv[it][w] & 0xffff0000u);
        gf[2 * w] = ok ? __uint_as_float(gs[w] << 16) : 0.f, gf[2 * w + 1] = ok ? __uint_as_float(gs[w] & 0xffff0000u) : 0.f;
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) sum += xf[e];
      const float mean = half_wave_sum(sum) * (1.f / C);
      float sq = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float d = xf[e] - mean;
        sq = fmaf(d, d, sq);
      }
      const float every = rsqrtf(half_wave_sum(sq) * (1.f / C) + a.eps), rstd = ok ? every : 0.f;
      float s1 = 0.f, s2 = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float xh = (xf[e] - mean) * rstd, d = gf[e], gg = d * gammas[8 * il + e];
        dg[e] = fmaf(d, xh, dg[e]);
        db[e] += d;
        xf[e] = xh, gf[e] = gg;
        s1 += gg;
        s2 = fmaf(gg, xh, s2);
      }
      s1 = half_wave_sum(s1) * (1.f / C);
      s2 = half_wave_sum(s2) * (1.f / C);
      u32x4 out;
#pragma unroll
      for (int w = 0; w < 4; ++w)
        out[w] = pack2(fmaf(rstd, gf[2 * w] - s1 - xf[2 * w] * s2, __uint_as_float(av[it][w] << 16)),
                       fmaf(rstd, gf[2 * w + 1] - s1 - xf[2 * w + 1] * s2, __uint_as_float(av[it][w] & 0xffff0000u)));
      __builtin_amdgcn_raw_buffer_store_b128(out, rows_of(a.dx), (rw * C + 8 * il) * 2, 0, STREAM);
      __builtin_amdgcn_sched_barrier(0);
    });
  }
  __syncthreads();
  float *red = reinterpret_cast<float *>(smem);  // [wave][2][256]
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float vg = dg[e] + __shfl_xor(dg[e], 32, 64), vb = db[e] + __shfl_xor(db[e], 32, 64);
    if (g == 0) red[(wave * 2 + 0) * C + 8 * i + e] = vg, red[(wave * 2 + 1) * C + 8 * i + e] = vb;
  }
  __syncthreads();
  float v = 0.f;
#pragma unroll
  for (int w = 0; w < 8; ++w) v += red[w * 2 * C + tid];
  a.partials[(int64_t)blockIdx.x * 2 * C + tid] = v;
}

bool rows_ln_backward_supported(int64_t rows, int64_t C, int64_t K) { return rows > 0 && C == 256 && K >= 64 && K % 32 == 0; }

// rows of a block: 64 spread 30 000 rows over all workgroups (41 us at K = 1 024), 128 take W^T half as often per row
static int block_rows(int64_t rows, int num_cu) { return rows > (int64_t)128 * num_cu ? 128 : 64; }

int64_t rows_ln_backward_groups(int64_t rows, int num_cu) {
  const int64_t per = block_rows(rows, num_cu), blocks = (rows + per - 1) / per;
  return blocks < 2 * num_cu ? blocks : 2 * num_cu;
}

template <int ROWS>
static int launch(const Args &a, int64_t groups, hipStream_t st) {
  const size_t lds = Tile<ROWS>::BYTES + 256 * 4;
  if (int rc = allow_dynamic_lds(rows_ln_backward_kernel<ROWS>, lds)) return rc;
  hipLaunchKernelGGL(rows_ln_backward_kernel<ROWS>, dim3((unsigned)groups), dim3(512), lds, st, a);
  return launch_status();
}

// partials: rows_ln_backward_groups(rows) * 512 floats; grads: d gamma (256), d beta (256)
int rows_ln_backward(int64_t rows, int64_t K, const void *dh, const void *wt, const void *x, const float *gamma, float eps,
                     const void *add, void *dx, float *partials, float *grads, int num_cu, hipStream_t st, wgrad::Sums &later) {
  const int64_t per = block_rows(rows, num_cu), groups = rows_ln_backward_groups(rows, num_cu);
  auto in = [](const void *p) { return static_cast<const uint16_t *>(p); };
  const Args a{in(dh), in(wt), in(x), in(add), gamma, static_cast<uint16_t *>(dx), partials, eps, rows, (rows + per - 1) / per, (int)K};
  const int rc = per == 128 ? launch<128>(a, groups, st) : launch<64>(a, groups, st);
  if (!rc) later.add(partials, grads, 512, groups);
  return rc;
}

}  // namespace norm
}  // namespace pa
