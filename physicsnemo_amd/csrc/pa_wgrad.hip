// Weight gradients: products over the row axis  P[oa][ob] = sum_m A[m][oa] B[m][ob]  with A = d out, B = the layer's
// input (or, for a grid convolution, its neighbours: one product per tap), plus the column sums of A (the bias
// gradient).  The row axis is cut into chunks, each leaves one partial result, and one small kernel adds the partials up
// in a fixed order, so results do not depend on the launch.
//
//   wgrad_kernel          bf16, up to 256 x 256 of P per workgroup, operands staged by direct global -> LDS loads
//   narrow_wgrad_kernel   one side with at most 16 columns (input features, output channels), bf16 or fp32
//   sum_partials_kernel   the fixed-order total, for several results in one launch
// The fp32 tile kernel (cols_gemm_f32_kernel) and the narrower bf16 one (cols_gemm_kernel) are in pa_gemm.hip.
#include "pa_common.h"
#include "pa_host.h"
#include "pa_mfma_ops.h"

namespace pa {
namespace wgrad {

using mfma::f32x16;
using mfma::load_unit_to_lds;
using mfma::u32x2;
using mfma::u32x4;

// ------------------------------------------------------------------------------------------------
// wgrad_kernel: a workgroup (8 waves, 4 along A's columns x 2 along B's, wave tile 64 x 128) owns a 256 x 256 block of P
// for its chunk of rows.  32 rows of both operands (32 KB) are one stage; four stages form a ring in LDS, filled by
// global_load_lds three stages ahead (96 KB in flight per CU, which is what the memory latency asks for at this rate),
// one barrier per stage.  A lane receives its operand -- eight consecutive rows of one column -- from two transposing
// reads (ds_read_b64_tr_b16: within a group of 16 lanes, lane l receives element l % 4 of what lanes l / 4, 4 + l / 4,
// 8 + l / 4, 12 + l / 4 address).  The direct loads write 1 KB contiguously, so the rows cannot be padded apart;
// instead position p of row r holds the 16-byte unit p ^ 4 (r % 4), which puts the four rows a half-wave reads on four
// different quarters of the banks.
// Workgroups that share a chunk of rows (the blocks of columns, the taps) are placed on the same XCD next to each
// other, so that the operand they share is read from memory once.
// Bound by HBM, 2 (OA + OB) bytes per row, where P is one or two blocks: 512 x 256 over 1 048 576 rows 0.35 ms = 4.6 TB/s
// (the copy of 1 GiB reaches 5.1); with register staging one stage ahead and twice the workgroups it took 0.44 ms.
// A 3 x 3 convolution's 512 x 256 x 9 over 32 768 grid points: 109 us (im2col and the GEMM library: 590 us).
// ------------------------------------------------------------------------------------------------
constexpr int kStages = 4, kStageBytes = 32 * 1024;

struct Args {
  const uint16_t *A, *B;
  int lda, ldb, OA, OB;
  int64_t M;
  int per;             // 32-row blocks per chunk
  int chunks, batches; // row chunks (of each batch element, 1 unless A is packed)
  int ny, nz;          // 256-column blocks of A; (tap, 256-column block of B)
  float *partials;     // [chunk][OA][taps][OB]
  float *col_sums;     // [chunk][OA] or NULL
  GridTaps grid;       // grid convolution: B's row for point m and a tap is the neighbour there, zero outside the grid
  // packed A (the slice weights of the MFMA kernels): [batch][tile of 32 points][chunk of 16 columns][lane] 16 bytes, the
  // chunk's lane (point p, half g) holding columns 4 g .. + 3 and 8 + 4 g .. + 3; chunks and M count per batch then
  const u32x4 *pack;
  int tpb, tile_units;  // tiles per batch, 16-byte units of a tile
};

// MODE 0: A and B are rows.  1: B gathered per tap of a convolution.  2: A packed, batch by batch; the chunks of a stage
// are copied as they lie, the 16-byte units permuted within a chunk so that the transposing reads of a half-wave (4
// points x 4 groups of slices x 2 chunks) fall on all banks: unit (p, g) of chunk c at position 32 g + (p ^ 4 g ^ 8 (c & 1)).
// Slice weights of points beyond N are zero, so B's rows there only need to be readable; col_sums are B's columns.
template <int MODE>
__global__ __launch_bounds__(512) void wgrad_kernel(Args a) {
  constexpr bool CONV = MODE == 1, PACKED = MODE == 2;
  typedef short v4i16 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) v4i16 *lds_v4i16;
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  extern __shared__ u32x4 ring[];  // [stage][A 32 rows x 512 bytes | B 32 rows x 512 bytes]
  const int t = threadIdx.x, lane = t & 63, i = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wa = (wave & 3) * 64, wb = (wave >> 2) * 128;
  // the (chunk, tile) pairs in chunk-major order are dealt out to the XCDs (= workgroup id mod 8) in eight equal runs
  const int tiles = a.ny * a.nz, item = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  const int chunk = item / tiles, tile = item - chunk * tiles;
  if (chunk >= a.chunks * a.batches) return;
  const int oa0 = (tile % a.ny) * 256, zt = tile / a.ny, nob = (a.OB + 255) / 256;
  const int tap = CONV ? zt / nob : 0, ob0 = (CONV ? zt % nob : zt) * 256;
  const int batch = PACKED ? chunk / a.chunks : 0;
  const int64_t nblk = (a.M + 31) / 32, blk0 = (int64_t)(chunk - batch * a.chunks) * a.per;
  const int64_t blk1 = blk0 + a.per < nblk ? blk0 + a.per : nblk;

  f32x16 acc[2][4];
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int v = 0; v < 4; ++v)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[u][v][r] = 0.f;
  float csum[4] = {0.f, 0.f, 0.f, 0.f};
  const bool sums = a.col_sums != nullptr && (PACKED ? oa0 == 0 && wa == 0 : zt == 0 && wb == 0);

  // this wave stages rows 4 wave .. + 3 of both operands, two rows per load: lane l carries position l % 32 of row
  // 4 wave + 2 k + l / 32, i.e. unit (l % 32) ^ 4 (row % 4); units past the operand's last column re-read its first one
  int ua[2], ub[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int unit = i ^ (4 * (2 * k + g));
    ua[k] = oa0 + unit * 8 < a.OA ? oa0 + unit * 8 : oa0;
    ub[k] = ob0 + unit * 8 < a.OB ? ob0 + unit * 8 : ob0;
  }
  const unsigned lds0 = (unsigned)(uintptr_t)ring + wave * 2048;
  // Convolution: the neighbour of row m at this tap is row m + shift where it lies inside the grid.  The grid coordinates
  // of a lane's two rows are divided out once and then advanced by the 32 rows of a stage with carries.
  int ci[2], cj[2], cl[2], du = 0, dv = 0, dz = 0, si = 0, sj = 0, sl = 0;
  int64_t shift = 0;
  const int gw = a.grid.gw, gh = a.grid.gh, gd = a.grid.gd > 0 ? a.grid.gd : 1;
  if constexpr (CONV) {
    const int ksd = a.grid.gd > 0 ? a.grid.ks : 1, uv = tap / ksd, pad = a.grid.ks / 2;
    du = uv / a.grid.ks - pad, dv = uv % a.grid.ks - pad, dz = a.grid.gd > 0 ? tap % ksd - pad : 0;
    shift = ((int64_t)du * gw + dv) * gd + dz;
    si = 32 / (gw * gd), sj = 32 / gd % gw, sl = 32 % gd;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      int n = (int)((blk0 * 32 + wave * 4 + 2 * k + g) % a.grid.N);
      cl[k] = n % gd;
      n /= gd;
      ci[k] = n / gw;
      cj[k] = n - ci[k] * gw;
    }
  }
  const uint16_t *pa[2], *pb[2];
  auto fetch = [&](int64_t blk) {  // past the chunk's end: its last block again, so that every stage counts four loads
    const unsigned dst = lds0 + (unsigned)((blk - blk0) & (kStages - 1)) * kStageBytes;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      if (blk < blk1) {
        const int64_t m = blk * 32 + wave * 4 + 2 * k + g, mc = m < a.M ? m : a.M - 1;
        if constexpr (PACKED) {
          const int c = 2 * wave + k, cs = oa0 + 16 * c < a.OA ? oa0 / 16 + c : oa0 / 16;
          pa[k] = reinterpret_cast<const uint16_t *>(a.pack + ((int64_t)batch * a.tpb + blk) * a.tile_units + cs * 64 +
                                                     32 * g + (i ^ (4 * g) ^ (8 * k)));
        } else {
          pa[k] = a.A + mc * a.lda + ua[k];
        }
        pb[k] = a.B + ((int64_t)batch * a.M + mc) * a.ldb + ub[k];
        if constexpr (CONV) {
          const int ii = ci[k] + du, jj = cj[k] + dv, ll = cl[k] + dz;
          const bool in = m < a.M && (unsigned)ii < (unsigned)gh && (unsigned)jj < (unsigned)gw && (unsigned)ll < (unsigned)gd;
          pb[k] = in ? pb[k] + shift * a.ldb : reinterpret_cast<const uint16_t *>(&mfma::kZeroUnit);
          cl[k] += sl;
          cj[k] += sj;
          ci[k] += si;
          if (cl[k] >= gd) cl[k] -= gd, ++cj[k];
          if (cj[k] >= gw) cj[k] -= gw, ++ci[k];
          while (ci[k] >= gh) ci[k] -= gh;
        }
      }
      load_unit_to_lds(pa[k], dst + k * 1024);
      load_unit_to_lds(pb[k], dst + 16384 + k * 1024);
    }
  };
  // reads: rows 16 ks + 8 g + l16 / 4 (+ 4); 16-byte units of 8 columns, see above
  const int l16 = lane & 15, q1 = (lane >> 4) & 1, rr = l16 >> 2;
  const int row_off = (8 * g + rr) * 512 + 32 * q1 + 8 * (l16 & 3);
  auto operand = [&](const char *base, int ks, int col) {  // rows 16 ks + 8 g .. + 7 of column col + lane % 32
    const char *p = base + row_off + 16 * ks * 512 + 64 * ((col >> 5) ^ rr);
    const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16)(uintptr_t)p));
    const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16)(uintptr_t)(p + 4 * 512)));
    return u32x4{lo[0], lo[1], hi[0], hi[1]};
  };
  // packed A: points 16 ks + 8 g + l16 / 4 (+ 4), group l16 % 4 of the chunk's four groups of four slices
  const int gu = l16 & 1, pk_base = q1 * 1024 + 512 * gu + 8 * ((l16 >> 1) & 1) + 16 * ((8 * (g ^ q1)) + rr);
  auto packed_operand = [&](const char *base, int ks, int col) {
    const char *p = base + (col >> 4) * 1024 + 256 * ks + pk_base;
    const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16)(uintptr_t)(p + 64 * gu)));
    const u32x2 hi =
        __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16)(uintptr_t)(p + 64 * (1 ^ gu))));
    return u32x4{lo[0], lo[1], hi[0], hi[1]};
  };
  const bf16x2 ones = {(__bf16)1.f, (__bf16)1.f};
  auto masked = [&](u32x4 v, int ks, int valid) {  // rows >= valid of a 32-row block to zero
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int r = 16 * ks + 8 * g + 2 * j;
      const uint32_t word = v[j];
      v[j] = r + 1 < valid ? word : r < valid ? (word & 0xffffu) : 0u;
    }
    return v;
  };
  auto add_columns = [&](u32x4 v, float &s) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t word = v[j];
      s = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, word), ones, s, false);
    }
  };

  if (blk0 < blk1) {
    fetch(blk0);
    fetch(blk0 + 1);
    fetch(blk0 + 2);
  }
  for (int64_t blk = blk0; blk < blk1; ++blk) {
    asm volatile("s_waitcnt vmcnt(8)" ::: "memory");  // this wave's share of the stage; the two younger stay in flight
    __syncthreads();
    fetch(blk + 3);  // into the stage multiplied one step ago, which every wave is past
    const char *at = reinterpret_cast<const char *>(ring) + ((blk - blk0) & (kStages - 1)) * kStageBytes;
    const char *bt = at + 16384;
    const int valid = (int)(a.M - blk * 32 < 32 ? a.M - blk * 32 : 32);  // rows of this block
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      u32x4 af[2], bf[4];
#pragma unroll
      for (int u = 0; u < 2; ++u) af[u] = PACKED ? packed_operand(at, ks, wa + 32 * u) : operand(at, ks, wa + 32 * u);
#pragma unroll
      for (int v = 0; v < 4; ++v) bf[v] = operand(bt, ks, wb + 32 * v);
      if (valid < 32) {  // the last rows of all: those beyond M hold a repeated row and must not count, infinite or not
#pragma unroll
        for (int v = 0; v < 4; ++v) bf[v] = masked(bf[v], ks, valid);
        if constexpr (!PACKED) {  // the packed weights are zero there
#pragma unroll
          for (int u = 0; u < 2; ++u) af[u] = masked(af[u], ks, valid);
        }
      }
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[u][v] = mfma::mma(af[u], bf[v], acc[u][v]);
      if (sums) {
        if constexpr (PACKED) {
#pragma unroll
          for (int v = 0; v < 4; ++v) add_columns(bf[v], csum[v]);
        } else {
#pragma unroll
          for (int u = 0; u < 2; ++u) add_columns(af[u], csum[u]);
        }
      }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing may still be landing in LDS when the workgroup ends
  const int64_t ld = (int64_t)(CONV ? a.grid.taps : 1) * a.OB;
  float *dst = a.partials + (int64_t)chunk * a.OA * ld + (int64_t)tap * a.OB;
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int ob = ob0 + wb + 32 * v + i;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int oa = oa0 + wa + 32 * u + mfma::rowmap(r, g);
        if (oa < a.OA && ob < a.OB) dst[(int64_t)oa * ld + ob] = acc[u][v][r];
      }
    }
  if (sums) {
#pragma unroll
    for (int u = 0; u < (PACKED ? 4 : 2); ++u) {
      const float total = csum[u] + __shfl_xor(csum[u], 32, 64);
      const int col = (PACKED ? ob0 + wb : oa0 + wa) + 32 * u + i, ncol = PACKED ? a.OB : a.OA;
      if (g == 0 && col < ncol) a.col_sums[(int64_t)chunk * ncol + col] = total;
    }
  }
}

// ------------------------------------------------------------------------------------------------
// narrow_wgrad_kernel: P[w][n] = sum_m W[m][w] V[m][n] with n < NN <= 16.  A thread keeps 4 columns of W against all
// columns of V in registers, four rows in flight per workgroup; V's rows pass through LDS as fp32 (64 at a time) and are
// read as broadcasts.  Also the column sums of W and of V.  Bound by reading W once.
// ------------------------------------------------------------------------------------------------
struct NarrowArgs {
  const void *W, *V;
  int ldw, ldv, OW, ON;
  int64_t M, per;      // rows per chunk
  float *partials;     // [chunk][OW][ON] (swap = 0) or [chunk][ON][OW] (swap = 1)
  float *sums_w, *sums_v;  // [chunk][OW], [chunk][ON]; NULL: not wanted
  int swap;
};

template <typename T, int NN>
__global__ __launch_bounds__(256) void narrow_wgrad_kernel(NarrowArgs a) {
  constexpr int ROWS = 64;
  __shared__ float vs[ROWS][NN];
  __shared__ float red[3][64][4 * NN + 5];
  typedef typename std::conditional<sizeof(T) == 2, u32x2, u32x4>::type quad;
  const T *W = static_cast<const T *>(a.W), *V = static_cast<const T *>(a.V);
  const int t = threadIdx.x, cg = t & 63, rl = t >> 6, c0 = blockIdx.y * 256 + 4 * cg;
  const bool live = c0 < a.OW;
  const int64_t m0 = (int64_t)blockIdx.x * a.per, m1 = m0 + a.per < a.M ? m0 + a.per : a.M;
  float acc[4][NN], sw[4] = {0.f, 0.f, 0.f, 0.f}, sv = 0.f;
#pragma unroll
  for (int k = 0; k < 4; ++k)
#pragma unroll
    for (int n = 0; n < NN; ++n) acc[k][n] = 0.f;
  for (int64_t mb = m0; mb < m1; mb += ROWS) {
    __syncthreads();
    for (int e = t; e < ROWS * NN; e += 256) {
      const int r = e / NN, n = e - r * NN;
      vs[r][n] = (mb + r < m1 && n < a.ON) ? load_as_f32(V + (mb + r) * a.ldv + n) : 0.f;
    }
    __syncthreads();
    quad w[ROWS / 4];
#pragma unroll
    for (int k = 0; k < ROWS / 4; ++k) {
      const int64_t m = mb + 4 * k + rl;
      w[k] = quad{};
      if (live && m < m1) w[k] = *reinterpret_cast<const quad *>(W + m * a.ldw + c0);
    }
#pragma unroll
    for (int k = 0; k < ROWS / 4; ++k) {
      float x[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if constexpr (sizeof(T) == 2) {
          const uint32_t word = w[k][j >> 1];
          x[j] = __uint_as_float((j & 1) ? (word & 0xffff0000u) : (word << 16));
        } else {
          const uint32_t word = w[k][j];
          x[j] = __uint_as_float(word);
        }
        sw[j] += x[j];
      }
      const float *v = vs[4 * k + rl];
#pragma unroll
      for (int n = 0; n < NN; ++n)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[j][n] = fmaf(x[j], v[n], acc[j][n]);
    }
    if (a.sums_v && blockIdx.y == 0 && t < NN)
      for (int r = 0; r < ROWS; ++r) sv += vs[r][t];
  }
  if (rl > 0) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
      for (int n = 0; n < NN; ++n) red[rl - 1][cg][j * NN + n] = acc[j][n];
      red[rl - 1][cg][4 * NN + j] = sw[j];
    }
  }
  __syncthreads();
  const int64_t chunk = blockIdx.x;
  if (rl == 0 && live) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
      for (int n = 0; n < NN; ++n) {
        const float v = ((acc[j][n] + red[0][cg][j * NN + n]) + red[1][cg][j * NN + n]) + red[2][cg][j * NN + n];
        if (n < a.ON)
          a.partials[chunk * a.OW * a.ON + (a.swap ? (int64_t)n * a.OW + c0 + j : (int64_t)(c0 + j) * a.ON + n)] = v;
      }
      if (a.sums_w)
        a.sums_w[chunk * a.OW + c0 + j] =
            ((sw[j] + red[0][cg][4 * NN + j]) + red[1][cg][4 * NN + j]) + red[2][cg][4 * NN + j];
    }
  }
  if (a.sums_v && blockIdx.y == 0 && t < a.ON) a.sums_v[chunk * a.ON + t] = sv;
}

// ------------------------------------------------------------------------------------------------
// sum_partials_kernel: dst[e] = sum_g src[g][e], up to eight results in one launch: a backward pass has three to eight of
// them, each 4 to 6 us for what is mostly too small to fill the chip.  A Transolver++ layer's step over 100 003 points takes
// 650 us with one launch at the end of its backward pass where it took 658 with three, the float32 grid model's 4 604 with
// one per layer and 4 653 with five.  A workgroup takes 4 consecutive elements
// per lane of its rows, every `parts`-th partial per row of lanes, and adds the parts up through LDS, always in the same
// order.  Bound by the read of the partials, which the product before has just written.
// blockIdx.y: a batch of such sums of the first result ([batch][g][e] -> [batch][e]); the others are formed by batch 0.
// 64 partials of 524 288 elements 25.3 -> 23.4 us (5.7 TB/s), 35 of them 25.7 -> 14.9; 14 of a 3 x 3 convolution's
// 1 179 648 28.6 -> 15.6; 1 024 of 512 elements 8.2 -> 4.9 (with 32 one-element lanes before).
// ------------------------------------------------------------------------------------------------
typedef float f32x4 __attribute__((ext_vector_type(4)));

// sum of load(g) over g = part, part + PARTS, .. < G, AHEAD loads in flight
template <int PARTS, int AHEAD, class V, class F>
__device__ __forceinline__ V sum_of_part(int part, int G, F &&load) {
  V s = {};
  int g = part;
  for (; g + (AHEAD - 1) * PARTS < G; g += AHEAD * PARTS) {
    V r[AHEAD];
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) r[u] = load(g + u * PARTS);
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) s += r[u];
  }
  for (; g < G; g += AHEAD / 2 * PARTS) {  // the rest, half as many in flight
    V r[AHEAD / 2];
#pragma unroll
    for (int u = 0; u < AHEAD / 2; ++u) r[u] = load(min(g + u * PARTS, G - 1));
#pragma unroll
    for (int u = 0; u < AHEAD / 2; ++u) s += g + u * PARTS < G ? r[u] : V{};
  }
  return s;
}

// sum of load(k) over k < PARTS (a power of two), halves added to halves: one after the other 32 parts of random signs were 1.3 to 1.6
// times as far from float64
template <int PARTS, class F>
__device__ __forceinline__ float sum_of_parts(F &&load) {
  float v[PARTS];
#pragma unroll
  for (int k = 0; k < PARTS; ++k) v[k] = load(k);
#pragma unroll
  for (int half = PARTS / 2; half > 0; half /= 2)
#pragma unroll
    for (int k = 0; k < half; ++k) v[k] += v[k + half];
  return v[0];
}

template <int LANES, int V>
__device__ __forceinline__ void sum_rows_of(const Sums::One &o, int64_t batch, float *part) {
  constexpr int PARTS = 256 / LANES, PER = LANES * V;
  typedef float fvec __attribute__((ext_vector_type(V)));
  const int64_t e0 = ((int64_t)blockIdx.x - o.first) * PER, n = o.n;
  const int lane = threadIdx.x % LANES, part_id = threadIdx.x / LANES;
  fvec s = {};
  if (e0 + lane * V < n) {  // V elements or none: n is a multiple of V
    const float *p = o.src + batch * o.G * n + e0 + lane * V;
    s = sum_of_part<PARTS, 8, fvec>(part_id, o.G,
                                    [&](int g) { return *reinterpret_cast<const fvec *>(p + (int64_t)g * n); });
  }
#pragma unroll
  for (int v = 0; v < V; ++v) part[part_id * PER + lane * V + v] = s[v];
  __syncthreads();
  const int64_t e = e0 + threadIdx.x;
  if (threadIdx.x >= PER || e >= n) return;
  const float v = sum_of_parts<PARTS>([&](int k) { return part[k * PER + threadIdx.x]; });
  int64_t at = batch * n + e;
  if (o.taps > 1) {
    const int64_t oa = e / (o.taps * (int64_t)o.OB), rest = e - oa * o.taps * o.OB, tap = rest / o.OB, ob = rest - tap * o.OB;
    at = (oa * o.OB + ob) * o.taps + tap;
  }
  o.dst[at] = v;
}

// [oa][tap][ob] -> [oa][ob][tap]: 256 neighbouring ob and kTaps taps at a time, so that a workgroup writes whole lines and
// not 4 bytes in every 4 taps
__device__ __forceinline__ void sum_taps_of(const Sums::One &o, float *part) {
  constexpr int PARTS = 4, PER = 256, K = Sums::kTaps;
  const int per_oa = o.OB / PER;
  const int64_t block = (int64_t)blockIdx.x - o.first, oa = block / per_oa, n = o.n;
  const int ob0 = (int)(block - oa * per_oa) * PER;
  const int lane = threadIdx.x % 64, part_id = threadIdx.x / 64;
  const float *src = o.src + oa * o.taps * o.OB + ob0 + 4 * lane;
  float *dst = o.dst + (oa * o.OB + ob0) * o.taps;
  for (int t0 = 0; t0 < o.taps; t0 += K) {
    const int nt = min(K, o.taps - t0);
    f32x4 acc[K] = {};
    for (int g = part_id; g < o.G; g += PARTS) {  // kTaps loads in flight
      const float *p = src + (int64_t)g * n + (int64_t)t0 * o.OB;
      f32x4 r[K];
#pragma unroll
      for (int t = 0; t < K; ++t) r[t] = *reinterpret_cast<const f32x4 *>(p + (int64_t)min(t, nt - 1) * o.OB);
#pragma unroll
      for (int t = 0; t < K; ++t) acc[t] += r[t];
    }
    if (t0 > 0) __syncthreads();
#pragma unroll
    for (int t = 0; t < K; ++t) *reinterpret_cast<f32x4 *>(part + (part_id * K + t) * PER + 4 * lane) = acc[t];
    __syncthreads();
    for (int e = threadIdx.x; e < PER * nt; e += 256) {
      const int ob = e / nt, t = e - ob * nt;
      dst[ob * o.taps + t0 + t] = sum_of_parts<PARTS>([&](int k) { return part[(k * K + t) * PER + ob]; });
    }
  }
}

// TAPS: some result takes a convolution's taps together (its own instance: it needs twice the registers)
template <bool TAPS>
__global__ __launch_bounds__(256) void sum_partials_kernel(Sums a) {
  extern __shared__ __align__(16) float part[];
  Sums::One o = a.r[0];
#pragma unroll
  for (int k = 1; k < Sums::kMost; ++k)
    if (k < a.count && (int64_t)blockIdx.x >= a.r[k].first) o = a.r[k];
  if (o.first > 0 && blockIdx.y > 0) return;
  if constexpr (TAPS) {
    if (o.lanes < 0) return sum_taps_of(o, part);
  }
  if (o.lanes == 64) sum_rows_of<64, 4>(o, blockIdx.y, part);
  else if (o.lanes == 32) sum_rows_of<32, 4>(o, blockIdx.y, part);
  else if (o.lanes == 16) sum_rows_of<16, 4>(o, blockIdx.y, part);
  else if (o.lanes == 8) sum_rows_of<8, 4>(o, blockIdx.y, part);
  else sum_rows_of<32, 1>(o, blockIdx.y, part);
}

// f(number of steps, first step) over n steps in batches of eight, four and one: a batch's loads are issued together.  (A loop
// around matrix instructions whose length is not known when it is compiled is not unrolled, whatever it is asked.)
template <class F>
__device__ __forceinline__ void in_batches(int n, F &&f) {
  int k = 0;
  for (; k + 8 <= n; k += 8) f(std::integral_constant<int, 8>{}, k);
  if (k + 4 <= n) f(std::integral_constant<int, 4>{}, k), k += 4;
  for (; k < n; ++k) f(std::integral_constant<int, 1>{}, k);
}

// ------------------------------------------------------------------------------------------------
// token_grad_kernel: what the layer's output gradient says about the slice tokens and out_linear, from the sums
// P[b][h S + s][c] = sum_n w[n, h, s] dy[n, c] (the packed product above) instead of from per-point d out_x and out_x:
//   d tok'[b, h, s, d] = sum_c P[b, h, s, c] W_out[c, 32 h + d]              workgroups 0 .. B H ceil(S / 32) - 1
//   d W_out[c, 32 h + d] = sum_b sum_s P[b, h, s, c] tok'[b, h, s, d]        the others, one per (`cb` batch elements, h,
//                                                                            32 rows c): a partial result per `cb` elements
// Four waves per 32 x 32 result tile on fp32 MFMA, each a quarter of the reduction, added up in order through LDS.  Bound
// by latency (P is a few hundred KB): the quarters took 60 us (one wave per tile) to 14 us at B = 1, S = 64, C = 256,
// their loads in batches that are issued together (in_batches) to 7.
// ------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void token_grad_kernel(const float *__restrict__ P, const uint16_t *__restrict__ w_out,
                                                         const float *__restrict__ out_token, float *__restrict__ d_token,
                                                         float *__restrict__ d_w_out, int B, int H, int S, int C, int cb) {
  __shared__ float part[3][16][64];
  const int lane = threadIdx.x & 63, i = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ST = (S + 31) / 32, HD = H * 32, first = B * H * ST;
  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  const bool to_token = (int)blockIdx.x < first;
  const int rest = blockIdx.x - first, per = H * (C / 32), chunk = to_token ? 0 : rest / per, e = rest - chunk * per;
  const int st = blockIdx.x % ST, bh = blockIdx.x / ST, h = to_token ? bh % H : e % H, c0 = e / H * 32;
  if (to_token) {
    const int s = 32 * st + i, cw = C / 4;
    const float *row = P + ((int64_t)bh * S + (s < S ? s : S - 1)) * C + wave * cw + 4 * g;
    const uint16_t *wcol = w_out + (int64_t)(wave * cw + 4 * g) * HD + 32 * h + i;
    in_batches(cw / 8, [&](auto n_, int k0) {  // lane half g supplies c + 4 g .. + 3, one pair (c + m, c + 4 + m) per MFMA
      constexpr int n = decltype(n_)::value;
      f32x4 p4[n];
      uint16_t w[n][4];
#pragma unroll
      for (int k = 0; k < n; ++k) {
        const int c = 8 * (k0 + k);
        p4[k] = *reinterpret_cast<const f32x4 *>(row + c);
#pragma unroll
        for (int m = 0; m < 4; ++m) w[k][m] = wcol[(int64_t)(c + m) * HD];
      }
      __builtin_amdgcn_sched_barrier(0);  // or the loads move down to their products
#pragma unroll
      for (int k = 0; k < n; ++k)
#pragma unroll
        for (int m = 0; m < 4; ++m) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(p4[k][m], bf16_bits_to_f32(w[k][m]), acc, 0, 0, 0);
    });
  } else {
    const int sw = S / 4, steps = sw / 2, b0 = chunk * cb, b_end = b0 + cb < B ? b0 + cb : B;
    in_batches((b_end - b0) * steps, [&](auto n_, int k0) {  // all batch elements of the chunk in one row of steps
      constexpr int n = decltype(n_)::value;
      float p[n], tk[n];
#pragma unroll
      for (int k = 0; k < n; ++k) {
        const int b = b0 + (k0 + k) / steps, s = 2 * ((k0 + k) % steps);
        const int64_t at = ((int64_t)b * H + h) * S + wave * sw + g + s;
        p[k] = P[at * C + c0 + i];
        tk[k] = out_token[at * 32 + i];
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < n; ++k) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(p[k], tk[k], acc, 0, 0, 0);
    });
  }
  if (wave > 0) {
#pragma unroll
    for (int r = 0; r < 16; ++r) part[wave - 1][r][lane] = acc[r];
  }
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const float v = ((acc[r] + part[0][r][lane]) + part[1][r][lane]) + part[2][r][lane];
    const int row = mfma::rowmap(r, g);
    if (!to_token) d_w_out[((int64_t)chunk * C + c0 + row) * HD + 32 * h + i] = v;
    else if (32 * st + row < S) d_token[((int64_t)bh * S + 32 * st + row) * 32 + i] = v;
  }
}

// ================================================================================================
// host side
// ================================================================================================
// Row chunks of a product of `tiles` workgroups per chunk: every workgroup resident at once (one 128 KB ring per CU), and
// not so many that writing and re-reading the partial results costs more than the shorter chunks save: a chunk of r rows
// takes about r 20 ns, a partial of n values about n ps, and their sum is smallest at G = sqrt(2e4 M / n).  Products and
// totals of a training step at sqrt(1e4 M / n) / here / sqrt(4e4 M / n): two blocks on 20 000 points 295 / 269 / 276 us, on a
// 64 x 64 grid 250 / 226 / 223, on two of 128 x 128 523 / 518 / 537; a layer of 16 384 points 58 / 54 / 54, of 50 000 75 / 72 / 72.
int64_t chunks_for(int64_t M, int64_t tiles, int64_t n, int num_cu) {
  const int64_t nblk = (M + 31) / 32;
  int64_t g = num_cu / tiles;
  int64_t best = 1;
  while ((best + 1) * (best + 1) <= 20000 * M / n) ++best;
  if (g > best) g = best;
  if (g > nblk) g = nblk;
  return g < 1 ? 1 : g;
}

static bool wide(int64_t OA, int64_t OB) { return OA % 32 == 0 && OB % 32 == 0 && OA >= 128 && OB >= 128; }

enum class Form { none, wide_bf16, tiles_bf16, tiles_f32, narrow };

static Form form_of(int dtype, int64_t OA, int64_t OB, int taps) {
  if (OA <= 0 || OB <= 0) return Form::none;
  if (dtype == PA_F32) {
    if (OA % 4 == 0 && OB % 4 == 0 && OA >= 16 && OB >= 16) return Form::tiles_f32;
  } else if (dtype == PA_BF16) {
    if (wide(OA, OB)) return Form::wide_bf16;
    if (taps == 1 && OA % 32 == 0 && (OA <= 256 || OA % 256 == 0) && (OB == 32 || OB == 64 || OB == 128 || OB == 256))
      return Form::tiles_bf16;
  }
  if (taps == 1 && ((OB <= 16 && OA % 4 == 0 && OA >= 16) || (OA <= 16 && OB % 4 == 0 && OB >= 16))) return Form::narrow;
  return Form::none;
}

static int64_t chunks_of(Form f, int64_t M, int64_t OA, int64_t OB, int taps, int num_cu) {
  switch (f) {
    case Form::wide_bf16: return chunks_for(M, ((OA + 255) / 256) * ((OB + 255) / 256) * taps, OA * OB * taps, num_cu);
    case Form::tiles_bf16: return gemm::cols_gemm_chunks(M, OA, num_cu);
    case Form::tiles_f32: return gemm::cols_gemm_f32_chunks(M, OA, OB * taps, num_cu);
    case Form::narrow: {
      const int64_t w = OA > OB ? OA : OB;
      int64_t g = 4 * (int64_t)num_cu / ((w + 255) / 256);
      const int64_t cap = (M + 127) / 128;
      if (g > cap) g = cap;
      return g < 1 ? 1 : g;
    }
    default: return 0;
  }
}

int64_t workspace_bytes(int dtype, int64_t M, int64_t OA, int64_t OB, int taps, int num_cu) {
  const Form f = form_of(dtype, OA, OB, taps);
  if (f == Form::none) return PA_ERR_UNSUPPORTED;
  return chunks_of(f, M, OA, OB, taps, num_cu) * (OA * OB * taps + OA) * 4;
}

template <typename T>
static int launch_narrow(const NarrowArgs &a, int64_t G, hipStream_t st) {
  const dim3 grid((unsigned)G, (unsigned)((a.OW + 255) / 256));
  if (a.ON <= 4) hipLaunchKernelGGL((narrow_wgrad_kernel<T, 4>), grid, dim3(256), 0, st, a);
  else if (a.ON <= 8) hipLaunchKernelGGL((narrow_wgrad_kernel<T, 8>), grid, dim3(256), 0, st, a);
  else hipLaunchKernelGGL((narrow_wgrad_kernel<T, 16>), grid, dim3(256), 0, st, a);
  return launch_status();
}

int launch_wide(const void *A, int64_t lda, int64_t OA, const void *B, int64_t ldb, int64_t OB, int64_t M, int64_t G,
                const pa_shape *grid, float *partials, float *col_sums, hipStream_t st) {
  Args a{};
  a.A = static_cast<const uint16_t *>(A);
  a.B = static_cast<const uint16_t *>(B);
  a.lda = (int)lda, a.ldb = (int)ldb, a.OA = (int)OA, a.OB = (int)OB;
  a.M = M;
  a.per = (int)(((M + 31) / 32 + G - 1) / G);
  a.grid = grid_taps(grid);
  a.chunks = (int)G, a.batches = 1;
  a.ny = (int)((OA + 255) / 256);
  a.nz = (int)((OB + 255) / 256) * a.grid.taps;
  a.partials = partials, a.col_sums = col_sums;
  auto kernel = grid ? wgrad_kernel<1> : wgrad_kernel<0>;
  const size_t lds = (size_t)kStages * kStageBytes;
  if (int rc = allow_dynamic_lds(kernel, lds)) return rc;
  hipLaunchKernelGGL(kernel, dim3((unsigned)((G * a.ny * a.nz + 7) / 8 * 8)), dim3(512), lds, st, a);
  return launch_status();
}

int product(int dtype, int64_t M, const void *A, int64_t lda, int64_t OA, const void *B, int64_t ldb, int64_t OB,
            const pa_shape *grid, void *workspace, float *out, float *col_sums, int num_cu, hipStream_t st, Sums *later) {
  const int taps = grid_taps(grid).taps;
  const Form f = form_of(dtype, OA, OB, taps);
  if (f == Form::none) return PA_ERR_UNSUPPORTED;
  const int64_t G = chunks_of(f, M, OA, OB, taps, num_cu), n = OA * OB * taps;
  float *partials = static_cast<float *>(workspace), *sums = col_sums ? partials + G * n : nullptr;
  int rc = PA_OK;
  switch (f) {
    case Form::wide_bf16: rc = launch_wide(A, lda, OA, B, ldb, OB, M, G, grid, partials, sums, st); break;
    case Form::tiles_bf16: rc = gemm::cols_gemm(A, lda, OA, B, ldb, OB, M, partials, sums, num_cu, st); break;
    case Form::tiles_f32: rc = gemm::cols_gemm_f32(A, lda, OA, B, ldb, OB, M, grid, partials, sums, num_cu, st); break;
    default: {
      NarrowArgs a{};
      const bool a_wide = OB <= 16 && OA >= 16 && OA % 4 == 0;
      a.W = a_wide ? A : B, a.V = a_wide ? B : A;
      a.ldw = (int)(a_wide ? lda : ldb), a.ldv = (int)(a_wide ? ldb : lda);
      a.OW = (int)(a_wide ? OA : OB), a.ON = (int)(a_wide ? OB : OA);
      a.M = M, a.per = (M + G - 1) / G;
      a.partials = partials;
      (a_wide ? a.sums_w : a.sums_v) = sums;
      a.swap = a_wide ? 0 : 1;
      rc = dtype == PA_F32 ? launch_narrow<float>(a, G, st) : launch_narrow<bf16>(a, G, st);
    }
  }
  if (rc) return rc;
  Sums own, &s = later ? *later : own;
  s.add(partials, out, n, G, taps, OB);
  if (col_sums) s.add(sums, col_sums, OA, G);
  return later ? PA_OK : launch_sums(own, st);
}

static int launch_sums(const Sums &sums, int64_t batches, hipStream_t st) {
  const dim3 grid((unsigned)sums.blocks, (unsigned)batches);
  if (sums.by_taps) hipLaunchKernelGGL((sum_partials_kernel<true>), grid, dim3(256), 1024 * Sums::kTaps * 4, st, sums);
  else hipLaunchKernelGGL((sum_partials_kernel<false>), grid, dim3(256), 1024 * 4, st, sums);
  return launch_status();
}
int launch_sums(const Sums &sums, hipStream_t st) { return launch_sums(sums, 1, st); }

// dst[e] = sum over `rows` rows of n floats
int sum_rows(const float *src, int64_t rows, int64_t n, float *dst, hipStream_t st) {
  Sums s;
  s.add(src, dst, n, rows);
  return launch_sums(s, st);
}

// ---- the layer's output gradient against the packed slice weights ----
static int64_t output_chunks(const pa_shape &s, int num_cu) {  // row chunks per batch element
  const int64_t HS = s.H * s.S, tiles = ((HS + 255) / 256) * ((s.C + 255) / 256), tpb = (s.N + 31) / 32;
  int64_t g = chunks_for(s.N, tiles * s.B, HS * s.C, num_cu);
  if (g > tpb) g = tpb;
  return g < 1 ? 1 : g;
}

// The sums P take n = H S C floats per batch element whatever its number of points, so many small clouds go through in
// groups that fill the chip once (128 at C = 256, S = 64; up to 64 MB of P), with no copy of P where a batch element is one
// chunk; and d W_out is formed from `cb` elements per workgroup, 32 partial results at most.  512 clouds of 64 points, 256 / 64:
// 338 us; all of P at once, copied, and one workgroup walking all clouds 2 731 us.
struct OutputPlan {
  int64_t G, Bg, cb, parts, n;                         // chunks and elements per group, elements per d W_out part, parts
  int64_t P, partials, sums, dw, total;                // floats into the workspace
};
static OutputPlan output_plan(const pa_shape &s, int num_cu) {
  OutputPlan p{};
  const int64_t HS = s.H * s.S, tiles = ((HS + 255) / 256) * ((s.C + 255) / 256);
  p.G = output_chunks(s, num_cu), p.n = HS * s.C;
  p.cb = (s.B + 31) / 32 > 4 ? (s.B + 31) / 32 : 4;
  p.parts = (s.B + p.cb - 1) / p.cb;
  p.Bg = (num_cu / tiles + p.cb - 1) / p.cb * p.cb;  // whole parts
  if (p.Bg < p.cb) p.Bg = p.cb;
  if (p.Bg > s.B) p.Bg = s.B;
  p.partials = p.Bg * p.n;
  p.sums = p.partials + (p.G > 1 ? p.Bg * p.G * p.n : 0);
  p.dw = p.sums + s.B * p.G * s.C;
  p.total = p.dw + (p.parts > 1 ? p.parts * s.C * s.H * 32 : 0);
  return p;
}

int64_t output_backward_workspace_bytes(const pa_shape &s, int num_cu) { return output_plan(s, num_cu).total * 4; }

// dy (B, N, C) bf16, w_pack and out_token of the forward, w_out (C, H*32) bf16 -> d tok' (B,H,S,32), d W_out, d b_out
int output_backward(const pa_shape &s, const void *w_pack, const void *dy, const float *out_token, const void *w_out,
                    void *workspace, float *d_out_token, float *d_w_out, float *d_b_out, int num_cu, hipStream_t st) {
  const OutputPlan p = output_plan(s, num_cu);
  const int64_t HS = s.H * s.S, tok = HS * 32, HD = s.H * 32, ST = (s.S + 31) / 32;
  float *ws = static_cast<float *>(workspace), *P = ws + p.P, *partials = p.G > 1 ? ws + p.partials : P, *sums = ws + p.sums,
        *dw = p.parts > 1 ? ws + p.dw : d_w_out;
  Args a{};
  a.ldb = (int)s.C, a.OA = (int)HS, a.OB = (int)s.C;
  a.M = s.N, a.tpb = (int)((s.N + 31) / 32), a.tile_units = (int)(HS / 16 * 64);
  a.per = (int)((a.tpb + p.G - 1) / p.G);
  a.grid = grid_taps(nullptr);
  a.chunks = (int)p.G;
  a.ny = (int)((HS + 255) / 256), a.nz = (int)((s.C + 255) / 256);
  a.partials = partials;
  const size_t lds = (size_t)kStages * kStageBytes;
  int rc = allow_dynamic_lds(wgrad_kernel<2>, lds);
  if (rc) return rc;
  for (int64_t b0 = 0; b0 < s.B; b0 += p.Bg) {
    const int64_t nb = s.B - b0 < p.Bg ? s.B - b0 : p.Bg;
    a.B = static_cast<const uint16_t *>(dy) + b0 * s.N * s.C;
    a.pack = static_cast<const u32x4 *>(w_pack) + b0 * a.tpb * a.tile_units;
    a.batches = (int)nb;
    a.col_sums = sums + b0 * p.G * s.C;
    hipLaunchKernelGGL(wgrad_kernel<2>, dim3((unsigned)((nb * p.G * a.ny * a.nz + 7) / 8 * 8)), dim3(512), lds, st, a);
    if ((rc = launch_status())) return rc;
    if (p.G > 1) {
      Sums sa;
      sa.add(partials, P, p.n, p.G);
      if (p.parts == 1) sa.add(sums, d_b_out, s.C, s.B * p.G);  // nothing else is to be added up
      if ((rc = launch_sums(sa, nb, st))) return rc;
    }
    const int64_t wgs = nb * s.H * ST + s.H * (s.C / 32) * ((nb + p.cb - 1) / p.cb);
    hipLaunchKernelGGL(token_grad_kernel, dim3((unsigned)wgs), dim3(256), 0, st, P, static_cast<const uint16_t *>(w_out),
                       out_token + b0 * tok, d_out_token + b0 * tok, dw + b0 / p.cb * s.C * HD, (int)nb, (int)s.H, (int)s.S,
                       (int)s.C, (int)p.cb);
    if ((rc = launch_status())) return rc;
  }
  if (p.parts == 1 && p.G > 1) return PA_OK;
  Sums sa;
  sa.add(sums, d_b_out, s.C, s.B * p.G);
  if (p.parts > 1) sa.add(dw, d_w_out, s.C * HD, p.parts);
  return launch_sums(sa, st);
}

}  // namespace wgrad
}  // namespace pa
