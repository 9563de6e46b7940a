// Row GEMM on the matrix cores for the general kernel family: out[m, o] = bias[o] + sum_k A(m, k) W[o, k], where
// A is either the rows of the input (Linear) or the gathered k x k (x k) neighbourhood of a grid point (Conv2d /
// Conv3d as implicit GEMM).  fp32 storage uses v_mfma_f32_32x32x2_f32 (fp32 products and sums: the result stays in
// the rtol-1e-4 class of the fp32 path), bf16 storage uses v_mfma_f32_32x32x16_bf16.
//
// Workgroup: 4 waves, 128 rows x (32 * NT) output columns; wave v owns rows 32v..32v+31 and NT accumulator tiles.
// The reduction axis is walked in blocks of 128 bytes per row (32 fp32 / 64 bf16 values = 8 units of 16 bytes).
// Both operand tiles are staged in LDS as [row][unit] with a row stride of 9 units: the 16 lanes of one 128-bit access
// phase (rows r..r+15, same unit) then fall on 16 distinct bank groups.  A lane (i, g) reads unit 2p + g of its row
// for p = 0..3: that is one bf16 MFMA operand (k = 8 values), or four fp32 operands (k = one value each).  Which k a
// lane holds is the same for A and W, so any assignment is a valid reduction order.
// The next block is fetched from global memory into registers while the MFMAs of the current one run.
#include "pa_common.h"
#include "pa_host.h"
#include "pa_mfma_ops.h"

namespace pa {
namespace gemm {

using mfma::f32x16;
using mfma::u32x4;

constexpr int kRows = 128;   // rows per workgroup
constexpr int kUnits = 8;    // 16-byte units per row and reduction block
constexpr int kRowU = 9;     // LDS row stride in units

template <typename T>
struct Unit;
template <>
struct Unit<float> {
  static constexpr int kElems = 4;
};
template <>
struct Unit<bf16> {
  static constexpr int kElems = 8;
};

__device__ __forceinline__ f32x16 mma_unit(const float *, u32x4 a, u32x4 b, f32x16 c) {
#pragma unroll
  for (int j = 0; j < 4; ++j)
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a[j]), __uint_as_float(b[j]), c, 0, 0, 0);
  return c;
}
__device__ __forceinline__ f32x16 mma_unit(const bf16 *, u32x4 a, u32x4 b, f32x16 c) { return mfma::mma(a, b, c); }

template <typename T, int NT>
__global__ __launch_bounds__(256) void rows_gemm_mfma_kernel(GemmArgs a) {
  constexpr int UE = Unit<T>::kElems, KB = kUnits * UE, BN = 32 * NT;
  __shared__ u32x4 As[kRows * kRowU];
  __shared__ u32x4 Ws[BN * kRowU];
  const int z = blockIdx.z;
  const T *in = static_cast<const T *>(a.in);
  const T *W = static_cast<const T *>(a.w[z]);
  const float *bias = a.bias[z];
  T *out = static_cast<T *>(a.out[z]);
  const int t = threadIdx.x, lane = t & 63, i = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int64_t m0 = (int64_t)blockIdx.x * kRows;
  const int o0 = blockIdx.y * BN;
  const int q = t & 7;    // the unit of a row this thread stages
  const int r0 = t >> 3;  // its first row; the others follow in steps of 32

  const int gd = a.gd > 0 ? a.gd : 1;
  const int ksd = a.gd > 0 ? a.ks : 1;
  const int taps = a.ks * a.ks * ksd;
  const int pad = a.ks / 2;

  // Row numbering: the rows of `in` in order, or (pack_tpb > 0) batch by batch with every batch padded to whole
  // 32-point tiles, so that a wave's 32 rows are one tile of one batch.
  const int64_t padded = (int64_t)a.pack_tpb * 32;  // rows per batch in the padded numbering
  auto real_row = [&](int64_t vm) -> int64_t {
    if (a.pack_tpb == 0) return vm < a.M ? vm : -1;
    const int64_t b = vm / padded, n = vm - b * padded;
    return (n < a.N && b * a.N + n < a.M) ? b * a.N + n : -1;
  };

  // the 4 input rows this thread stages: global row, and for a convolution its batch offset and grid coordinates
  int64_t arow[4];
  int ci[4], cj[4], cl[4];
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const int64_t m = m0 + r0 + 32 * p;
    arow[p] = real_row(m);
    ci[p] = cj[p] = cl[p] = 0;
    if (a.ks > 0 && arow[p] >= 0) {  // grid coordinates from the real row (the padded numbering skips rows)
      const int64_t b = arow[p] / a.N;
      int n = (int)(arow[p] - b * a.N);
      cl[p] = n % gd;
      n /= gd;
      ci[p] = n / a.gw;
      cj[p] = n - ci[p] * a.gw;
      arow[p] = b * a.N;  // first point of the row's batch
    }
  }

  u32x4 pa[4], pw[NT];
  auto fetch = [&](int kb) {
    const int k = kb * KB + q * UE;
    const bool k_ok = k < a.K;
    if (a.ks == 0) {
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        pa[p] = u32x4{0, 0, 0, 0};
        if (k_ok && arow[p] >= 0) pa[p] = *reinterpret_cast<const u32x4 *>(in + arow[p] * a.K + k);
      }
#pragma unroll
      for (int p = 0; p < NT; ++p) {
        const int o = o0 + r0 + 32 * p;
        pw[p] = u32x4{0, 0, 0, 0};
        if (k_ok && o < a.O) pw[p] = *reinterpret_cast<const u32x4 *>(W + (int64_t)o * a.K + k);
      }
    } else {
      const int tap = k / a.C, c = k - tap * a.C;
      const int uv = tap / ksd, zz = tap - uv * ksd;
      const int u = uv / a.ks, v = uv - u * a.ks;
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const int ii = ci[p] + u - pad, jj = cj[p] + v - pad, ll = cl[p] + (a.gd > 0 ? zz - pad : 0);
        pa[p] = u32x4{0, 0, 0, 0};
        if (k_ok && arow[p] >= 0 && ii >= 0 && ii < a.gh && jj >= 0 && jj < a.gw && ll >= 0 && ll < gd)
          pa[p] = *reinterpret_cast<const u32x4 *>(in + (arow[p] + ((int64_t)ii * a.gw + jj) * gd + ll) * a.C + c);
      }
#pragma unroll
      for (int p = 0; p < NT; ++p) {
        const int o = o0 + r0 + 32 * p;
        if (a.w_tap_major) {  // W[o][tap][c]: the unit is contiguous, as for a Linear
          pw[p] = u32x4{0, 0, 0, 0};
          if (k_ok && o < a.O) pw[p] = *reinterpret_cast<const u32x4 *>(W + (int64_t)o * a.K + k);
        } else {
          alignas(16) T e[UE];
#pragma unroll
          for (int j = 0; j < UE; ++j) {
            e[j] = T{};
            if (k_ok && o < a.O) e[j] = W[(int64_t)o * a.K + (int64_t)(c + j) * taps + tap];
          }
          pw[p] = *reinterpret_cast<const u32x4 *>(e);
        }
      }
    }
  };

  f32x16 acc[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[nt][r] = 0.f;

  const int nkb = (a.K + KB - 1) / KB;
  fetch(0);
  for (int kb = 0; kb < nkb; ++kb) {
#pragma unroll
    for (int p = 0; p < 4; ++p) As[(r0 + 32 * p) * kRowU + q] = pa[p];
#pragma unroll
    for (int p = 0; p < NT; ++p) Ws[(r0 + 32 * p) * kRowU + q] = pw[p];
    __syncthreads();
    fetch(kb + 1 < nkb ? kb + 1 : kb);  // the last block re-fetches itself: no branch around the loads
    const u32x4 *ar = As + (wave * 32 + i) * kRowU + g;
    const u32x4 *wr = Ws + i * kRowU + g;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const u32x4 av = ar[2 * p];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[nt] = mma_unit(in, av, wr[nt * 32 * kRowU + 2 * p], acc[nt]);
    }
    __syncthreads();
  }

  const int64_t tile = (int64_t)blockIdx.x * 4 + wave;  // this wave's 32 rows (one (batch, tile) when packing)
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int o = o0 + nt * 32 + i;
    if (o >= a.O) continue;
    const float bv = bias ? bias[o] : 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[nt][r] += bv;
    if (a.act == 1) {
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[nt][r] = gelu_erf(acc[nt][r]);
    }
    if (out) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int64_t m = real_row(tile * 32 + mfma::rowmap(r, g));
        if (m >= 0) store_from_f32(out + m * a.O + o, acc[nt][r]);
      }
    }
    if constexpr (sizeof(T) == 2) {
      u32x4 *pk = static_cast<u32x4 *>(a.out_pack[z]);
      const int head = (o0 >> 5) + nt;
      if (a.pack_tpb > 0 && pk && tile * 32 < (a.M / a.N) * padded) {
        pk[((tile * a.pack_heads + head) * 2 + 0) * 64 + lane] = mfma::pack_half<0>(acc[nt]);
        pk[((tile * a.pack_heads + head) * 2 + 1) * 64 + lane] = mfma::pack_half<1>(acc[nt]);
      }
    }
  }
}

// ------------------------------------------------------------------------------------------------
// rows_linear_kernel: the bf16 Linear over very many rows, weights stationary.  out = in . W^T + bias with
// K = 16 * KS in {128, 256, 512} and up to 256 output columns per workgroup (grid.y walks wider outputs, grid.z the
// second (W, bias, out) set).  One wave per 32 output columns keeps its W rows in registers (KS operand fragments) for
// the whole kernel; the workgroup walks the 32-row tiles g, g + G, ... of its batch range; a tile's rows are staged in
// LDS by the whole workgroup with full-row coalesced loads ([row][unit] with one unit of stagger per row, see above)
// and read back as operand fragments by every wave; the next tile is fetched into registers while the current one is
// multiplied.  The product is formed as out^T (channels x rows: lanes <-> rows, registers <-> channels) so that a
// row's 32 channels leave as 16-byte stores; with packing on, the un-transposed tile (lanes <-> channels) is formed
// as well and written in the packed operand layout of the slice kernels.
// Rows are numbered as in rows_gemm_mfma_kernel (padded per batch when pack_tpb > 0).
// Bound by memory latency: a workgroup has one tile (16 KB at K = 256) on its way.  LEAN (K = 256, 256 columns per
// workgroup, natural output only) fits 128 registers, so two workgroups share a CU and one's loads cover the other's:
// 256 -> 2 x 256 at 1 048 576 rows 441 -> 394 us (4.1 TB/s), 256 -> 256 228 -> 212 us (5.1 TB/s).
// ------------------------------------------------------------------------------------------------
template <int KS, bool LEAN>
__global__ __launch_bounds__(512, LEAN ? 4 : 2) void rows_linear_kernel(GemmArgs a) {
  constexpr int K = 16 * KS, UPR = K / 8, ROWU = UPR + 1;
  constexpr int PT = LEAN ? 32 * UPR / 512 : 4;  // 16-byte units a thread stages per tile, at most
  extern __shared__ u32x4 xs_all[];
  u32x4(*xs)[32 * ROWU] = reinterpret_cast<u32x4(*)[32 * ROWU]>(xs_all);  // two tile buffers
  const int z = blockIdx.z;
  const uint16_t *in = static_cast<const uint16_t *>(a.in);
  const uint16_t *W = static_cast<const uint16_t *>(a.w[z]);
  uint16_t *out = static_cast<uint16_t *>(a.out[z]);
  u32x4 *pk = LEAN ? nullptr : static_cast<u32x4 *>(a.out_pack[z]);
  const int tid = threadIdx.x, lane = tid & 63, i = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int NT = LEAN ? 512 : blockDim.x;
  const int o0 = blockIdx.y * 256 + wave * 32;  // this wave's output columns

  u32x4 wf[KS];  // W[o0 + i][16 ks + 8 g + j]: the A operand of out^T and the B operand of the un-transposed tile
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
    wf[ks] = *reinterpret_cast<const u32x4 *>(W + (int64_t)(o0 + i) * K + 16 * ks + 8 * g);
  float bias_t[16];  // bias of channel rowmap(r, g) (out^T: registers <-> channels); LEAN reads it from LDS per tile
  __shared__ float bias_s[LEAN ? 256 : 1];
  if constexpr (LEAN) {
    if (tid < 256) bias_s[tid] = a.bias[z] ? a.bias[z][blockIdx.y * 256 + tid] : 0.f;
  } else {
#pragma unroll
    for (int r = 0; r < 16; ++r) bias_t[r] = a.bias[z] ? a.bias[z][o0 + mfma::rowmap(r, g)] : 0.f;
  }
  const float bias_n = !LEAN && a.bias[z] ? a.bias[z][o0 + i] : 0.f;

  const int tpb = LEAN ? 0 : a.pack_tpb;
  const int64_t padded = (int64_t)tpb * 32;
  const int64_t ntiles = tpb > 0 ? (a.M / a.N) * tpb : (a.M + 31) / 32;
  auto real_row = [&](int64_t vm) -> int64_t {
    if (tpb == 0) return vm < a.M ? vm : -1;
    const int64_t b = vm / padded, n = vm - b * padded;
    return (n < a.N && b * a.N + n < a.M) ? b * a.N + n : -1;
  };
  // staging: unit idx = k * NT + tid of the tile -> row idx / UPR, position idx % UPR; 32 * UPR units per tile
  const int per_thread = (32 * UPR + NT - 1) / NT;
  u32x4 stg[PT];  // per_thread <= PT for every supported (K, workgroup size) pair
  auto stage_load = [&](int64_t tile) {
#pragma unroll
    for (int k = 0; k < PT; ++k) {
      const int idx = k * NT + tid;
      stg[k] = u32x4{0, 0, 0, 0};
      if (k < per_thread && idx < 32 * UPR) {
        const int rc = idx / UPR, pos = idx - rc * UPR;
        const int64_t m = real_row(tile * 32 + rc);
        if (m >= 0) stg[k] = *reinterpret_cast<const u32x4 *>(in + m * K + pos * 8);
      }
    }
  };
  auto stage_store = [&](int buf) {
#pragma unroll
    for (int k = 0; k < PT; ++k) {
      const int idx = k * NT + tid;
      if (k < per_thread && idx < 32 * UPR) {
        const int rc = idx / UPR, pos = idx - rc * UPR;
        xs[buf][rc * ROWU + pos] = stg[k];
      }
    }
  };

  int64_t tile = blockIdx.x;
  if (tile < ntiles) {
    stage_load(tile);
    stage_store(0);
  }
  __syncthreads();
  int buf = 0;
  for (; tile < ntiles; tile += gridDim.x, buf ^= 1) {
    const int64_t next = tile + gridDim.x < ntiles ? tile + gridDim.x : tile;  // the last tile re-fetches itself
    stage_load(next);
    const u32x4 *xb = &xs[buf][i * ROWU + g];
    f32x16 acc_t, acc_n;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      acc_t[r] = LEAN ? bias_s[wave * 32 + mfma::rowmap(r, g)] : bias_t[r];
      acc_n[r] = bias_n;
    }
    if (pk) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const u32x4 xf = xb[2 * ks];
        acc_t = mfma::mma(wf[ks], xf, acc_t);
        acc_n = mfma::mma(xf, wf[ks], acc_n);
      }
    } else {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) acc_t = mfma::mma(wf[ks], xb[2 * ks], acc_t);
    }
    if (out) {
      const int64_t m = real_row(tile * 32 + i);
      mfma::store_tile_natural(acc_t, out + (m >= 0 ? m : 0) * a.O + o0, g, m >= 0);
    }
    if (pk) {
      const int head = o0 >> 5;
      pk[((tile * a.pack_heads + head) * 2 + 0) * 64 + lane] = mfma::pack_half<0>(acc_n);
      pk[((tile * a.pack_heads + head) * 2 + 1) * 64 + lane] = mfma::pack_half<1>(acc_n);
    }
    stage_store(buf ^ 1);
    __syncthreads();
  }
}

// ------------------------------------------------------------------------------------------------
// rows_linear_ring_kernel: the same for K = 512 in natural layout, 256 columns per workgroup.  The weights take 128 registers, so one
// workgroup owns a CU, and what hides memory's latency is what it alone has on its way: the rows go from memory straight into a ring of
// four 32-row tiles in LDS (33 KB each), three of them in flight while one is multiplied, one barrier per tile.  One load is one row of
// 1 024 bytes; rows lie 16 bytes more apart, so that the lanes of an access phase (32 rows, one unit) fall on different banks.
// Loads and stores leave the counter in order: behind a tile's four loads a wave has issued the loads of up to two tiles and the two
// stores each of up to three.  Bound by HBM: 1 048 576 rows into 256 columns, with rows_linear_kernel / here, in a layer's training step
// 412 / 297 us (5.4 TB/s); called again and again, the two in turn, 4 096 rows (the fewest that come here) 11.1 / 10.5, 12 000 13.5 / 13.3,
// 30 000 18.3 / 18.5, 65 536 27.3 / 27.0, 131 072 49.2 / 45.0, 262 144 94 / 85; into 512 columns 11.4 / 10.9, 16.4 / 15.5, 26.9 / 24.8,
// 44.4 / 41.7, 86 / 76, 168 / 147: 1 % slower at one of twelve sizes (30 000 x 256), which is no reason for a line.
// ------------------------------------------------------------------------------------------------
struct LinearRing {
  static constexpr int K = 512, KS = K / 16, ROWU = K / 8 + 1, TILE = 32 * ROWU * 16, STAGES = 4, BYTES = STAGES * TILE + 256 * 4;
};

__global__ __launch_bounds__(512, 2) void rows_linear_ring_kernel(GemmArgs a) {
  using Q = LinearRing;
  constexpr int K = Q::K;
  extern __shared__ u32x4 xs_all[];
  float *bias_s = reinterpret_cast<float *>(xs_all + Q::STAGES * (Q::TILE / 16));
  const int z = blockIdx.z;
  const uint16_t *in = static_cast<const uint16_t *>(a.in);
  const uint16_t *W = static_cast<const uint16_t *>(a.w[z]);
  const int tid = threadIdx.x, lane = tid & 63, i = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int o0 = blockIdx.y * 256 + wave * 32;  // this wave's output columns

  const int64_t ntiles = (a.M + 31) / 32, stride = gridDim.x;  // grid.x <= ntiles: a workgroup has a tile
  auto fetch = [&](int64_t tile, int stage) {
    if (tile >= ntiles) return;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int row = 4 * wave + k;
      const int64_t m = tile * 32 + row < a.M ? tile * 32 + row : a.M - 1;  // past the last row: that one
      mfma::load_unit_to_lds(in + m * K, lane * 16, (unsigned)(uintptr_t)xs_all + stage * Q::TILE + row * (Q::ROWU * 16));
    }
  };
  int64_t tile = blockIdx.x;
  fetch(tile, 0);
  const float bias = tid < 256 && a.bias[z] ? a.bias[z][blockIdx.y * 256 + tid] : 0.f;
  u32x4 wf[Q::KS];  // W[o0 + i][16 ks + 8 g + j]
#pragma unroll
  for (int ks = 0; ks < Q::KS; ++ks) wf[ks] = *reinterpret_cast<const u32x4 *>(W + (int64_t)(o0 + i) * K + 16 * ks + 8 * g);
#pragma unroll
  for (int ks = 0; ks < Q::KS; ++ks) asm volatile("" : "+v"(wf[ks]));  // they are waited for here and not in the loop
  if (tid < 256) bias_s[tid] = bias;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // with the first tile: the loop counts from here
#pragma unroll
  for (int s = 1; s < Q::STAGES - 1; ++s) fetch(tile + s * stride, s);
  int stage = 0, done = 0;  // done: tiles whose stores may be on their way, at most three
  for (; tile < ntiles; tile += stride) {
    const int later = tile + 2 * stride < ntiles ? 2 : tile + stride < ntiles ? 1 : 0;  // tiles behind this one that are on their way
    switch (2 * later + done) {
      case 0: asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); break;
      case 1: asm volatile("s_waitcnt vmcnt(2)" ::: "memory"); break;
      case 2: asm volatile("s_waitcnt vmcnt(4)" ::: "memory"); break;
      case 3: asm volatile("s_waitcnt vmcnt(6)" ::: "memory"); break;
      case 4: asm volatile("s_waitcnt vmcnt(8)" ::: "memory"); break;
      case 5: asm volatile("s_waitcnt vmcnt(10)" ::: "memory"); break;
      case 6: asm volatile("s_waitcnt vmcnt(12)" ::: "memory"); break;
      default: asm volatile("s_waitcnt vmcnt(14)" ::: "memory"); break;
    }
    done = done < 3 ? done + 1 : 3;
    __syncthreads();  // every wave's rows of the tile are there, and every wave is past the tile before
    fetch(tile + (Q::STAGES - 1) * stride, (stage + Q::STAGES - 1) % Q::STAGES);
    const u32x4 *xb = xs_all + stage * (Q::TILE / 16) + i * Q::ROWU + g;
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = bias_s[wave * 32 + mfma::rowmap(r, g)];
#pragma unroll
    for (int ks = 0; ks < Q::KS; ++ks) acc = mfma::mma(wf[ks], xb[2 * ks], acc);
    // stores past the last row are dropped by the buffer's range, so that every tile counts two of them
    const int64_t row0 = tile * 32;
    const int have = (int)(a.M - row0 < 32 ? a.M - row0 : 32);
    const auto rows = __builtin_amdgcn_make_buffer_rsrc(static_cast<uint16_t *>(a.out[z]) + row0 * a.O, 0, have * a.O * 2, 0x00027000);
    u32x4 s0, s1;
    mfma::tile_natural(acc, s0, s1);
    const int at = (i * a.O + o0 + 16 * g) * 2;
    __builtin_amdgcn_raw_buffer_store_b128(s0, rows, at, 0, 0);
    __builtin_amdgcn_raw_buffer_store_b128(s1, rows, at + 16, 0, 0);
    stage = (stage + 1) % Q::STAGES;
  }
}

bool linear_serves(const GemmArgs &a, int nsets, size_t elem_bytes) {
  if (elem_bytes != 2 || a.ks != 0 || a.act != 0) return false;  // activations: the tiled kernel
  if (a.K != 128 && a.K != 256 && a.K != 512) return false;
  if (a.O % 32 != 0 || (a.O > 256 && a.O % 256 != 0)) return false;
  if (a.M < 4096) return false;  // small problems: the tiled kernel has less fixed cost
  if ((a.O < 256 ? a.O : 256) * 2 < a.K) return false;  // staging: at most 4 units per thread and tile
  if (!aligned16(a.in)) return false;
  for (int z = 0; z < nsets; ++z)
    if (!aligned16(a.w[z]) || !aligned16(a.out[z]) || (!a.out[z] && !a.out_pack[z])) return false;
  return true;
}

int linear_launch(const GemmArgs &a, int nsets, int num_cu, hipStream_t st) {
  const int64_t ntiles = a.pack_tpb > 0 ? (a.M / a.N) * a.pack_tpb : (a.M + 31) / 32;
  const int waves = (a.O < 256 ? a.O : 256) / 32;
  // resident workgroups: the register-held weights leave room for one 8-wave workgroup per CU, two for K = 128 and the
  // lean form.  The second one of the lean form pays from eight tiles per CU on, where its weights (128 KB) are covered:
  // 256 -> 256, two against one: 16 384 rows 12.0 / 9.1 us, 32 768 14.5 / 12.5; from 65 536 rows against one of the other
  // form: 19.5 / 20.8, 1 048 576 rows 211 / 227.
  const bool natural = a.O % 256 == 0 && a.pack_tpb == 0 && !a.out_pack[0] && !a.out_pack[nsets - 1], lean = a.K == 256 && natural;
  const int64_t sides = (a.O + 255) / 256 * nsets;
  int64_t gx = (a.K == 128 || (lean && ntiles * sides >= 8 * (int64_t)num_cu) ? 2 : 1) * (int64_t)num_cu / sides;
  if (gx < 1) gx = 1;
  if (gx > ntiles) gx = ntiles;
  const dim3 grid((unsigned)gx, (unsigned)((a.O + 255) / 256), (unsigned)nsets), block((unsigned)(waves * 64));
  if (a.K == 512 && natural) {
    if (int rc = allow_dynamic_lds(rows_linear_ring_kernel, LinearRing::BYTES)) return rc;
    hipLaunchKernelGGL(rows_linear_ring_kernel, grid, block, LinearRing::BYTES, st, a);
    return launch_status();
  }
  const size_t lds = (size_t)2 * 32 * (a.K / 8 + 1) * 16;  // only K = 512 exceeds the default limit
  if (int rc = allow_dynamic_lds(rows_linear_kernel<32, false>, a.K == 512 ? lds : 0)) return rc;
  switch (a.K) {
    case 128: hipLaunchKernelGGL((rows_linear_kernel<8, false>), grid, block, lds, st, a); break;
    case 256:
      if (lean) hipLaunchKernelGGL((rows_linear_kernel<16, true>), grid, block, lds, st, a);
      else hipLaunchKernelGGL((rows_linear_kernel<16, false>), grid, block, lds, st, a);
      break;
    case 512: hipLaunchKernelGGL((rows_linear_kernel<32, false>), grid, block, lds, st, a); break;
    default: return PA_ERR_UNSUPPORTED;
  }
  return launch_status();
}

// ------------------------------------------------------------------------------------------------
// cols_gemm_kernel: weight-gradient products  P[oa][ob] = sum_m A[m][oa] * B[m][ob]  over a huge row count m (bf16
// rows in natural layout, fp32 result).  grid (G row chunks, OA / 256); workgroup = one wave per 32 columns of A (up to
// 8); wave w owns output rows 32w..32w+31 and all NB = OB / 32 column groups.  Both operands have the reduction index m
// as their slow index in memory, so each 32-row block is transposed on the matrix cores first: the natural 16-byte
// loads are MFMA A operands (lane <-> row m, k <-> channel); multiplied by 0/1 selection matrices they give an exact copy
// of the block with lanes <-> channels and registers <-> rows, which, converted back to bf16, is an operand whose
// reduction index is m.  Every wave transposes its own A group; the B groups are transposed once per workgroup and
// shared through LDS (double buffered, one barrier per block).  Each chunk leaves one partial result
// partials[g][oa][ob]; the caller adds the G partials up in index order.
// ------------------------------------------------------------------------------------------------
template <int NB>
__global__ __launch_bounds__(512) void cols_gemm_kernel(const uint16_t *__restrict__ A, int lda, int OA,
                                                        const uint16_t *__restrict__ B, int ldb, int64_t M,
                                                        int64_t blocks_per_chunk, float *__restrict__ partials,
                                                        float *__restrict__ col_sums) {
  constexpr int OB = 32 * NB;
  __shared__ u32x4 bts[2][NB * 2 * 64];
  const int tid = threadIdx.x, lane = tid & 63, i = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nwaves = blockDim.x >> 6;
  const int a0 = blockIdx.y * 256 + wave * 32;  // first A column of this wave

  u32x4 sel[2];  // sel[kk]: column i receives the k element whose channel is 16kk + 8g + j
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    mfma::bf16x8 s8;
#pragma unroll
    for (int j = 0; j < 8; ++j) s8[j] = (__bf16)((i == 16 * kk + 8 * g + j) ? 1.f : 0.f);
    sel[kk] = __builtin_bit_cast(u32x4, s8);
  }
  // a 32 x 32 block (rows m0.., columns c0..) of a natural-layout matrix -> two operands whose k index runs over m
  auto transposed = [&](const uint16_t *base, int ld, int64_t m0, int c0, u32x4 &t0, u32x4 &t1) {
    const int64_t m = m0 + i;
    u32x4 f0 = u32x4{0, 0, 0, 0}, f1 = f0;
    if (m < M) {
      const uint16_t *row = base + m * ld + c0 + 8 * g;
      f0 = *reinterpret_cast<const u32x4 *>(row);
      f1 = *reinterpret_cast<const u32x4 *>(row + 16);
    }
    f32x16 t;
#pragma unroll
    for (int r = 0; r < 16; ++r) t[r] = 0.f;
    t = mfma::mma(f0, sel[0], t);
    t = mfma::mma(f1, sel[1], t);
    t0 = mfma::pack_half<0>(t);
    t1 = mfma::pack_half<1>(t);
  };

  f32x16 acc[NB], acc_s;  // acc_s: A^T . 1 (every column the same): the column sums of A
#pragma unroll
  for (int r = 0; r < 16; ++r) acc_s[r] = 0.f;
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[nb][r] = 0.f;
  const u32x4 ones = u32x4{0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};  // 8 x bf16(1.0)

  const int64_t blk0 = (int64_t)blockIdx.x * blocks_per_chunk;
  const int64_t nblk = (M + 31) / 32;
  int64_t blk_end = blk0 + blocks_per_chunk;
  if (blk_end > nblk) blk_end = nblk;
  int buf = 0;
  for (int64_t blk = blk0; blk < blk_end; ++blk, buf ^= 1) {
    const int64_t m0 = blk * 32;
    u32x4 at0, at1;
    transposed(A, lda, m0, a0, at0, at1);
    if (col_sums) {
      acc_s = mfma::mma(at0, ones, acc_s);
      acc_s = mfma::mma(at1, ones, acc_s);
    }
    for (int nb = wave; nb < NB; nb += nwaves) {
      u32x4 b0, b1;
      transposed(B, ldb, m0, 32 * nb, b0, b1);
      bts[buf][(nb * 2 + 0) * 64 + lane] = b0;
      bts[buf][(nb * 2 + 1) * 64 + lane] = b1;
    }
    __syncthreads();
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      acc[nb] = mfma::mma(at0, bts[buf][(nb * 2 + 0) * 64 + lane], acc[nb]);
      acc[nb] = mfma::mma(at1, bts[buf][(nb * 2 + 1) * 64 + lane], acc[nb]);
    }
  }
  float *dst = partials + ((int64_t)blockIdx.x * OA + a0) * OB;
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int r = 0; r < 16; ++r) dst[(int64_t)mfma::rowmap(r, g) * OB + 32 * nb + i] = acc[nb][r];
  if (col_sums && i == 0) {
#pragma unroll
    for (int r = 0; r < 16; ++r) col_sums[(int64_t)blockIdx.x * OA + a0 + mfma::rowmap(r, g)] = acc_s[r];
  }
}

// row chunks: about two workgroups per CU over all column groups, and at least 32 blocks of 32 rows per chunk so that
// ------------------------------------------------------------------------------------------------
// cols_gemm_f32_kernel: the float32 form of the weight-gradient product  P[oa][ob] = sum_m A[m][oa] * B[m][ob].
// v_mfma_f32_32x32x2_f32 reduces over two rows m per instruction with lane (i, g) supplying one value of row m0 + g of either
// operand: consecutive lanes hold consecutive columns of a row, so natural row-major operands need no transposition.  A workgroup
// (4 waves) owns a 128 x 128 block of P for one chunk of rows, wave w the 64 x 64 sub-block (w & 1, w >> 1); lane i takes columns
// 2 i and 2 i + 1 of both operands, one 8-byte load each per pair of rows, for the 4 MFMAs (256 cycles) of the pair.  The operands
// go straight from memory to registers, 16 pairs (32 rows) ahead: at this rate four waves ask for 16 bytes a cycle, 8 of them
// beyond the L1 where the two waves that share a column meet there, and no wave waits for another.  Rows beyond the chunk and
// neighbours outside the grid are out of the buffers' range and read as zero.
// Row chunks come back as partials P[g][oa][ob] (fixed-order sum by the caller); col_sums[g][oa] = sum_m A[m][oa] from the same
// pass.  Workgroups that share a chunk (the blocks of columns, the taps) run on one XCD, one after the other.
// Bound by the float32 MFMAs: 4 x 85 x 85 grid points, 3 x 3 taps, 128 -> 2 x 128 (17 GFLOP) 149 us, 128 x 128 over 28 900 rows 16 us;
// through LDS, one barrier per 32 rows, 176 and 20; with all loads of a block behind its matrix instructions 169 and 20.
// ------------------------------------------------------------------------------------------------
constexpr int kF32Tile = 128, kF32Rows = 32;

__global__ __launch_bounds__(256, 2) void cols_gemm_f32_kernel(const float *__restrict__ A, int lda, int OA,
                                                               const float *__restrict__ B, int ldb, int OB, int64_t M,
                                                               int64_t rows_per_chunk, int chunks, GridTaps grid,
                                                               float *__restrict__ partials, float *__restrict__ col_sums) {
  typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
  constexpr int kPairs = kF32Rows / 2;
  constexpr unsigned kOut = 0x80000000u;  // an offset no buffer here reaches
  const int t = threadIdx.x, lane = t & 63, i = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int noa = (OA + kF32Tile - 1) / kF32Tile, nob = (OB + kF32Tile - 1) / kF32Tile, tiles = noa * nob * grid.taps;
  // the (chunk, tile) pairs in chunk-major order are dealt out to the XCDs (= workgroup id mod 8) in eight equal runs
  const int item = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  const int chunk = __builtin_amdgcn_readfirstlane(item / tiles), tile = item - chunk * tiles;
  if (chunk >= chunks) return;
  const int zt = __builtin_amdgcn_readfirstlane(tile / noa), tap = __builtin_amdgcn_readfirstlane(zt / nob);
  const int oa0 = (tile - zt * noa) * kF32Tile, ob0 = (zt - tap * nob) * kF32Tile;
  const int64_t m_begin = (int64_t)chunk * rows_per_chunk;
  const int64_t m_end = M < m_begin + rows_per_chunk ? M : m_begin + rows_per_chunk;
  const int wa = (wave & 1) * 64, wb = (wave >> 1) * 64;  // this wave's sub-block of the tile

  f32x16 acc[2][2];
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int v = 0; v < 2; ++v)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[u][v][r] = 0.f;
  float csum[2] = {0.f, 0.f};

  // Convolution: row m's neighbour at this tap is row m + shift where that lies inside the grid.  Lane l looks after row l % 32 of
  // a block: its grid coordinates are divided out once and then advanced by the 32 rows of a block with carries.
  const bool conv = grid.ks > 0;
  const int gd = grid.gd > 0 ? grid.gd : 1, gw = conv ? grid.gw : 1, gh = conv ? grid.gh : 1, ksd = grid.gd > 0 ? grid.ks : 1;
  const int pad = grid.ks / 2, pad_d = grid.gd > 0 ? pad : 0;
  const int uv = conv ? __builtin_amdgcn_readfirstlane(tap / ksd) : 0, tap_u = conv ? __builtin_amdgcn_readfirstlane(uv / grid.ks) : 0;
  const int tu = tap_u - pad, tv = uv - tap_u * grid.ks - pad, tz = tap - uv * ksd - pad_d;
  const int64_t shift = conv ? ((int64_t)tu * gw + tv) * gd + tz : 0;
  const int step_l = kF32Rows % gd, step_j = kF32Rows / gd % gw, step_i = kF32Rows / gd / gw;
  unsigned n0 = conv ? (unsigned)((m_begin + i) % grid.N) : 0u;
  int cl = (int)(n0 % gd), cj = (int)(n0 / gd % gw), ci = (int)(n0 / gd / gw);
  // byte offsets of this lane's columns in the first pair of a block
  const int ca = oa0 + wa + 2 * i, cb = ob0 + wb + 2 * i;
  const unsigned a_off = ca < OA ? (unsigned)(g * lda + ca) * 4u : kOut, b_off = cb < OB ? (unsigned)(g * ldb + cb) * 4u : kOut;
  u32x2 av[kPairs], bv[kPairs];  // the operands of a block of rows
  const float *pa = A + m_begin * lda, *pb = B + (m_begin + shift) * ldb;  // the block requested next (pb: may lie before B, unread)
  int left = (int)(m_end - m_begin);                                       // rows from there to the chunk's end
  unsigned outside = 0;  // bit 2 p: this lane's row of pair p has no neighbour
  __amdgpu_buffer_rsrc_t ra, rb;
  auto resource = [](const float *p, int bytes) {  // wave-uniform, and said to be
    const uint64_t at = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((int)(uint32_t)at), hi = __builtin_amdgcn_readfirstlane((int)(uint32_t)(at >> 32));
    return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void *>((uint64_t)hi << 32 | lo), 0,
                                             __builtin_amdgcn_readfirstlane(bytes), 0x00027000);
  };
  auto next_block = [&]() {
    if (conv) {
      const bool in = ((unsigned)(ci + tu) < (unsigned)gh) & ((unsigned)(cj + tv) < (unsigned)gw) & ((unsigned)(cl + tz) < (unsigned)gd);
      outside = ~(unsigned)__builtin_amdgcn_ballot_w64(in) >> g;
      cl += step_l, cj += step_j, ci += step_i;
      if (cl >= gd) cl -= gd, ++cj;
      if (cj >= gw) cj -= gw, ++ci;
      ci = (int)((unsigned)ci % (unsigned)gh);  // the next batch element; no loop: the loads in flight would be waited for
    }
    const int rows = left < 0 ? 0 : left < kF32Rows ? left : kF32Rows;
    ra = resource(pa, rows * lda * 4), rb = resource(pb, rows * ldb * 4);
    pa += (int64_t)kF32Rows * lda, pb += (int64_t)kF32Rows * ldb;
    left -= kF32Rows;
  };
  auto request = [&](int p) {
    av[p] = __builtin_amdgcn_raw_buffer_load_b64(ra, a_off + (unsigned)(8 * p * lda), 0, 0);
    bv[p] = __builtin_amdgcn_raw_buffer_load_b64(rb, (b_off + (unsigned)(8 * p * ldb)) | ((outside << (31 - 2 * p)) & kOut), 0, 0);
  };
  next_block();
#pragma unroll
  for (int p = 0; p < kPairs; ++p) {
    request(p);
    __builtin_amdgcn_sched_barrier(0);  // in the order in which the loop waits for them
  }
  for (int64_t m0 = m_begin; m0 < m_end; m0 += kF32Rows) {
    next_block();  // behind the last one: no rows, every load a zero
#pragma unroll
    for (int p = 0; p < kPairs; ++p) {
      const uint32_t w[4] = {av[p][0], av[p][1], bv[p][0], bv[p][1]};
      const float a0 = __uint_as_float(w[0]), a1 = __uint_as_float(w[1]), b0 = __uint_as_float(w[2]), b1 = __uint_as_float(w[3]);
      acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0, b0, acc[0][0], 0, 0, 0);
      acc[0][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0, b1, acc[0][1], 0, 0, 0);
      acc[1][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, b0, acc[1][0], 0, 0, 0);
      acc[1][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, b1, acc[1][1], 0, 0, 0);
      csum[0] += a0;
      csum[1] += a1;
      request(p);
      __builtin_amdgcn_sched_barrier(0);  // the requests stay between the matrix instructions, a block ahead of their use
    }
  }
  // C/D layout: lane (i, g) holds column 2 i + v, register r holds row 2 rowmap(r, g) + u of the sub-block
  const int64_t ld = (int64_t)grid.taps * OB;
  const int row0 = oa0 + wa, rows = OA - row0 < 64 ? OA - row0 : 64;  // of the sub-block
  if (rows > 0) {
    const auto out = resource(partials + ((int64_t)chunk * OA + row0) * ld + (int64_t)tap * OB, (int)((rows - 1) * ld + OB) * 4);
    const unsigned at = cb < OB ? (unsigned)cb * 4u : kOut, step = (unsigned)ld * 4u;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int r = 0; r < 16; ++r)  // rows beyond OA are out of range
        __builtin_amdgcn_raw_buffer_store_b64(u32x2{__float_as_uint(acc[u][0][r]), __float_as_uint(acc[u][1][r])}, out,
                                              at + (unsigned)(2 * mfma::rowmap(r, g) + u) * step, 0, 0);
  }
  if (col_sums && zt == 0 && (wave >> 1) == 0) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const float total = csum[u] + __shfl_xor(csum[u], 32, 64);  // the two row parities
      if (g == 0 && ca < OA) col_sums[(int64_t)chunk * OA + ca + u] = total;
    }
  }
}

// Two workgroups per compute unit in all, and no more chunks than pay for their partial results: 32 rows of a tile take
// about 2 us, a partial of n values about 2 n ps to write and read back, their sum is smallest at sqrt(3e4 M / n).
int64_t cols_gemm_f32_chunks(int64_t M, int64_t OA, int64_t OB, int num_cu) {
  const int64_t tiles = ((OA + kF32Tile - 1) / kF32Tile) * ((OB + kF32Tile - 1) / kF32Tile);
  int64_t g = 2 * (int64_t)num_cu / tiles, best = 1;
  while ((best + 1) * (best + 1) <= 30000 * M / (OA * OB)) ++best;
  if (g > best) g = best;
  const int64_t cap = (M + 63) / 64;
  if (g > cap) g = cap;
  return g < 1 ? 1 : g;
}

// `shape` with conv_k > 0: B's rows are the neighbours at every tap, the partials [g][oa][tap][ob]
int cols_gemm_f32(const void *A, int64_t lda, int64_t OA, const void *B, int64_t ldb, int64_t OB, int64_t M,
                  const pa_shape *shape, float *partials, float *col_sums, int num_cu, hipStream_t st) {
  if (OA <= 0 || OB <= 0 || OA % 4 != 0 || OB % 4 != 0 || lda % 4 != 0 || ldb % 4 != 0) return PA_ERR_UNSUPPORTED;
  const GridTaps grid_geom = grid_taps(shape);
  const int64_t G = cols_gemm_f32_chunks(M, OA, OB * grid_geom.taps, num_cu);
  int64_t per = (M + G - 1) / G;
  per = (per + kF32Rows - 1) / kF32Rows * kF32Rows;
  const int64_t wgs = G * ((OA + kF32Tile - 1) / kF32Tile) * ((OB + kF32Tile - 1) / kF32Tile) * grid_geom.taps;
  hipLaunchKernelGGL(cols_gemm_f32_kernel, dim3((unsigned)((wgs + 7) / 8 * 8)), dim3(256), 0, st, static_cast<const float *>(A),
                     (int)lda, (int)OA, static_cast<const float *>(B), (int)ldb, (int)OB, M, per, (int)G, grid_geom, partials,
                     col_sums);
  return launch_status();
}

// the partial results stay small next to the rows a chunk reads
int64_t cols_gemm_chunks(int64_t M, int64_t OA, int num_cu) {
  const int64_t nblk = (M + 31) / 32, gy = (OA + 255) / 256;
  int64_t g = 2 * (int64_t)num_cu / gy;
  if (g > nblk / 32) g = nblk / 32;
  return g < 1 ? 1 : g;
}

int cols_gemm(const void *A, int64_t lda, int64_t OA, const void *B, int64_t ldb, int64_t OB, int64_t M,
              float *partials, float *col_sums, int num_cu, hipStream_t st) {
  if (OA % 32 != 0 || OB % 32 != 0 || OA <= 0 || OB <= 0 || lda % 8 != 0 || ldb % 8 != 0) return PA_ERR_UNSUPPORTED;
  if (OA > 256 && OA % 256 != 0) return PA_ERR_UNSUPPORTED;
  const int64_t G = cols_gemm_chunks(M, OA, num_cu);
  const int64_t nblk = (M + 31) / 32;
  const int64_t per = (nblk + G - 1) / G;
  const dim3 grid((unsigned)G, (unsigned)((OA + 255) / 256)), block((unsigned)((OA < 256 ? OA : 256) * 2));
  const uint16_t *a = static_cast<const uint16_t *>(A), *b = static_cast<const uint16_t *>(B);
  if (OA >= 128 && OB >= 128 && OB <= 256)  // wide products (the 256 x 256 tile would idle on narrow ones)
    return wgrad::launch_wide(A, lda, OA, B, ldb, OB, M, G, nullptr, partials, col_sums, st);
#define PA_COLS(NBV) \
  hipLaunchKernelGGL((cols_gemm_kernel<NBV>), grid, block, 0, st, a, (int)lda, (int)OA, b, (int)ldb, M, per, partials, col_sums)
  switch (OB / 32) {
    case 1: PA_COLS(1); break;
    case 2: PA_COLS(2); break;
    case 4: PA_COLS(4); break;
    case 8: PA_COLS(8); break;
    default: return PA_ERR_UNSUPPORTED;
  }
#undef PA_COLS
  return launch_status();
}

// ------------------------------------------------------------------------------------------------
// conv_gemm_kernel: the grid convolutions as implicit GEMM (rows x taps * channels) . W^T with whole steps of 128 bytes of
// channels (64 bf16, 32 float32) of one tap.  Workgroup: bf16 8 waves, 128 rows x 256 outputs, wave tile 64 x 64; float32
// 128 outputs, wave tile 32 x 64, 8 waves and 128 rows (TALL) or 4 and 64 (conv_tall() below).  One step of both operands (48, 32 or
// 24 KB) is a stage; three, four or six stages form a ring in LDS, filled one stage less ahead by direct global -> LDS loads (the
// neighbours' rows are gathered by their addresses, a unit of zeros outside the grid), one barrier per step.  The loads
// write 8 rows of 128 bytes contiguously, so position p of row r holds the row's 16-byte unit p ^ (r % 8): the eight
// lanes of an access phase then fall on all banks.
// Outputs: rows as 16-byte pieces (the product formed as out^T, lanes <-> rows), or with `out_pack` the un-transposed
// tile, in the packed operand layout and as 2-byte pieces of rows.
// bf16: bound by LDS reads (one 1 KB fragment per MFMA and wave: 128 bytes a cycle) and by issue.  32 768 grid points, 3 x 3, 256 -> 2 x
// 256 and 512 -> 256 (77 GFLOP each): 79 us; 95 with a step's addresses formed in full (64-bit products) ahead of its matrix
// instructions, 88 with them between these.  rows_gemm_mfma_kernel (registers one step ahead, two barriers per step, no ring): 254
// and 219 us.
// float32: bound by v_mfma_f32_32x32x2_f32 and by whole rounds of workgroups: 4 x 85 x 85 points, 128 -> 2 x 128 and 256 -> 128 (17
// GFLOP each) 162 us against 177 (addresses in full, two 64-row workgroups of three stages per CU: the one that came second took 95 us,
// the first 75); 57 600 points 322 against 348; 1 600 points 62 against 70.
// ------------------------------------------------------------------------------------------------
template <typename T, bool TALL>
struct ConvTile {  // waves: WR along the rows, WC along the outputs; a wave stages 16 rows and OW weight rows of a step
  static constexpr int RT = sizeof(T) == 2 ? 2 : 1, WR = sizeof(T) == 4 && TALL ? 4 : 2, WC = sizeof(T) == 2 ? 4 : 2, kWaves = WR * WC;
  static constexpr int kRows = 32 * RT * WR, kOut = 64 * WC, kStageBytes = (kRows + kOut) * 128, KB = 128 / (int)sizeof(T);
  static constexpr int OW = kOut / kWaves, kLoads = 2 + OW / 8, kStages = sizeof(T) == 2 ? 3 : TALL ? 4 : 6;
};

template <typename T, bool TALL>
__global__ __launch_bounds__((ConvTile<T, TALL>::kWaves * 64)) void conv_gemm_kernel(GemmArgs a) {
  using Q = ConvTile<T, TALL>;
  constexpr int RT = Q::RT, UE = Unit<T>::kElems, kConvStages = Q::kStages;
  extern __shared__ u32x4 ring[];  // [stage][kRows input rows | kOut weight rows] of 128 bytes
  const int z = blockIdx.z, t = threadIdx.x, lane = t & 63, i = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6), wr = wave % Q::WR * (32 * RT), wc = wave / Q::WR * 64;
  const T *in = static_cast<const T *>(a.in);
  const int64_t m0 = (int64_t)blockIdx.x * Q::kRows;
  const int o0 = blockIdx.y * Q::kOut;
  const int gd = a.gd > 0 ? a.gd : 1, ksd = a.gd > 0 ? a.ks : 1, pad = a.ks / 2, pad_d = a.gd > 0 ? pad : 0;
  // rows are numbered as in rows_gemm_mfma_kernel: first real row of 32-row tile `tile`, and how many of its rows exist
  const unsigned tpb = a.pack_tpb > 0 ? (unsigned)a.pack_tpb : 0u;
  auto tile_rows = [&](unsigned tile, int64_t &first, int &count) {
    const unsigned b = tpb ? tile / tpb : 0u;
    first = tpb ? (int64_t)b * a.N + (int64_t)(tile - b * tpb) * 32 : (int64_t)tile * 32;
    const int64_t end = tpb && (int64_t)(b + 1) * a.N < a.M ? (int64_t)(b + 1) * a.N : a.M, left = end - first;
    count = left < 0 ? 0 : left < 32 ? (int)left : 32;
  };
  // this wave stages input rows 16 wave + 8 k + lane / 8 (k = 0, 1) and weight rows OW wave + 8 k + lane / 8
  const int unit = (lane & 7) ^ (lane >> 3);
  const T *base[2], *wu = static_cast<const T *>(a.w[z]) + (int64_t)(o0 + Q::OW * wave) * a.K;  // wu: wave-uniform
  const int w_off = ((lane >> 3) * a.K + UE * unit) * (int)sizeof(T);
  int ci[2], cj[2], cl[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    int64_t first;
    int count;
    tile_rows((unsigned)(m0 / 32) + (wave >> 1), first, count);
    const int local = 16 * (wave & 1) + 8 * k + (lane >> 3);
    const int64_t m = local < count ? first + local : 0;
    unsigned n = (unsigned)(m % a.N);
    cl[k] = (int)(n % gd);
    n /= gd;
    ci[k] = local < count ? (int)(n / a.gw) : -(1 << 20);  // no row: never inside the grid
    cj[k] = (int)(n % a.gw);
    base[k] = in + m * a.C + UE * unit;
  }
  const int nkb = a.K / Q::KB, cblocks = a.C / Q::KB;
  int fu = 0, fv = 0, fz = 0, fc = 0;  // tap and channel block of the step fetched next
  // The addresses of a step are the ones before it plus 128 bytes, but at a new tap: formed in full at every step, 64-bit products
  // included, they cost as much issue time as the matrix instructions between which they stood.
  const char *xp[2];
  int x_step[2];
  auto enter_tap = [&]() {
    const int64_t shift = (((int64_t)(fu - pad) * a.gw + fv - pad) * gd + fz - pad_d) * a.C;  // the neighbour, from the row
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const bool ok = ((unsigned)(ci[k] + fu - pad) < (unsigned)a.gh) & ((unsigned)(cj[k] + fv - pad) < (unsigned)a.gw) &
                      ((unsigned)(cl[k] + fz - pad_d) < (unsigned)gd);
      xp[k] = ok ? reinterpret_cast<const char *>(base[k] + shift) : reinterpret_cast<const char *>(&mfma::kZeroUnit);
      x_step[k] = ok ? 128 : 0;
    }
  };
  enter_tap();
  const unsigned ring0 = (unsigned)(uintptr_t)ring;
  unsigned slot = 0;  // of the ring, in bytes: where the next step goes
  // a step's loads in four parts between the matrix instructions; past the last step: that one again, so that every step counts as
  // many loads
  auto fetch_part = [&](int kb, auto part_) {
    constexpr int part = decltype(part_)::value;
    const unsigned dst = ring0 + slot;
    if constexpr (part < 2) {
      mfma::load_unit_to_lds(xp[part], dst + (16 * wave + 8 * part) * 128);
    } else {
#pragma unroll
      for (int k = 2 * part - 4; k < 2 * part - 2 && k < Q::OW / 8; ++k)
        mfma::load_unit_to_lds(wu + (int64_t)8 * k * a.K, w_off, dst + Q::kRows * 128 + (Q::OW * wave + 8 * k) * 128);
    }
    if constexpr (part == 3) {
      slot = slot == (kConvStages - 1) * Q::kStageBytes ? 0 : slot + Q::kStageBytes;
      if (kb + 1 < nkb) {
        wu += Q::KB;
        xp[0] += x_step[0], xp[1] += x_step[1];
        if (++fc == cblocks) {
          fc = 0;
          if (++fz == ksd) {
            fz = 0;
            if (++fv == a.ks) fv = 0, ++fu;
          }
          enter_tap();
        }
      }
    }
  };
  auto fetch = [&](int kb) { mfma::static_for<4>([&](auto part) { fetch_part(kb, part); }); };
  f32x16 acc[2][RT];  // [output tile][row tile]
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int v = 0; v < RT; ++v)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[u][v][r] = 0.f;
  u32x4 *pk = static_cast<u32x4 *>(a.out_pack[z]);
  const int row_off = i * 8, swz = i & 7;
  auto multiply = [&](auto turned_) {
    constexpr bool turned = decltype(turned_)::value;
    mfma::static_for<kConvStages - 1>([&](auto s) { fetch(decltype(s)::value); });
    unsigned at_slot = 0;
    for (int kb = 0; kb < nkb; ++kb) {
      // this wave's share of the step; the younger ones stay in flight
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kConvStages - 2) * Q::kLoads) : "memory");
      __syncthreads();
      const u32x4 *xs = ring + at_slot / 16 + wr * 8 + row_off, *ws = ring + at_slot / 16 + (Q::kRows + wc) * 8 + row_off;
      at_slot = at_slot == (kConvStages - 1) * Q::kStageBytes ? 0 : at_slot + Q::kStageBytes;
      u32x4 w[2][2], x[2][RT];  // a unit's operands, one unit ahead
      auto read = [&](int ks) {
        const int at = (2 * ks + g) ^ swz;
        w[ks & 1][0] = ws[at], w[ks & 1][1] = ws[32 * 8 + at];
#pragma unroll
        for (int v = 0; v < RT; ++v) x[ks & 1][v] = xs[32 * 8 * v + at];
      };
      read(0);
      mfma::static_for<4>([&](auto ks_) {
        constexpr int ks = decltype(ks_)::value;
        if constexpr (ks < 3) read(ks + 1);
        if constexpr (sizeof(T) == 4) __builtin_amdgcn_sched_barrier(0);  // bf16: 84 us so, 79 without
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int v = 0; v < RT; ++v)
            acc[u][v] = turned ? mma_unit(in, w[ks & 1][u], x[ks & 1][v], acc[u][v]) : mma_unit(in, x[ks & 1][v], w[ks & 1][u], acc[u][v]);
        fetch_part(kb + kConvStages - 1, ks_);  // into the stage multiplied one step ago, which every wave is past
      });
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing may still be landing in LDS when the workgroup ends
  };
  if constexpr (sizeof(T) == 2) {
    if (pk) multiply(std::false_type{});
    else multiply(std::true_type{});
  } else {
    multiply(std::true_type{});
  }

  T *out = static_cast<T *>(a.out[z]);
  const float *bias = a.bias[z];
#pragma unroll
  for (int v = 0; v < RT; ++v) {
    const unsigned tile = (unsigned)((m0 + wr) / 32) + v;
    int64_t first;
    int count;
    tile_rows(tile, first, count);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int oc = o0 + wc + 32 * u;
      f32x16 &c = acc[u][v];
      if (!pk) {
        if (bias) {
#pragma unroll
          for (int r = 0; r < 16; ++r) c[r] += bias[oc + mfma::rowmap(r, g)];
        }
        T *row = out + (first + (i < count ? i : 0)) * a.O + oc;
        if constexpr (sizeof(T) == 2) {
          mfma::store_tile_natural(c, reinterpret_cast<uint16_t *>(row), g, i < count);
        } else if (i < count) {
#pragma unroll
          for (int q = 0; q < 4; ++q)
            *reinterpret_cast<float4 *>(row + 8 * q + 4 * g) = float4{c[4 * q], c[4 * q + 1], c[4 * q + 2], c[4 * q + 3]};
        }
        continue;
      }
      const float bv = bias ? bias[oc + i] : 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r) c[r] += bv;
      if (out) {
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (mfma::rowmap(r, g) < count) store_from_f32(out + (first + mfma::rowmap(r, g)) * a.O + oc + i, c[r]);
      }
      if (tpb && (int64_t)tile * 32 < a.M / a.N * tpb * 32) {
        pk[(((int64_t)tile * a.pack_heads + oc / 32) * 2 + 0) * 64 + lane] = mfma::pack_half<0>(c);
        pk[(((int64_t)tile * a.pack_heads + oc / 32) * 2 + 1) * 64 + lane] = mfma::pack_half<1>(c);
      }
    }
  }
}

// whole steps of one tap, whole workgroups of outputs; weights in the reduction's order
template <typename T>
static bool conv_serves(const GemmArgs &a, int nsets) {
  using Q = ConvTile<T, false>;
  if (a.ks <= 0 || a.act != 0 || !a.w_tap_major || a.C % Q::KB != 0 || a.O % Q::kOut != 0 || a.K < 2 * Q::KB) return false;
  for (int z = 0; z < nsets; ++z)
    if (a.out_pack[z] ? sizeof(T) != 2 : !aligned16(a.out[z])) return false;
  return true;
}

template <typename T, bool TALL>
static int conv_launch(const GemmArgs &a, int nsets, hipStream_t st) {
  using Q = ConvTile<T, TALL>;
  const int64_t rows = a.pack_tpb > 0 ? (a.M / a.N) * a.pack_tpb * 32 : a.M;
  const size_t lds = (size_t)Q::kStages * Q::kStageBytes;
  auto kernel = conv_gemm_kernel<T, TALL>;
  if (int rc = allow_dynamic_lds(kernel, lds)) return rc;
  const dim3 grid((unsigned)((rows + Q::kRows - 1) / Q::kRows), (unsigned)(a.O / Q::kOut), (unsigned)nsets);
  hipLaunchKernelGGL(kernel, grid, dim3(Q::kWaves * 64), lds, st, a);
  return launch_status();
}

// float32: one workgroup per CU in either form, so a round of 128-row workgroups takes twice the matrix time of a round of 64-row
// ones, 10 % behind that rate with its two waves per SIMD against 20 % with one: whichever needs less for its whole rounds.
static bool conv_tall(const GemmArgs &a, int nsets, int num_cu) {
  auto rounds = [&](int64_t rows) { return ((a.M + rows - 1) / rows * (a.O / 128) * nsets + num_cu - 1) / num_cu; };
  return 2 * 11 * rounds(128) <= 12 * rounds(64);
}

bool serves(const GemmArgs &a, int nsets, size_t elem_bytes) {
  const int ue = (int)(16 / elem_bytes);
  if (a.K % ue != 0) return false;                      // rows must be whole 16-byte units
  if (a.ks > 0 && a.C % ue != 0) return false;          // a unit must not straddle two taps
  if (!aligned16(a.in)) return false;
  for (int z = 0; z < nsets; ++z)
    if (!aligned16(a.w[z]) || (!a.out[z] && !a.out_pack[z])) return false;
  return true;
}

template <typename T, int NT>
static int launch_t(const GemmArgs &a, int nsets, hipStream_t st) {
  const int64_t rows = a.pack_tpb > 0 ? (a.M / a.N) * a.pack_tpb * 32 : a.M;
  dim3 grid((unsigned)((rows + kRows - 1) / kRows), (unsigned)((a.O + 32 * NT - 1) / (32 * NT)), (unsigned)nsets);
  hipLaunchKernelGGL((rows_gemm_mfma_kernel<T, NT>), grid, dim3(256), 0, st, a);
  return launch_status();
}

template <typename T>
static int launch_n(const GemmArgs &a, int nsets, hipStream_t st) {
  // the widest tile of outputs the shape fills, narrower ones where it leaves CUs without a workgroup (8 rows, 16 -> 2 x 256:
  // 69 us on one 256-wide workgroup per set, 21 us on four 64-wide ones)
  const int64_t rows = a.pack_tpb > 0 ? (a.M / a.N) * a.pack_tpb * 32 : a.M, row_tiles = (rows + kRows - 1) / kRows * nsets;
  auto fills = [&](int nt) { return row_tiles * ((a.O + 32 * nt - 1) / (32 * nt)) >= 256; };
  if (a.O > 128 && fills(8)) return launch_t<T, 8>(a, nsets, st);
  if (a.O > 64 && fills(4)) return launch_t<T, 4>(a, nsets, st);
  return launch_t<T, 2>(a, nsets, st);
}

static int device_cus() {
  int dev = 0, cus = 256;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
    cus = 256;
  return cus;
}

int launch(const GemmArgs &a, int nsets, int dtype, hipStream_t st) {
  if (dtype == PA_BF16 && linear_serves(a, nsets, 2)) return linear_launch(a, nsets, device_cus(), st);
  if (dtype == PA_BF16 && conv_serves<bf16>(a, nsets)) return conv_launch<bf16, false>(a, nsets, st);
  if (dtype == PA_F32 && conv_serves<float>(a, nsets))
    return conv_tall(a, nsets, device_cus()) ? conv_launch<float, true>(a, nsets, st) : conv_launch<float, false>(a, nsets, st);
  return dtype == PA_F32 ? launch_n<float>(a, nsets, st) : launch_n<bf16>(a, nsets, st);
}

}  // namespace gemm
}  // namespace pa
