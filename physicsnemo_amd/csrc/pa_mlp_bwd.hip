// Backward of the block MLP's hidden layer on gfx950 MFMA (bf16 rows of 256 channels).  For y = W2 gelu(W1 u + b1) + b2
//   h  = W1 u + b1 (again: 4 F C operations per row cost less than 4 F bytes written and read back)
//   g  = gelu(h)                       (the input of the second Linear, for d W2)
//   dh = (W2^T dy) * gelu'(h)          (the gradient of the first Linear's output, for d W1, d b1 and d u)
// in one pass over the rows; the forward (mlp_rows2_kernel) leaves nothing of the hidden layer in memory.
#include "pa_host.h"
#include "pa_mfma_ops.h"

namespace pa {
namespace mlp {

using mfma::f32x16;
using mfma::load_4k_to_lds;
using mfma::mma;
using mfma::pack2;
using mfma::rowmap;
using mfma::static_for;
using mfma::u32x2;
using mfma::u32x4;

// Chunk c (32 hidden units) of the weight stream: 32 fragments, k-step ks of W1's rows 32 c .. + 31 (fragment 2 ks) and
// of W2's columns 32 c .. + 31 (fragment 2 ks + 1), both with the reduction index running over the channels
// and, with w1_t, W1^T (C, F)
__global__ __launch_bounds__(256) void hidden_backward_pack_kernel(const uint16_t *__restrict__ w1,
                                                                   const uint16_t *__restrict__ w2,
                                                                   u32x4 *__restrict__ blob, u32x4 *__restrict__ w1_t, int C, int F) {
  const int KS = C / 16;
  const int64_t total = (int64_t)F / 32 * 2 * KS * 64;
  for (int64_t u = (int64_t)blockIdx.x * 256 + threadIdx.x; u < total; u += (int64_t)gridDim.x * 256) {
    // the fastest index runs over hidden units, W2's contiguous axis
    const int lane = (int)(u & 63), i = lane & 31, g = lane >> 5;
    const int64_t f = u >> 6;
    const int ks = (int)(f >> 1) % KS, c = (int)((f >> 1) / KS), row = 32 * c + i, col = 16 * ks + 8 * g;
    if ((f & 1) == 0) {
      blob[u] = *reinterpret_cast<const u32x4 *>(w1 + (int64_t)row * C + col);
    } else {
      u32x4 e;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        e[j] = (uint32_t)w2[(int64_t)(col + 2 * j) * F + row] | ((uint32_t)w2[(int64_t)(col + 2 * j + 1) * F + row] << 16);
      blob[u] = e;
    }
  }
  if (!w1_t) return;
  for (int64_t u = (int64_t)blockIdx.x * 256 + threadIdx.x; u < (int64_t)C * F / 8; u += (int64_t)gridDim.x * 256) {
    const int c = (int)(u % C), f = (int)(u / C);  // eight hidden units from 8 f on
    u32x4 e;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      e[j] = (uint32_t)w1[(int64_t)(8 * f + 2 * j) * C + c] | ((uint32_t)w1[(int64_t)(8 * f + 2 * j + 1) * C + c] << 16);
    w1_t[((int64_t)c * F + 8 * f) / 8] = e;
  }
}

// ---------------------------------------------------------------------------------------------------------------
// hidden_backward_kernel.  Workgroup = 8 waves, two per SIMD; an item is 256 rows and F / splits hidden units, a wave
// owns 32 rows (u and dy as B operands, 128 registers).  Weights stream through LDS in slots of 32 hidden units (32 KB,
// two buffers, one barrier per slot); per slot a wave runs
//   h^T = W1[chunk] u^T + b1 and d^T = W2[:, chunk]^T dy^T     16 + 16 MFMAs, the two accumulators taking turns
//   with the 16 values a lane holds of the chunk before turned into g and dh behind them, two per four MFMAs; two chunks
//   are collected in 8 KB of LDS per wave and leave as whole 128-byte lines.
// Rows past M repeat row M - 1 and write the same values to the same place, so that the number of stores in flight,
// which the wait at a slot's start counts, is the same for every wave.
// splits: the hidden units are independent of each other, so short inputs spread them over the chip.
// Bound by its vector work (330 vector and 32 transcendental instructions per slot of 32 matrix ones) and the stores
// behind it (4 C + 4 F bytes per row): 262 144 rows, F = 1024: 405 us, 415 with the accumulators of one chunk copied over for
// the next instead of two sets taking turns, and 64-bit addresses per store.  Of those 415, GELU in the logistic form, good to
// 2.6e-5, 24 less; with it 309 without the stores, 492 with 64-byte pieces of rows leaving after every slot, 436 with ordinary
// instead of streaming stores.
// ---------------------------------------------------------------------------------------------------------------
template <int C>
__global__ __launch_bounds__(512) void hidden_backward_kernel(const u32x4 *__restrict__ blob, const float *__restrict__ b1,
                                                              const uint16_t *__restrict__ u, const uint16_t *__restrict__ dy,
                                                              uint16_t *__restrict__ act, uint16_t *__restrict__ dh, int64_t M,
                                                              int F, int splits, int64_t items) {
  constexpr int KS = C / 16, SU = 2 * KS * 64, WU = SU / 8;
  static_assert(KS == 16 && WU == 256, "a wave fetches one group of four loads per slot; one value per k-step");
  extern __shared__ u32x4 smem[];
  u32x4 *wbuf = smem;  // 2 * SU
  const int tid = threadIdx.x, lane = tid & 63, i = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform: addresses derived from it stay scalar
  char *stage = reinterpret_cast<char *>(wbuf + 2 * SU) + wave * 8192;  // g: 32 rows of 128 bytes, then dh
  float *b1s = reinterpret_cast<float *>(reinterpret_cast<char *>(wbuf + 2 * SU) + 8 * 8192);
  const int CPS = F / 32 / splits;  // chunks of an item
  for (int k = tid; k < F; k += 512) b1s[k] = b1[k];
  __syncthreads();
  int64_t gs = 0;
  auto fetch = [&](int64_t slot, int c) {
    load_4k_to_lds(blob + (int64_t)c * SU + wave * WU, lane * 16, (unsigned)(uintptr_t)(wbuf + (slot & 1) * SU + wave * WU));
  };
  u32x4 ub[KS], db[KS];
  auto load_rows = [&](int64_t item) {
    int64_t r = item / splits * 256 + wave * 32 + i;
    if (r >= M) r = M - 1;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      ub[ks] = *reinterpret_cast<const u32x4 *>(u + r * C + 8 * g + 16 * ks);
      db[ks] = *reinterpret_cast<const u32x4 *>(dy + r * C + 8 * g + 16 * ks);
    }
  };
  f32x16 h[2], d[2];  // of an even and of an odd chunk
  uint32_t gp[2], dp[2];
  float geven = 0.f, deven = 0.f;
  // value k of an even or odd chunk; the staged row i holds its 16-byte granule j at j ^ i % 8
  auto activate = [&](auto k_, auto odd_) {
    constexpr int k = decltype(k_)::value, q = k >> 2, odd = decltype(odd_)::value;
    const float x = h[odd][k];
    const GeluParts p = gelu_parts(x);
    const float dv = d[odd][k] * gelu_grad(x, p);
    if constexpr (k % 2 == 0) {
      geven = x * p.phi, deven = dv;
    } else {
      gp[(k >> 1) & 1] = pack2(geven, x * p.phi);
      dp[(k >> 1) & 1] = pack2(deven, dv);
    }
    if constexpr (k % 4 == 3) {
      char *at = stage + i * 128 + (((q ^ (i & 7)) << 4) ^ (odd << 6)) + 8 * g;
      *reinterpret_cast<u32x2 *>(at) = u32x2{gp[0], gp[1]};
      *reinterpret_cast<u32x2 *>(at + 4096) = u32x2{dp[0], dp[1]};
    }
  };
  uint32_t row_at[4];  // this lane's pieces of the item's rows, elements from the wave's first row on
  auto store_pair = [&](int64_t row0, int c) {  // chunks c, c + 1; the wave's LDS operations complete in order
    uint16_t *ga = act + row0 * F + 32 * c, *da = dh + row0 * F + 32 * c;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int rw = 8 * t + (lane >> 3);
      const char *at = stage + rw * 128 + (((lane & 7) ^ (rw & 7)) << 4);
      store_streaming(reinterpret_cast<u32x4 *>(ga + row_at[t]), *reinterpret_cast<const u32x4 *>(at));
      store_streaming(reinterpret_cast<u32x4 *>(da + row_at[t]), *reinterpret_cast<const u32x4 *>(at + 4096));
    }
  };
  // Workgroups go round their chunks from different starts: all at the same one would write the same 128 bytes of every
  // 2 F bytes, a few of the memory channels, at the same time.
  const int rot = 2 * (int)(blockIdx.x >> 3) % CPS;
  auto chunk_of = [&](int c0, int c) { return c0 + (c + rot < CPS ? c + rot : c + rot - CPS); };
  if ((int64_t)blockIdx.x < items) {
    fetch(0, chunk_of((int)(blockIdx.x % splits) * CPS, 0));
    load_rows(blockIdx.x);
  }
  for (int64_t item = blockIdx.x; item < items; item += gridDim.x) {
    // a wave whose rows all lie past M works on the last row
    const int64_t row = item / splits * 256 + wave * 32, row0 = row < M ? row : M - 1, next = item + gridDim.x < items ? item + gridDim.x : item;
    const int c0 = (int)(item % splits) * CPS, cn = (int)(next % splits) * CPS;
    const int last = (int)(M - 1 - row0 < 31 ? M - 1 - row0 : 31);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int rw = 8 * t + (lane >> 3);
      row_at[t] = (uint32_t)((rw < last ? rw : last) * F + 8 * (lane & 7));
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) h[1][r] = d[1][r] = 0.f;
    // the rows are here: said to the compiler, which otherwise waits for them (and all that follows them) in every slot
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    auto slot = [&](int c, auto odd_) {
      constexpr int odd = decltype(odd_)::value;
      // slot gs has landed (every wave waits for its own share, then all meet) and the other buffer is free.  Its loads
      // were issued before the eight stores of an even slot, which may still be in flight.
      if (!odd || c == 1) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      else asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
      __syncthreads();
      const int ch = chunk_of(c0, c);
      fetch(gs + 1, c + 1 < CPS ? chunk_of(c0, c + 1) : chunk_of(cn, 0));
      const u32x4 *wb = wbuf + (gs & 1) * SU + lane;
#pragma unroll
      for (int r = 0; r < 16; ++r) h[odd][r] = b1s[32 * ch + rowmap(r, g)], d[odd][r] = 0.f;
      constexpr int RING = 8, AHEAD = 4;
      u32x4 fr[RING];
      static_for<AHEAD>([&](auto q) { fr[decltype(q)::value] = wb[decltype(q)::value * 64]; });
      static_for<KS / 2>([&](auto p_) {
        constexpr int p = decltype(p_)::value;
        static_for<4>([&](auto q) {
          constexpr int f = 4 * p + decltype(q)::value + AHEAD;
          if constexpr (f < 2 * KS) fr[f % RING] = wb[f * 64];
        });
        constexpr std::integral_constant<int, 1 - odd> before{};
        h[odd] = mma(fr[(4 * p) % RING], ub[2 * p], h[odd]);
        d[odd] = mma(fr[(4 * p + 1) % RING], db[2 * p], d[odd]);
        activate(std::integral_constant<int, 2 * p>{}, before);
        h[odd] = mma(fr[(4 * p + 2) % RING], ub[2 * p + 1], h[odd]);
        d[odd] = mma(fr[(4 * p + 3) % RING], db[2 * p + 1], d[odd]);
        activate(std::integral_constant<int, 2 * p + 1>{}, before);
        __builtin_amdgcn_sched_barrier(0);
      });
      ++gs;
    };
    for (int c = 0; c < CPS; c += 2) {
      slot(c, std::integral_constant<int, 0>{});
      if (c > 0) store_pair(row0, chunk_of(c0, c - 2));
      slot(c + 1, std::integral_constant<int, 1>{});
    }
    load_rows(next);
    static_for<16>([&](auto k) { activate(k, std::integral_constant<int, 1>{}); });
    store_pair(row0, chunk_of(c0, CPS - 2));
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing may still be landing in LDS when the workgroup ends
}

static int64_t hidden_backward_lds(int64_t F) { return 2 * 32768 + 8 * 8192 + 4 * F; }

bool hidden_backward_supported(int64_t rows, int64_t C, int64_t F) {
  return rows > 0 && C == 256 && F % 64 == 0 && hidden_backward_lds(F) <= 160 * 1024;
}

constexpr int64_t kItemChunks = 8;

int64_t hidden_backward_blob_bytes(int64_t C, int64_t F) { return 4 * C * F; }

int hidden_backward(int64_t rows, int64_t C, int64_t F, const void *w1, const float *b1, const void *w2, const void *u,
                    const void *dy, void *act, void *dh, void *blob, void *w1_t, int cus, hipStream_t st) {
  hidden_backward_pack_kernel<<<(unsigned)(C * F / 4 / 256 < 1024 ? C * F / 4 / 256 : 1024), 256, 0, st>>>(
      static_cast<const uint16_t *>(w1), static_cast<const uint16_t *>(w2), static_cast<u32x4 *>(blob), static_cast<u32x4 *>(w1_t), (int)C,
      (int)F);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return (int)e;
  const int64_t blocks = (rows + 255) / 256, chunks = F / 32;
  // The split with the shortest way for the busiest CU, its items' chunks and, for each item, the row loads and last stores that
  // nothing covers: 10 us, three chunks of a full chip; taken as eight, because chunks go faster where CUs are left idle (the
  // stores bound them).  Against two items per CU wherever the rows do not give them: 14 450 rows 50 -> 40 us, 24 200 72 -> 55,
  // 32 768 74 -> 65, 60 000 128 -> 99, 100 000 197 -> 177, 2 500 and 8 000 the same; taken as three, 40 000 rows 98 against 87.
  int splits = 1;
  auto way = [&](int64_t n) { return (blocks * n + cus - 1) / cus * (chunks / n + kItemChunks); };
  for (int n = 2; chunks % (2 * n) == 0 && chunks / n >= 4; n *= 2)
    if (way(n) < way(splits)) splits = n;
  const int64_t items = blocks * splits;
  const int lds = (int)hidden_backward_lds(F);
  e = hipFuncSetAttribute(reinterpret_cast<const void *>(hidden_backward_kernel<256>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e != hipSuccess) return (int)e;
  hidden_backward_kernel<256><<<(unsigned)(items < cus ? items : cus), 512, lds, st>>>(
      static_cast<const u32x4 *>(blob), b1, static_cast<const uint16_t *>(u), static_cast<const uint16_t *>(dy),
      static_cast<uint16_t *>(act), static_cast<uint16_t *>(dh), rows, (int)F, splits, items);
  e = hipGetLastError();
  return e == hipSuccess ? PA_OK : (int)e;
}

}  // namespace mlp
}  // namespace pa
