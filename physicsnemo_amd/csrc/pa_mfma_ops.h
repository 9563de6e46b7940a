// MFMA operand types and small helpers shared by the bf16 kernels (v_mfma_f32_32x32x16_bf16, gfx950).
//
// Register layouts (lane = 32*g + i, i = lane % 32, g = lane / 32):
//   A operand (32 x 16): lane holds row i, k = 8g + j, j = 0..7.      B operand (16 x 32): column i, k = 8g + j.
//   C/D (32 x 32): lane holds column i; register r = 0..15 is row  rowmap(r, g) = 8*(r/4) + 4*g + r%4.
// A C/D tile converted to bf16 is directly a pair of A (or B) operands of a following MFMA whose reduction index is
// the C/D row index taken in the order kperm(kk, g, j), provided the other operand uses the same permutation.
#pragma once

#include "pa_common.h"

#include <type_traits>
#include <utility>

namespace pa {
namespace mfma {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ f32x16 mma(u32x4 a, u32x4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

__device__ __forceinline__ int rowmap(int r, int g) { return 8 * (r >> 2) + 4 * g + (r & 3); }
__device__ __forceinline__ int kperm(int kk, int g, int j) { return 16 * kk + 8 * (j >> 2) + 4 * g + (j & 3); }

// registers 8*HALF .. 8*HALF+7 of an accumulator, scaled, as 8 bf16 (round to nearest even)
template <int HALF>
__device__ __forceinline__ u32x4 pack_half(const f32x16 &v, float scale = 1.f) {
  bf16x8 o;
#pragma unroll
  for (int j = 0; j < 8; ++j) o[j] = (__bf16)(v[8 * HALF + j] * scale);
  return __builtin_bit_cast(u32x4, o);
}

// the same for what pack_half leaves over: v - bf16(v)
template <int HALF>
__device__ __forceinline__ u32x4 pack_half_rest(const f32x16 &v) {
  bf16x8 o;
#pragma unroll
  for (int j = 0; j < 8; ++j) o[j] = (__bf16)(v[8 * HALF + j] - (float)(__bf16)v[8 * HALF + j]);
  return __builtin_bit_cast(u32x4, o);
}

__device__ __forceinline__ uint16_t to_bf16_bits(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }

// 2 floats -> 2 bf16 (round to nearest even), the first in the low half
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  bf16x2 o;
  o[0] = (__bf16)a;
  o[1] = (__bf16)b;
  return __builtin_bit_cast(uint32_t, o);
}

// Operand fragment of 16 slices from float32 rows of 32 channels, `src` at the lane's channel of the first one: element j is
// slice rowmap(j, g), as bf16 and as the bf16 remainder of that rounding.
__device__ __forceinline__ void token_fragment(const float *src, int g, u32x4 &hi, u32x4 &lo) {
  bf16x8 h, l;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float v = src[((j & 3) + 8 * (j >> 2) + 4 * g) * 32];
    h[j] = (__bf16)v;
    l[j] = (__bf16)(v - (float)h[j]);
  }
  hi = __builtin_bit_cast(u32x4, h);
  lo = __builtin_bit_cast(u32x4, l);
}

// Four direct global -> LDS loads of 64 x 16 bytes each (no registers): the wave's lanes read sbase + 1024 q + 16 lane
// (q = 0..3) and the data land at LDS byte address lds + 1024 q + 16 lane; the instruction offset advances the
// global and the LDS address alike.  sbase and lds are wave-uniform.  The loads are asynchronous and counted by
// vmcnt; their data must not be read before a wait and a barrier.
__device__ __forceinline__ void load_4k_to_lds(const void *sbase, unsigned lane16, unsigned lds) {
  asm volatile(
      "s_mov_b32 m0, %2\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, %0\n\t"
      "global_load_lds_dwordx4 %1, %0 offset:1024\n\t"
      "global_load_lds_dwordx4 %1, %0 offset:2048\n\t"
      "global_load_lds_dwordx4 %1, %0 offset:3072" ::"s"(sbase),
      "v"(lane16), "s"(lds)
      : "memory");
}

// what such a load reads where a convolution's neighbour lies outside the grid; a vector type, so on a 16-byte boundary
__device__ const u32x4 kZeroUnit = {0u, 0u, 0u, 0u};
static_assert(alignof(u32x4) == 16, "one 16-byte load");

// One such load with a 16-byte address per lane: lane l's unit lands at dst + 16 l.
__device__ __forceinline__ void load_unit_to_lds(const void *p, unsigned dst) {  // lane l's 16 bytes land at dst + 16 l
  asm volatile(
      "s_mov_b32 m0, %1\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %0, off" ::"v"(p), "s"(dst)
      : "memory");
}

// The same with a wave-uniform base and a byte offset per lane.
__device__ __forceinline__ void load_unit_to_lds(const void *sbase, int off, unsigned dst) {
  asm volatile(
      "s_mov_b32 m0, %2\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, %0" ::"s"(sbase), "v"(off), "s"(dst)
      : "memory");
}

// f(integral_constant<int, 0>{}), ..., f(integral_constant<int, N - 1>{}): a loop whose index is a constant expression
template <class F, int... I>
__device__ __forceinline__ void static_for_impl(F &&f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F &&f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// value of lane l combined with the value of lane l ^ 32, without a trip through LDS: v_permlane32_swap hands every
// lane the lower-half and the upper-half value of its column
__device__ __forceinline__ float half_max(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float half_sum(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// sum over the 32 lanes of this lane's half of the wave, returned in every lane of the half: DPP steps inside each
// row of 16 lanes, then v_permlane16_swap pairs the two rows of the half
__device__ __forceinline__ float half_wave_sum(float v) {
  auto step = [](float x, auto ctrl) {
    constexpr int c = decltype(ctrl)::value;
    return x + __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(x), c, 0xf, 0xf, true));
  };
  v = step(v, std::integral_constant<int, 0xB1>{});   // quad_perm [1,0,3,2]
  v = step(v, std::integral_constant<int, 0x4E>{});   // quad_perm [2,3,0,1]
  v = step(v, std::integral_constant<int, 0x141>{});  // row_half_mirror
  v = step(v, std::integral_constant<int, 0x140>{});  // row_mirror
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// A 32 x 32 accumulator tile (lane (i, g) <-> point i, register r <-> channel rowmap(r, g)) to bf16 rows in natural
// layout: `row` points at channel 0 of this lane's point.  Registers 4q..4q+3 hold channels 8q + 4g .. + 3; swapping
// halves with lane ^ 32 gives each lane 8 consecutive channels (g = 0: 0-7 and 8-15, g = 1: 16-23 and 24-31), so a
// point's 64 bytes leave as four 16-byte stores.  `nch` = valid channels (32, or 16: the lower half only).
__device__ __forceinline__ void tile_natural(const f32x16 &v, u32x4 &s0, u32x4 &s1) {
  uint32_t p[4][2];
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int w = 0; w < 2; ++w)
      p[q][w] = pack2(v[4 * q + 2 * w], v[4 * q + 2 * w + 1]);
#pragma unroll
  for (int w = 0; w < 2; ++w) {
    // lower half-wave: (own piece 0, partner's piece 0); upper half-wave: (partner's piece 2, own piece 2)
    const auto a = __builtin_amdgcn_permlane32_swap(p[0][w], p[2][w], false, false);
    s0[w] = a[0];
    s0[2 + w] = a[1];
    const auto b = __builtin_amdgcn_permlane32_swap(p[1][w], p[3][w], false, false);
    s1[w] = b[0];
    s1[2 + w] = b[1];
  }
}
__device__ __forceinline__ void store_tile_natural(const f32x16 &v, uint16_t *row, int g, bool ok, int nch = 32) {
  u32x4 s0, s1;
  tile_natural(v, s0, s1);
  if (ok && (g == 0 || nch > 16)) {
    *reinterpret_cast<u32x4 *>(row + 16 * g) = s0;
    *reinterpret_cast<u32x4 *>(row + 16 * g + 8) = s1;
  }
}

// ------------------------------------------------------------------------------------------------
// The slice weights of one head for one tile of 32 points, formed in registers: logits, temperature softmax, bf16
// operand chunks.  chunk[cq] (cq = 0 .. S/16 - 1) is what the slice-softmax kernels store: as an A operand its rows
// are the points and its reduction index the slices 16 cq + kperm order; the same registers serve as a B operand
// whose columns are the points.  The kernels that use this recompute the weights from x_mid instead of passing them through
// memory (S/16 KB per point and head group written once and read twice otherwise).  The token sums use
// bf16(e_s / sum e), the hand-back bf16(e_s) divided by the sum of those rounded values: the same softmax, each rounded
// once.
// ------------------------------------------------------------------------------------------------
// DEFER: the chunks hold bf16(exp2(..)) without the division by their sum; the caller divides what it forms from them
// by the sum of the same rounded values (one more MFMA column), which saves a pass over the S values per point.
// PARTS: sets of fragments in wsl, W_slice as that many bf16 values (three hold a float32 value to the last bit).
template <int S, bool DEFER = false, int PARTS = 1>
__device__ __forceinline__ void slice_weights_of_tile(const u32x4 *__restrict__ wsl, const float *__restrict__ bsl,
                                                      u32x4 xm0, u32x4 xm1, float sc, bool valid, int lane, int g,
                                                      u32x4 (&chunk)[S / 16]) {
  constexpr int ST = (S + 31) / 32, NCH = S / 16;
  f32x16 lg[ST];
#pragma unroll
  for (int st = 0; st < ST; ++st) {
#pragma unroll
    for (int r = 0; r < 16; ++r) lg[st][r] = bsl[32 * st + rowmap(r, g)];
#pragma unroll
    for (int p = 0; p < PARTS; ++p) {
      lg[st] = mma(wsl[((p * ST + st) * 2 + 0) * 64 + lane], xm0, lg[st]);
      lg[st] = mma(wsl[((p * ST + st) * 2 + 1) * 64 + lane], xm1, lg[st]);
    }
  }
  float mx = -INFINITY;
#pragma unroll
  for (int st = 0; st < ST; ++st)
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, lg[st][r]);
  mx = half_max(mx);
  const float off = mx * sc;
  if constexpr (DEFER) {
#pragma unroll
    for (int st = 0; st < ST; ++st)
#pragma unroll
      for (int r = 0; r < 16; ++r) lg[st][r] = __builtin_amdgcn_exp2f(fmaf(lg[st][r], sc, -off));
#pragma unroll
    for (int cq = 0; cq < NCH; ++cq) chunk[cq] = (cq & 1) ? pack_half<1>(lg[cq >> 1]) : pack_half<0>(lg[cq >> 1]);
  } else {
    float sum = 0.f;
#pragma unroll
    for (int st = 0; st < ST; ++st)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float e = __builtin_amdgcn_exp2f(fmaf(lg[st][r], sc, -off));
        lg[st][r] = e;
        sum += e;
      }
    sum = half_sum(sum);
    const float inv = valid ? __builtin_amdgcn_rcpf(sum) : 0.f;
#pragma unroll
    for (int cq = 0; cq < NCH; ++cq) chunk[cq] = (cq & 1) ? pack_half<1>(lg[cq >> 1], inv) : pack_half<0>(lg[cq >> 1], inv);
  }
}

// W_slice as A operands and the slice bias in LDS, as slice_weights_of_tile reads them; the reduction index runs over
// d in natural order (x_mid read from its rows) or in kperm order (PACKED_X: x_mid read as packed operand tiles);
// PARTS: followed by the fragments of what the rounding to bf16 left over, and of what that one's left
template <int S, bool PACKED_X, int PARTS = 1>
__device__ __forceinline__ void stage_slice_projection(const float *__restrict__ w_slice, const float *__restrict__ b_slice,
                                                       u32x4 *wsl, float *bsl) {
  constexpr int ST = (S + 31) / 32;
  for (int u = threadIdx.x; u < ST * 2 * 64; u += blockDim.x) {
    const int ul = u & 63, ui = ul & 31, ug = ul >> 5, f = u >> 6, st = f >> 1, kk = f & 1;
    const int s = 32 * st + ui;
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = s < S ? w_slice[s * 32 + (PACKED_X ? kperm(kk, ug, j) : 16 * kk + 8 * ug + j)] : 0.f;
#pragma unroll
    for (int p = 0; p < PARTS; ++p) {
      bf16x8 e;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        e[j] = (__bf16)v[j];
        v[j] = isinf((float)e[j]) ? 0.f : v[j] - (float)e[j];  // nothing is left of an infinity
      }
      wsl[p * ST * 2 * 64 + u] = __builtin_bit_cast(u32x4, e);
    }
  }
  for (int s = threadIdx.x; s < ST * 32; s += blockDim.x) bsl[s] = s < S ? b_slice[s] : -1e30f;  // slices beyond S: weight 0
}

// ------------------------------------------------------------------------------------------------
// Operand fragments of the per-point backward kernels (16-byte units, one per lane; lane = 32g + i; j = 0..7):
//   shared   wsl[(st*2 + kk)]   = W_slice[32st + i][16kk + 8g + j]                 A of the logits (k = d, natural order)
//            wsT[cq]            = W_slice[16cq + rowmap(j, g)][i]                   A of d x_mid (k = slices, chained order)
//            (Transolver++: the same two groups for the first Linear of proj_temperature)
//   per (b,h) tokA[(st*2 + kk)] = tok'[32st + i][16kk + 8g + j]                    A of d w, first half of k
//            dnA[(st*2 + kk)]   = d num[32st + i][16kk + 8g + j]                   A of d w, second half of k
//            dnT[cq]            = d num[16cq + rowmap(j, g)][i]                     A of d fx_mid
// Slices >= S read as zero.  SPLIT tables carry the remainders t - bf16(t) in a second set of fragments behind each group,
// so that products with them keep 16 bits of the table (float_tables() says for which layers).
// ------------------------------------------------------------------------------------------------
struct BwdTablePlan {
  int st2, nch, group, nshared, nhead;  // fragments: of the two kinds, of a shared group, shared, per (b, h)
  int64_t shared_units, per_head_units;
};
__host__ __device__ inline BwdTablePlan bwd_table_plan(int S, bool plus, bool split) {
  BwdTablePlan p;
  p.st2 = 2 * ((S + 31) / 32);
  p.nch = S / 16;
  p.group = (p.st2 + p.nch) * (split ? 2 : 1);
  p.nshared = p.group * (plus ? 2 : 1);
  p.nhead = (2 * p.st2 + p.nch) * (split ? 2 : 1);
  p.shared_units = (int64_t)p.nshared * 64;
  p.per_head_units = (int64_t)p.nhead * 64;
  return p;
}

// floats of a workgroup's row of partial gradients: d W_slice, d b_slice, d T (Transolver++: and d W1, d b1, d w2, d b2)
__host__ __device__ inline int point_grads(int S, int H, bool plus) { return S * 33 + H + (plus ? S * 34 + 1 : 0); }

}  // namespace mfma
}  // namespace pa
