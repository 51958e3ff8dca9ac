// What the attention kernels share: matrix operand types, the constants of the softmax, the S^T product of a tile and Q
// quantized in the layout its matrix operand wants.
#pragma once

#include "sage_device.h"
#include "sage_kernels.h"

namespace ksana_sage {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int kMagicI = 0x4B400000;       // bits of 12582912.0f = 1.5 * 2^23: fp32 values are 1 apart there
constexpr float kMagicF = 12582912.0f;
// Head size 64 runs on rows whose upper 64 channels are zeros before the Hadamard transform - and a copy of the lower
// 64 after it (H128 [x; 0] = [H64 x; H64 x]): the dot product over 128 channels is twice the one over the lower 64.
// The kernel then multiplies the lower half only and starts its accumulators at 1.5 * 2^24, where fp32 values are 2
// apart: the bits read as fp32 are 25165824 + 2 * dot, the full product, with no instruction spent on the doubling
// (|dot| <= 127 * 127 * 64 < 2^21).
constexpr int kMagicI2 = 0x4BC00000;      // bits of 25165824.0f = 1.5 * 2^24
constexpr float kMagicF2 = 25165824.0f;
// P is scaled by 2^6 before the e4m3 cast, and the reference point of a row (its "running maximum") is moved only when
// a tile's maximum exceeds it by more than kLazyMax octaves: probabilities then reach 2^(6 + 2.7) = 416 < 448, the
// largest e4m3 value, and the accumulators are rescaled in a few per cent of the steps instead of up to half of them
// (rows of flat attention set a new maximum every few tiles, by small amounts).  An e4m3 rounding does not depend on
// the power of two in front, so the result differs only where probabilities fall off the subnormal end, 2^-15 of the
// reference point.
// The piecewise-linear path keeps 2^8 and moves the reference point at every new maximum: its code formula is wrong
// for the subnormal codes (it fades them linearly), which must stay 2^-14 below the true maximum to be harmless.
constexpr float kPShift = 6.0f, kPShiftPwl = 8.0f;
constexpr float kLazyMax = 2.7f, kLazyMaxPwl = 0.0f;

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// The counts of batch entry b in place of the lengths lq, lk the tensors have, where the caller gave any: one wait for both
// scalar loads.  (Left to the compiler they are vector loads, one after the other: two memory latencies before a workgroup
// knows whether it has anything to do.)
__device__ __forceinline__ void take_counts(const int32_t* q_lens, const int32_t* k_lens, int b, int& lq, int& lk) {
  typedef const __attribute__((address_space(4))) int32_t* Constant;
  if (q_lens == nullptr && k_lens == nullptr) return;
  const int nq = *reinterpret_cast<Constant>(reinterpret_cast<uintptr_t>((q_lens != nullptr ? q_lens : k_lens) + b));
  const int nk = *reinterpret_cast<Constant>(reinterpret_cast<uintptr_t>((k_lens != nullptr ? k_lens : q_lens) + b));
  if (q_lens != nullptr) lq = rows_counted(nq, lq);
  if (k_lens != nullptr) lk = rows_counted(nk, lk);
}

// Opaque use+def at this program point: keeps the optimizer from sinking the computation of
// `x` into a later basic block (it emits no instruction).
template <typename T>
__device__ __forceinline__ void pin(T& x) {
  asm volatile("" : "+v"(x));
}

template <int DT>
__device__ __forceinline__ uint2 half4(float a, float b, float c, float d) {
  uint32_t lo, hi;
  if constexpr (DT == KSANA_SAGE_BF16) {
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    b2 x = {(__bf16)a, (__bf16)b}, y = {(__bf16)c, (__bf16)d};
    lo = __builtin_bit_cast(uint32_t, x);
    hi = __builtin_bit_cast(uint32_t, y);
  } else {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    h2 x = {(_Float16)a, (_Float16)b}, y = {(_Float16)c, (_Float16)d};
    lo = __builtin_bit_cast(uint32_t, x);
    hi = __builtin_bit_cast(uint32_t, y);
  }
  return make_uint2(lo, hi);
}
template <int DT>
__device__ __forceinline__ void store4(uint16_t* dst, float a, float b, float c, float d) {
  *reinterpret_cast<uint2*>(dst) = half4<DT>(a, b, c, d);
}

// 16 bytes per lane from global memory straight into LDS at `lds_dst + 16 * lane` (lds_dst is
// wave-uniform).  Written as inline assembly on purpose: the compiler's wait-count model treats
// the builtin form as a possible LDS access through the flat path and from then on waits for
// ALL outstanding LDS reads before every use (lgkmcnt(0)), which serialises the operand
// prefetch.  The copy is tracked by hand instead (vmcnt, see tile_barrier).
// The global address is a wave-uniform base (scalar registers) plus a 32-bit per-lane offset.
// M0 is written and named as clobbered; the compiler remarks that M0 is a register it reserves (it re-materialises
// M0 before each of its own uses and never keeps a value live in it), which is the behaviour relied on here.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void lds_copy16(const void* gbase, unsigned lane_off, const void* lds_dst) {
  const unsigned lds_off = (unsigned)(uintptr_t)(const __attribute__((address_space(3))) void*)lds_dst;
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :
               : "s"(lds_off), "v"(lane_off), "s"(gbase)
               : "memory", "m0");
}
// ... and 4 bytes per lane, to `lds_dst + 4 * lane`
__device__ __forceinline__ void lds_copy4(const void* gbase, unsigned lane_off, const void* lds_dst) {
  const unsigned lds_off = (unsigned)(uintptr_t)(const __attribute__((address_space(3))) void*)lds_dst;
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
               :
               : "s"(lds_off), "v"(lane_off), "s"(gbase)
               : "memory", "m0");
}
#pragma clang diagnostic pop

// Tiles of which a lane's query sees the first n keys only - the one on a wave's diagonal (n depends on the lane) and a
// head's last one where its keys are no multiple of 64: the scores of the others drop below every real score (hh = lane / 32)
// (kHalves: 1 where only the tile's first 32 keys are looked at)
template <int kMagicBits, int kHalves = 2>
__device__ __forceinline__ void blank_scores(v16i (&blk)[2], int hh, int n) {
#pragma unroll
  for (int t = 0; t < kHalves; ++t) {
    // (pinned: what follows is the same in every step, and hoisted out of the key loop it would sit in
    // 32 scalar register pairs for a block that runs once per wave)
    int last = n - 1 - 4 * hh;
    pin(last);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int beyond = (last - (32 * t + 8 * (r >> 2) + (r & 3))) >> 31;  // all-ones where the key is one of those
      blk[t][r] = (blk[t][r] & ~beyond) | ((kMagicBits - (1 << 22)) & beyond);
    }
  }
}
// ... and their probability bytes are cleared outright (code 0 is +0.0 in e4m3), so that a row
// whose scale is zero does not count them either
template <int kHalves = 2>
__device__ __forceinline__ void blank_probs(v8i& pf, int hh, int n) {
  int first = n - 4 * hh;
  pin(first);
#pragma unroll
  for (int w = 0; w < 4 * kHalves; ++w) {
    // bytes of the first min(max(m, 0), 4) keys of this dword stay
    const int m = min(max(first - (32 * (w >> 2) + 8 * (w & 3)), 0), 4);
    const unsigned keep = m >= 4 ? 0xffffffffu : ((1u << (8 * m)) - 1u);
    pf[w] &= (int)keep;
  }
}

// Moves the reference point of a lane's row where this tile's maximum asks for it (imax: the lane's maximum, over half the
// row's keys; sc, mneg: the tile's scale and -magic * scale) and returns 2^(old point - new point), exactly 1 where the point stays.
// A row whose scores are not numbers (an infinity in its q, or in a key) gets the factor NaN, which makes its
// accumulators and sums NaN, and goes on with zero scores: its probabilities must stay numbers, for the 16x16 row sums
// multiply them by another row's zeros.
template <bool kPwlExp = false>
__device__ __forceinline__ float move_point(int imax, float& sc, float& mneg, float& qs, float& m_run, float& x_base, float& x_limit) {
  {
    // the other half of the row's keys lives in lane +- 32
    int other = imax;
    const auto sw = __builtin_amdgcn_permlane32_swap(imax, other, false, false);
    imax = max((int)sw[0], (int)sw[1]);
  }
  // the accumulator read as fp32 is magic + dot, so one fma gives sc * dot (mneg = -magic * sc)
  const float m_tile = __builtin_fmaf(__int_as_float(imax), sc, mneg);
  const bool nan = m_tile != m_tile;
  const float m_new = nan ? 0.0f : (m_tile > x_limit ? m_tile : m_run);  // the limit is -inf at the first tile: always taken
  const float alpha = fast_exp2((nan ? m_tile : m_run) - m_new);
  sc = nan ? 0.0f : sc;
  mneg = nan ? 0.0f : mneg;
  qs = nan ? 0.0f : qs;
  m_run = m_new;
  x_limit = m_new + (kPwlExp ? kLazyMaxPwl : kLazyMax);
  x_base = (kPwlExp ? kPShiftPwl : kPShift) - m_new;
  return alpha;
}

// the probabilities of a tile as the product with V takes them: 2^(sc * dot + xc - magic * sc), the magic folded into xc, in e4m3
template <int kHalves = 2>
__device__ __forceinline__ v8i tile_probs(const v16i (&s)[2], float sc, float xc) {
  v8i pf = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
  for (int w = 0; w < 4 * kHalves; ++w) {
    float e[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) e[i] = fast_exp2(__builtin_fmaf(__int_as_float(s[w >> 2][4 * (w & 3) + i]), sc, xc));
    int code = __builtin_amdgcn_cvt_pk_fp8_f32(e[0], e[1], __float_as_int(e[0]), false);  // both halves get written
    pf[w] = __builtin_amdgcn_cvt_pk_fp8_f32(e[2], e[3], code, true);
  }
  return pf;
}

// S^T tile (64 keys x 32 queries) of one wave: two 32-key sub-tiles, kG 32-channel steps (the channel groups that
// hold data: 4, or 2 for head size 64, whose upper 64 channels are zeros on both sides).
template <int kG>
__device__ __forceinline__ void qk_tile(const uint8_t* k_stage, int lane, const v4i (&qf)[4], const v16i& magic,
                                        v16i (&acc)[2]) {
  acc[0] = magic;
  acc[1] = magic;
#pragma unroll
  for (int s = 0; s < kG; ++s) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const v4i kf = *reinterpret_cast<const v4i*>(k_stage + ((t * 4 + s) * 64 + lane) * 16);
      acc[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(kf, qf[s], acc[t], 0, 0, 0);
    }
  }
}

// Q quantized where it is used.  Lane l of a wave holds the channels 32 s + 16 (l / 32) + 0 .. 15, s < kG, of the wave's row
// l % 32 - those of its matrix operand - so the row's transform is strides 1 .. 8 inside sixteen channels, 16 between lanes
// l and l ^ 32, 32 and 64 between the groups: the order, the roundings and therefore the bits of the separate quantizer
// (fwht128, pack_int8x16).  Head size 64 (kG == 2): the upper half of an extended row repeats the lower, so stride 64 and
// the row's other half change nothing.  Bound by its latency in the set-up (two or three waves' worth of instructions per
// SIMD, all at once); what it saves is the quantizer's pass over Q, which is HBM-bound.  Whole calls, us, before / with it:
// 32760 queries on 512 keys, 40 heads 373 / 336; padded batch (B=3, 24 heads, 3001 x 4099) 210 / 202; causal 8191, 32 heads
// 352 / 345; 9001 tokens of 64 channels, B=2, 16 heads 563 / 557.  Which calls take it: q_in_attention_pays.
// The butterflies between the halves move half of the values across the wave and not back: what crosses back are bytes (8 kG and
// 2 kG swaps a row in place of 16 kG), and one division yields the factor and the scale.  us, before / with it: 32760 queries on
// 512 keys 312.0 / 306.6, 75600 on 512 693.2 / 685.7, 2 x 20000 of 24 heads on 120 157.4 / 156.3; with channels 2 i and 2 i + 1
// as pairs, whose bytes have to be woven afterwards, 309.8, 689.3, 156.3.
template <int DT, int kG>
__device__ __forceinline__ void quant_q_rows(const uint4 (&raw)[8], float premul, v4i (&qf)[4], float& qs) {
  float x[kG][16];
#pragma unroll
  for (int s = 0; s < kG; ++s) {
    widen8<DT>(raw[2 * s], x[s]);
    widen8<DT>(raw[2 * s + 1], x[s] + 8);
#pragma unroll
    for (int st = 1; st < 16; st <<= 1)
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if ((i & st) == 0) {
          const float a = x[s][i], b = x[s][i + st];
          x[s][i] = a + b;
          x[s][i + st] = a - b;
        }
    // two values at a time, channels i and i + 4: the swap gives the lower lanes both ends of the first's butterfly and the
    // upper lanes both ends of the second's, and there the results stay until they are bytes: x[s][i] belongs to the lower
    // sixteen channels, x[s][i + 4] to the upper sixteen
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int i = 2 * j - (j & 3);  // 0 .. 3, 8 .. 11
      const auto ab = __builtin_amdgcn_permlane32_swap(__float_as_uint(x[s][i]), __float_as_uint(x[s][i + 4]), false, false);
      const float a = __uint_as_float(ab[0]), b = __uint_as_float(ab[1]);
      x[s][i] = a + b;
      x[s][i + 4] = a - b;
    }
  }
#pragma unroll
  for (int st = 1; st < kG; st <<= 1)
#pragma unroll
    for (int s = 0; s < kG; ++s)
      if ((s & st) == 0)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const float a = x[s][i], b = x[s + st][i];
          x[s][i] = a + b;
          x[s + st][i] = a - b;
        }
  float amax = 0.0f;
#pragma unroll
  for (int s = 0; s < kG; ++s)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      x[s][i] = x[s][i] * premul;
      amax = fmaxf(amax, fabsf(x[s][i]));
    }
  const auto halves = __builtin_amdgcn_permlane32_swap(__float_as_uint(amax), __float_as_uint(amax), false, false);
  amax = fmaxf(__uint_as_float(halves[0]), __uint_as_float(halves[1]));
  // one division for both quotients (int8_scale): the lower lanes' is the factor, the upper lanes' the scale
  const bool upper = (threadIdx.x & 32) != 0;
  float quot = __fdiv_rn(upper ? amax : 127.0f, upper ? 127.0f : amax);
  quot = amax > 0.0f ? quot : 0.0f;
  const auto both = __builtin_amdgcn_permlane32_swap(__float_as_uint(quot), __float_as_uint(quot), false, false);
  const float inv = __uint_as_float(both[0]);
  qs = __uint_as_float(both[1]);
#pragma unroll
  for (int s = 0; s < kG; ++s) {
    // of the lower sixteen channels codes.x holds 0 .. 3 in the lower lanes and 4 .. 7 in the upper ones, codes.z 8 .. 11 and
    // 12 .. 15; .y and .w the same of the upper sixteen
    const uint4 codes = pack_int8x16(x[s], inv);
    const auto first = __builtin_amdgcn_permlane32_swap(codes.x, codes.y, false, false);
    const auto second = __builtin_amdgcn_permlane32_swap(codes.z, codes.w, false, false);
    qf[s] = v4i{(int)first[0], (int)first[1], (int)second[0], (int)second[1]};
  }
}

}  // namespace ksana_sage
