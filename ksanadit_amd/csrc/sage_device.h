// Steps on the 16 channels a lane holds, shared by the quantizers and by the attention kernels that quantize what they read.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/ksana_sage_hip.h"
#include "sage_kernels.h"

namespace ksana_sage {

// Arguments of a kernel that are wanted at once: one from each of their 64-byte lines, so that the lines come into the
// scalar cache together and not one after the other as the code gets to them.
template <typename A, typename B, typename C, typename D, typename E>
__device__ __forceinline__ void want(A a, B b, C c, D d, E e) {
  asm volatile("" : : "s"(a), "s"(b), "s"(c), "s"(d), "s"(e));
}

template <int DT>
__device__ __forceinline__ void widen8(const uint4& raw, float* out) {
  const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (DT == KSANA_SAGE_BF16) {
      out[2 * i] = __uint_as_float(w[i] << 16);
      out[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    } else {
      typedef _Float16 h2 __attribute__((ext_vector_type(2)));
      h2 p = __builtin_bit_cast(h2, w[i]);
      out[2 * i] = (float)p[0];
      out[2 * i + 1] = (float)p[1];
    }
  }
}

// rne(x * inv) as int8, sixteen at a time, the product exact: one fused multiply-add onto 1.5 * 2^23, where the fp32
// grid is the integers, rounds the exact sum to nearest, ties to even, and leaves the two's-complement int8 in the low
// byte.  No clamp: |x| <= amax and inv = fl(127 / amax) keep |x * inv| below 127.5.  One instruction per value plus
// three byte-gathers per four.
__device__ __forceinline__ uint4 pack_int8x16(const float* x, float inv) {
  uint32_t w[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t z[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) z[j] = __float_as_uint(__fmaf_rn(x[4 * i + j], inv, 12582912.0f));
    const uint32_t lo = __builtin_amdgcn_perm(z[1], z[0], 0x0c0c0400u);  // bytes 0, 1 <- low bytes of z0, z1
    const uint32_t hi = __builtin_amdgcn_perm(z[3], z[2], 0x04000c0cu);  // bytes 2, 3 <- low bytes of z2, z3
    w[i] = lo | hi;
  }
  return make_uint4(w[0], w[1], w[2], w[3]);
}

// The same row as it sits in memory (two 16-byte loads), for code that wants the next row in flight while it works
// on the current one.
__device__ __forceinline__ void fetch_row16(const uint16_t* row_ptr, bool valid, uint4 (&raw)[2]) {
  raw[0] = raw[1] = make_uint4(0, 0, 0, 0);
  if (valid) {
    raw[0] = *reinterpret_cast<const uint4*>(row_ptr);
    raw[1] = *reinterpret_cast<const uint4*>(row_ptr + 8);
  }
}

__device__ __forceinline__ float round_to_half_dtype(float x, int dtype) {
  if (dtype == KSANA_SAGE_BF16) return (float)(__bf16)x;
  return (float)(_Float16)x;
}

// Value of lane (id ^ M) for M = 1, 2, 4, through DPP (the exchange then rides on the consuming
// VALU instruction instead of a round trip through the LDS crossbar).
//   quad_perm [1,0,3,2] = id ^ 1;  quad_perm [2,3,0,1] = id ^ 2;
//   row_half_mirror (id -> 7 - id within 8 lanes) followed by quad_perm [3,2,1,0] (id ^ 3) = id ^ 4.
template <int M>
__device__ __forceinline__ float lane_xor(float v) {
  static_assert(M == 1 || M == 2 || M == 4, "only within groups of 8 lanes");
  const int iv = __float_as_int(v);
  if constexpr (M == 1) return __int_as_float(__builtin_amdgcn_mov_dpp(iv, 0xB1, 0xF, 0xF, true));
  if constexpr (M == 2) return __int_as_float(__builtin_amdgcn_mov_dpp(iv, 0x4E, 0xF, 0xF, true));
  const int t = __builtin_amdgcn_mov_dpp(iv, 0x141, 0xF, 0xF, true);
  return __int_as_float(__builtin_amdgcn_mov_dpp(t, 0x1B, 0xF, 0xF, true));
}

// The factor into int8 and the scale back of a largest absolute value that lanes i and i ^ 1 share: 127 / amax and
// amax / 127, both 0 for 0.  A correctly rounded division is about ten instructions on a wave's every lane, so one is
// done for the two quotients, the first by the even lanes and the second by the odd ones, and they exchange them.
// us, two divisions / one: short calls in one launch, replayed from a graph, 65 tokens of 4 x 24 heads 9.53 / 9.38, 250 of 40 16.50 /
// 16.32; joint block of 2 x 2577 tokens of 24 heads 164.3 / 163.7; dense calls are the same.
struct Int8Scale {
  float inv, scale;
};
__device__ __forceinline__ Int8Scale int8_scale(float amax) {
  const bool odd = (threadIdx.x & 1) != 0;
  float mine = __fdiv_rn(odd ? amax : 127.0f, odd ? 127.0f : amax);
  mine = amax > 0.0f ? mine : 0.0f;
  const float other = lane_xor<1>(mine);
  return odd ? Int8Scale{other, mine} : Int8Scale{mine, other};
}

// Reductions over the lanes of a wave without the LDS crossbar: partners meet through DPP and the lane swaps, whose results the
// next instruction can have, where a shuffle is an LDS round trip - 48 of them stood between a chunk's last row and its sums.  us per
// call, shuffles / this, the rest alike: 40 heads of 1560 tokens 57.4 / 55.4, with V smoothing 75.6 / 73.4, 2 x 16 of 3000 114.2 /
// 112.5, 24 of 4352 172.0 / 171.1, joint block of 2 x 774 tokens of 24 heads 51.5 / 50.8, sparse-linear call of 2 x 40 heads of 29672
// rows 3170 / 3125 (the averages of its blocks), of 40 of 32760 1858 / 1840.
struct Sum {
  static __device__ __forceinline__ float of(float a, float b) { return a + b; }
};
struct Max {
  static __device__ __forceinline__ float of(float a, float b) { return fmaxf(a, b); }
};
// v of this lane and of lane ^ 32
template <typename Op>
__device__ __forceinline__ float over_halves(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return Op::of(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
// v of this lane and of lane ^ 8, ^ 16, ^ 32 in turn: the adjacent-pair tree over a wave's eight row slots
template <typename Op>
__device__ __forceinline__ float over_slots(float v) {
  v = Op::of(v, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x128, 0xF, 0xF, true)));  // row_ror:8
  const auto r16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = Op::of(__uint_as_float(r16[0]), __uint_as_float(r16[1]));
  return over_halves<Op>(v);
}
// The same tree for the sixteen channels of a lane, each result in a quarter of the lanes only: a swap hands over one value
// while it fetches another, so two channels cost one exchange.  Lane: channels 8 (lane / 16 % 2) + 4 (lane / 32) + 0 .. 3.
template <typename Op>
__device__ __forceinline__ float4 over_slots16(const float (&v)[16]) {
  float x[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) x[e] = Op::of(v[e], __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v[e]), 0x128, 0xF, 0xF, true)));
  float y[8], z[4];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x[e]), __float_as_uint(x[e + 8]), false, false);
    y[e] = Op::of(__uint_as_float(r[0]), __uint_as_float(r[1]));
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(y[e]), __float_as_uint(y[e + 4]), false, false);
    z[e] = Op::of(__uint_as_float(r[0]), __uint_as_float(r[1]));
  }
  return make_float4(z[0], z[1], z[2], z[3]);
}
// .. and where it goes: the wave's 128 channels, 16-byte aligned
__device__ __forceinline__ void store_slots16(const float4& v, int lane, float* row) {
  if ((lane & 8) == 0) *reinterpret_cast<float4*>(row + (lane & 7) * 16 + 8 * ((lane >> 4) & 1) + 4 * (lane >> 5)) = v;
}
// all 64 lanes, as a tree over adjacent pairs; every lane gets the result
template <typename Op>
__device__ __forceinline__ float over_lanes(float v) {
  v = Op::of(v, lane_xor<1>(v));
  v = Op::of(v, lane_xor<2>(v));
  v = Op::of(v, lane_xor<4>(v));
  return over_slots<Op>(v);
}

// Number `lane` of the kBatchStarts, by a whole wave; and entry `lane`'s counts (lanes 0 .. B - 1)
__device__ __forceinline__ int batch_number(const BatchNumbers& n, int lane, int& rows, int& keys) {
  const bool zeros = lane >= n.B;
  const int b = min(zeros ? lane - n.B : lane, n.B - 1);
  rows = n.q_lens != nullptr ? rows_counted(n.q_lens[b], n.Lq) : n.Lq;
  keys = n.k_lens != nullptr ? rows_counted(n.k_lens[b], n.Lk) : n.Lk;
  const int with_rows = batch_blocks(rows, keys, n.rows_wg), all = (n.Lq + n.rows_wg - 1) / n.rows_wg;
  const int share = lane < 2 * n.B ? batch_share(n.Hq, zeros ? all - with_rows : with_rows) : 0;
  int rank = 0;  // of this lane's entry
  for (int j = 0; j < n.B; ++j) {
    const int other = __builtin_amdgcn_readlane(keys, j);
    rank += other > keys || (other == keys && j < b) ? 1 : 0;
  }
  const int run = lane < 2 * n.B ? rank + (zeros ? n.B : 0) : lane;
  int start = 0, entries = 0;
  for (int i = 0; i < 2 * n.B; ++i) {
    const int some = __builtin_amdgcn_readlane(share, i), r = __builtin_amdgcn_readlane(run, i);
    start += r < run ? some : 0;
    if (i < n.B) entries |= i << (4 * r);
  }
  return __builtin_amdgcn_ds_permute(4 * run, run == 0 ? entries : (run < 2 * n.B ? start : INT32_MAX));
}

// One butterfly stage across lanes c16 and c16 ^ M: every lane takes `own + sign * other` with sign = -1 on the lane
// that holds the "b" half of a pair.  That lane ought to take `other - own`: it ends up with the negative of its
// value, exactly (a sum and its mirror image round alike).  Both lanes of any LATER stage's pair agree in bit M of
// c16, so they carry the same factor and the later butterfly is the mirror image of the right one as a whole: after
// the three stages a lane holds its transform times (-1)^popcount(c16), which the caller folds into the factor it
// multiplies with next (fwht_lane_sign).  Written this way the stage is one multiply-add per value whose first
// operand arrives through DPP - no separate sign flip, and no register written just ahead of the DPP read.
// The instruction is written out: the compiler keeps the DPP move and the multiply-add apart (two instructions per
// value).  Eight values per statement; `s_nop 1` in front gives the two wait states a DPP read needs after a
// vector-ALU write of the same register, whatever instruction the compiler placed just before; inside a statement
// every register is read at least eight instructions after it was written.
#define KSANA_FMAC_DPP8(CTRL)                                                                                      \
  "v_fmac_f32_dpp %0, %0, %8 " CTRL " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"                                 \
  "v_fmac_f32_dpp %1, %1, %8 " CTRL " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"                                 \
  "v_fmac_f32_dpp %2, %2, %8 " CTRL " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"                                 \
  "v_fmac_f32_dpp %3, %3, %8 " CTRL " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"                                 \
  "v_fmac_f32_dpp %4, %4, %8 " CTRL " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"                                 \
  "v_fmac_f32_dpp %5, %5, %8 " CTRL " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"                                 \
  "v_fmac_f32_dpp %6, %6, %8 " CTRL " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"                                 \
  "v_fmac_f32_dpp %7, %7, %8 " CTRL " row_mask:0xf bank_mask:0xf bound_ctrl:1"
template <int M>
__device__ __forceinline__ void fwht_cross_stage(float* x, int c16) {
  const float sign = (c16 & M) ? -1.0f : 1.0f;
#pragma unroll
  for (int g = 0; g < 2; ++g) {
    float* y = x + 8 * g;
    if constexpr (M == 1) {
      asm volatile("s_nop 1\n\t" KSANA_FMAC_DPP8("quad_perm:[1,0,3,2]")
                   : "+v"(y[0]), "+v"(y[1]), "+v"(y[2]), "+v"(y[3]), "+v"(y[4]), "+v"(y[5]), "+v"(y[6]), "+v"(y[7])
                   : "v"(sign));
    } else if constexpr (M == 2) {
      asm volatile("s_nop 1\n\t" KSANA_FMAC_DPP8("quad_perm:[2,3,0,1]")
                   : "+v"(y[0]), "+v"(y[1]), "+v"(y[2]), "+v"(y[3]), "+v"(y[4]), "+v"(y[5]), "+v"(y[6]), "+v"(y[7])
                   : "v"(sign));
    } else {
      // lane ^ 4 within 8 = row_half_mirror (lane -> 7 - lane) followed by quad_perm [3,2,1,0] (lane ^ 3)
      float t[8];
      asm volatile("s_nop 1\n\t"
                   "v_mov_b32_dpp %8, %0 row_half_mirror row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
                   "v_mov_b32_dpp %9, %1 row_half_mirror row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
                   "v_mov_b32_dpp %10, %2 row_half_mirror row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
                   "v_mov_b32_dpp %11, %3 row_half_mirror row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
                   "v_mov_b32_dpp %12, %4 row_half_mirror row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
                   "v_mov_b32_dpp %13, %5 row_half_mirror row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
                   "v_mov_b32_dpp %14, %6 row_half_mirror row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
                   "v_mov_b32_dpp %15, %7 row_half_mirror row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
                   "v_fmac_f32_dpp %0, %8, %16 quad_perm:[3,2,1,0] row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
                   "v_fmac_f32_dpp %1, %9, %16 quad_perm:[3,2,1,0] row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
                   "v_fmac_f32_dpp %2, %10, %16 quad_perm:[3,2,1,0] row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
                   "v_fmac_f32_dpp %3, %11, %16 quad_perm:[3,2,1,0] row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
                   "v_fmac_f32_dpp %4, %12, %16 quad_perm:[3,2,1,0] row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
                   "v_fmac_f32_dpp %5, %13, %16 quad_perm:[3,2,1,0] row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
                   "v_fmac_f32_dpp %6, %14, %16 quad_perm:[3,2,1,0] row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
                   "v_fmac_f32_dpp %7, %15, %16 quad_perm:[3,2,1,0] row_mask:0xf bank_mask:0xf bound_ctrl:1"
                   : "+v"(y[0]), "+v"(y[1]), "+v"(y[2]), "+v"(y[3]), "+v"(y[4]), "+v"(y[5]), "+v"(y[6]), "+v"(y[7]),
                     "=&v"(t[0]), "=&v"(t[1]), "=&v"(t[2]), "=&v"(t[3]), "=&v"(t[4]), "=&v"(t[5]), "=&v"(t[6]), "=&v"(t[7])
                   : "v"(sign));
    }
  }
}

// The factor fwht128 leaves on the values of lane c16 (see fwht_cross_stage).
__device__ __forceinline__ float fwht_lane_sign(int c16) { return (__popc(c16 & 7) & 1) ? -1.0f : 1.0f; }

// Unnormalised Walsh-Hadamard transform of one 128-channel row held by 8 adjacent lanes x 16
// values (channel = 16*c16 + e), TIMES fwht_lane_sign(c16).  Butterflies (a, b) -> (a + b, a - b) with stride 1, 2,
// 4, 8 inside the lane, then 16, 32, 64 across lanes c16 ^ 1, ^ 2, ^ 4 - in exactly that order.
__device__ __forceinline__ void fwht128(float* x, int c16) {
#pragma unroll
  for (int s = 1; s < 16; s <<= 1) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      if ((i & s) == 0) {
        const float a = x[i], b = x[i + s];
        x[i] = a + b;
        x[i + s] = a - b;
      }
    }
  }
  fwht_cross_stage<1>(x, c16);
  fwht_cross_stage<2>(x, c16);
  fwht_cross_stage<4>(x, c16);
}

}  // namespace ksana_sage
