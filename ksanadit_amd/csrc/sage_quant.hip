// HBM-bound quantizer kernels for gfx950 (MI355X).
//
// Every kernel works on 128-channel rows of a [B, L, H, D] half tensor with the same thread
// mapping: 256 threads = 32 row slots x 8 lanes, each lane owning 16 consecutive channels
// (two 16-byte loads), so a wave reads four full 256-byte rows per load pair.
//
// The arithmetic is fixed to the last bit (it is compared bit-exactly with a PyTorch
// specification): plain IEEE fp32 add / sub / mul / div, round-half-even, no contraction.
#include "sage_device.h"
#include "sage_kernels.h"
#include "sage_sla_device.h"

#include <cstdlib>
#include <cstring>
#include <mutex>
#include <type_traits>

#include "../../include/ksana_sage_hip.h"

namespace ksana_sage {
namespace {

constexpr int kThreads = 256;
constexpr int kSlots = 32;  // row slots per workgroup

// 16 channels of one row; rows at or beyond L read as zero.
template <int DT>
__device__ __forceinline__ void load_row16(const uint16_t* row_ptr, bool valid, float* out) {
  uint4 a = make_uint4(0, 0, 0, 0), b = make_uint4(0, 0, 0, 0);
  if (valid) {
    a = *reinterpret_cast<const uint4*>(row_ptr);
    b = *reinterpret_cast<const uint4*>(row_ptr + 8);
  }
  widen8<DT>(a, out);
  widen8<DT>(b, out + 8);
}

// 16 bytes of quantizer output.  Non-temporal: the tiles are written once and read next by another kernel, after
// half a gigabyte of other traffic; stores that do not linger in the caches on their way out measured 6 % off the
// three quantizers together (405 -> 380 us at B=1 H=40 L=32760), with the attention kernel's time unchanged.
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void store_out16(void* p, uint4 v) {
  const u32x4 w = {v.x, v.y, v.z, v.w};
  __builtin_nontemporal_store(w, reinterpret_cast<u32x4*>(p));
}

// ---------------------------------------------------------------------------------------
// The step before attention, on the 16 channels [16*c16, 16*c16+16) of head h, token `row`:
//   y = half( (x * inv_rms[row]) * weight[ch] )                         RMSNorm, fp32, in this order
//   (y[2i], y[2i+1]) -> half( float( (y[2i] + i*y[2i+1]) * freqs[p, i] ) )   rotation in fp64
// with p the token's frame / row / column index for pair i in [0,22) / [22,43) / [43,64).
// Each result is rounded to the tensor's half type exactly where a separate norm kernel and a
// separate rotation kernel would have stored it (the fp64 product first to fp32, as a
// conversion from double goes), so the quantizer sees the same bits.
// Tokens at or beyond frames*height*width are normed but not rotated.
// ---------------------------------------------------------------------------------------
template <int DT>
__device__ __forceinline__ float through_half(float x) {
  // The fp32 value has to exist before it is narrowed: left alone, the compiler merges the
  // multiply that produced it with the conversion (v_fma_mixlo_f16), which rounds once
  // instead of twice and so differs from "compute in fp32, then store as half" in rare ties.
  asm volatile("" : "+v"(x));
  if constexpr (DT == KSANA_SAGE_BF16) return (float)(__bf16)x;
  return (float)(_Float16)x;
}

// Two values at a time: one packed conversion instead of two (bf16), the same roundings.
template <int DT>
__device__ __forceinline__ void through_half2(float& a, float& b) {
  asm volatile("" : "+v"(a), "+v"(b));  // as in through_half: the fp32 values exist before they are narrowed
  if constexpr (DT == KSANA_SAGE_BF16) {
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    const b2 p = {(__bf16)a, (__bf16)b};
    const uint32_t w = __builtin_bit_cast(uint32_t, p);
    a = __uint_as_float(w << 16);
    b = __uint_as_float(w & 0xffff0000u);
  } else {
    a = (float)(_Float16)a;
    b = (float)(_Float16)b;
  }
}

// Rotation factors for the rows of one workgroup, copied to LDS once.  The model's table is
// [position on an axis][64 pairs] of complex128; a lane needs 8 of them (128 bytes) per row, four
// times its payload, and fetched straight from the table those reads are 16 bytes out of 30-odd
// different cache lines per load instruction - the L1 tag rate, not HBM, then sets the pace.  The
// table is separable, so what a run of consecutive rows needs is small: the frames it touches
// (22 pairs each), the image rows it touches (21 pairs each) and every column (21 pairs each).
struct RopeLds {
  const double2* frame;   // [frames touched][22], first = frame f0
  const double2* height;  // [image rows touched][21], first = image row gr0 (counted across frames)
  const double2* width;   // [grid width][21]
  int f0, gr0;
};

constexpr int kRopeN0 = kRopeSplit0, kRopeN1 = kRopeSplit1 - kRopeSplit0, kRopeN2 = kD / 2 - kRopeSplit1;

// All threads of the workgroup call this; rows [row0, row0 + nrows) of batch entry b are the
// ones the workgroup will rotate.  Ends with a barrier.
__device__ __forceinline__ RopeLds stage_rope(const PrepParams& pp, int b, int row0, int nrows, double2* lds) {
  RopeLds rl;
  rl.frame = lds;
  rl.height = lds + pp.lds_frames * kRopeN0;
  rl.width = rl.height + pp.lds_heights * kRopeN1;
  const int gh = pp.grid[b][1], gw = pp.grid[b][2], plane = gh * gw;
  const int r1 = min(row0 + nrows, pp.grid[b][0] * plane);  // exclusive; rows from here on are not rotated
  rl.f0 = row0 / plane;
  rl.gr0 = row0 / gw;
  if (row0 < r1) {
    const double2* tab = reinterpret_cast<const double2*>(pp.freqs);
    const int nf = (r1 - 1) / plane - rl.f0 + 1, nh = (r1 - 1) / gw - rl.gr0 + 1;
    const int t = threadIdx.x, nt = blockDim.x;
    for (int idx = t; idx < nf * kRopeN0; idx += nt) {
      const int r = idx / kRopeN0, i = idx - r * kRopeN0;
      lds[idx] = tab[(int64_t)(rl.f0 + r) * (kD / 2) + i];
    }
    double2* hdst = lds + pp.lds_frames * kRopeN0;
    for (int idx = t; idx < nh * kRopeN1; idx += nt) {
      const int r = idx / kRopeN1, i = idx - r * kRopeN1;
      hdst[idx] = tab[(int64_t)((rl.gr0 + r) % gh) * (kD / 2) + kRopeSplit0 + i];
    }
    double2* wdst = hdst + pp.lds_heights * kRopeN1;
    for (int idx = t; idx < gw * kRopeN2; idx += nt) {
      const int r = idx / kRopeN2, i = idx - r * kRopeN2;
      wdst[idx] = tab[(int64_t)r * (kD / 2) + kRopeSplit1 + i];
    }
  }
  __syncthreads();
  return rl;
}

// n / d for 0 <= n < 2^24, 1 <= d: the fp32 quotient is off by at most one, fixed by the remainder test
__device__ __forceinline__ int small_div(int n, int d, int* rem) {
  int q = (int)(__int2float_rn(n) * __frcp_rn(__int2float_rn(d)));
  int r = n - q * d;
  if (r < 0) {
    --q;
    r += d;
  } else if (r >= d) {
    ++q;
    r -= d;
  }
  *rem = r;
  return q;
}


// The Qwen-Image block's step before attention on the 16 channels [16*c16, 16*c16+16) of one head of token `row`
// (the 8 lanes c16 = 0..7 of the row are adjacent):
//   y = half( (x * r) * weight[ch] ),  r = 1 / sqrt(mean_{128 channels}(x^2) + eps)
//       mean: every lane adds its 16 squares in channel order, the 8 lane sums meet in an adjacent-pair tree
//   (y[2i], y[2i+1]) -> half( (y[2i] + i*y[2i+1]) * freqs[row, i] )    complex64: four products, one subtraction and
//       one addition, each rounded to fp32
//
// What a row's lane reads besides the row, the same for all heads: where its 16 norm weights are, and 8 rotation factors.
struct QwenRow {
  const float4* w;  // nullptr: no norm
  bool rotate;
  float4 cs[4];  // two factors each, (re, im), (re, im)
};
__device__ __forceinline__ void qwen_row(QwenRow& f, const PrepParams& pp, int row, int c16) {
  const bool txt = row < pp.txt_len;
  const float* w = txt ? pp.weight_txt : pp.weight_img;
  const float2* tab = txt ? pp.freqs_txt : pp.freqs_img;
  f.w = w != nullptr ? reinterpret_cast<const float4*>(w + c16 * 16) : nullptr;
  f.rotate = tab != nullptr;
  if (f.rotate) {
    const float4* t4 = reinterpret_cast<const float4*>(tab + (int64_t)(txt ? row : row - pp.txt_len) * (kD / 2) + c16 * 8);
#pragma unroll
    for (int j = 0; j < 4; ++j) f.cs[j] = t4[j];
  }
}
// kFused: the squares of half values are exact (bf16: from 2^-63 up), so a fused multiply-add rounds like the sum alone and is an
// instruction less.  us, apart / fused: several heads per item, whose vector units are busy over half of the time, 2 x 4352 tokens of
// 24 heads 345.7 / 344.3, 2 x 1328 73.1 / 72.2; one head per item, bound by the length of its chain, the other way round: 2 x 774
// 49.4 / 50.3, 2 x 1024 53.2 / 54.1, 1756 61.8 / 62.5.  K's only chunk (at most 256 tokens) takes it fused: 256 of 24 heads 27.8 / 27.6,
// two of them 28.8 / 28.5.
template <int DT, bool kFused>
__device__ __forceinline__ void prep16_qwen(float* x, const QwenRow& f, float eps) {
  if (f.w != nullptr) {
    float ss = 0.0f;
#pragma unroll
    for (int e = 0; e < 16; ++e) ss = kFused ? __fmaf_rn(x[e], x[e], ss) : (e == 0 ? x[0] * x[0] : ss + x[e] * x[e]);
    ss = ss + lane_xor<1>(ss);
    ss = ss + lane_xor<2>(ss);
    ss = ss + lane_xor<4>(ss);
    const float r = __fdiv_rn(1.0f, sqrtf(__fdiv_rn(ss, (float)kD) + eps));
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float4 wj = f.w[j];
      x[4 * j + 0] = (x[4 * j + 0] * r) * wj.x;
      x[4 * j + 1] = (x[4 * j + 1] * r) * wj.y;
      x[4 * j + 2] = (x[4 * j + 2] * r) * wj.z;
      x[4 * j + 3] = (x[4 * j + 3] * r) * wj.w;
      through_half2<DT>(x[4 * j + 0], x[4 * j + 1]);
      through_half2<DT>(x[4 * j + 2], x[4 * j + 3]);
    }
  }
  if (f.rotate) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float4 cs = f.cs[j];
      const float a0 = x[4 * j], b0 = x[4 * j + 1], a1 = x[4 * j + 2], b1 = x[4 * j + 3];
      x[4 * j + 0] = a0 * cs.x - b0 * cs.y;
      x[4 * j + 1] = a0 * cs.y + b0 * cs.x;
      x[4 * j + 2] = a1 * cs.z - b1 * cs.w;
      x[4 * j + 3] = a1 * cs.w + b1 * cs.z;
      through_half2<DT>(x[4 * j + 0], x[4 * j + 1]);
      through_half2<DT>(x[4 * j + 2], x[4 * j + 3]);
    }
  }
}

template <int DT, bool kFused>
__device__ __forceinline__ void prep16_qwen(float* x, const PrepParams& pp, int row, int c16) {
  QwenRow f;
  qwen_row(f, pp, row, c16);
  prep16_qwen<DT, kFused>(x, f, pp.eps);
}

// The pieces of the Wan step on the 16 channels of a lane.
//   norm16:   y = half( (x * r) * weight[ch] ), r the row's 1 / sqrt(mean(x^2) + eps)
template <int DT>
__device__ __forceinline__ void norm16(float* x, float r, const float* w16) {
  const float4* w4 = reinterpret_cast<const float4*>(w16);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float4 w = w4[j];
    x[4 * j + 0] = (x[4 * j + 0] * r) * w.x;
    x[4 * j + 1] = (x[4 * j + 1] * r) * w.y;
    x[4 * j + 2] = (x[4 * j + 2] * r) * w.z;
    x[4 * j + 3] = (x[4 * j + 3] * r) * w.w;
    through_half2<DT>(x[4 * j + 0], x[4 * j + 1]);
    through_half2<DT>(x[4 * j + 2], x[4 * j + 3]);
  }
}
//   rotate_pair: (a, b) -> half( float( (a + i b) * (c + i s) ) ) in fp64, unfused
template <int DT>
__device__ __forceinline__ void rotate_pair(float& xa, float& xb, const double2 cs) {
  const double a = (double)xa, bb = (double)xb;
  const double re = a * cs.x - bb * cs.y;
  const double im = a * cs.y + bb * cs.x;
  xa = (float)re;
  xb = (float)im;
  through_half2<DT>(xa, xb);
}
//   comfy_pair: apply_comfyui_rope (utils/rope.py:180-212): out[2i+e] = m[e][0] * x[2i] + m[e][1] * x[2i+1] in fp32, the
//   first product rounded on its own, the second fused into the sum (what torch's mul followed by addcmul_ computes)
template <int DT>
__device__ __forceinline__ void comfy_pair(float& xa, float& xb, const float4 m) {
  const float a = xa, bb = xb;
  xa = __fmaf_rn(m.y, bb, __fmul_rn(m.x, a));
  xb = __fmaf_rn(m.w, bb, __fmul_rn(m.z, a));
  through_half2<DT>(xa, xb);
}

// Where the 8 rotation factors of lane c16 (pairs 8 * c16 + j) sit for a token at (frame f, image row hi, column wi):
// two of the table's three segments at most, the second from pair `split` on.  first / second are element indices of
// pair 8 * c16 + 0 as if the whole lane lay in that segment (the table is [position][64 pairs]).
struct RopeLaneIndex {
  int first, second, split;
};
__device__ __forceinline__ RopeLaneIndex rope_lane_index(int c16, int base_f, int base_h, int base_w) {
  const int i0 = c16 * 8, i7 = c16 * 8 + 7;
  RopeLaneIndex r;
  r.first = (i0 < kRopeSplit0 ? base_f : (i0 < kRopeSplit1 ? base_h : base_w)) + i0;
  r.second = (i7 < kRopeSplit0 ? base_f : (i7 < kRopeSplit1 ? base_h : base_w)) + i0;
  // pairs [0, 22) frame, [22, 43) image row, [43, 64) column: lane 2 changes segment at pair 22, lane 5 at pair 43
  r.split = c16 == 2 ? kRopeSplit0 - 16 : (c16 == 5 ? kRopeSplit1 - 40 : 8);
  return r;
}

// KIND: PrepParams::kind, a template argument so that every kernel instantiation carries the registers of its own
// variant only (with a run-time switch the three variants' table reads add up).
template <int DT, int KIND, bool kFused = false>
__device__ __forceinline__ void prep16(float* x, const PrepParams& pp, const RopeLds& rl, int b, int row, int h,
                                       int c16, bool staged = true, const float* row_rms = nullptr) {
  if constexpr (KIND == 2) {
    prep16_qwen<DT, kFused>(x, pp, row, c16);
    return;
  }
  if (pp.inv_rms != nullptr) {
    // (row_rms: the row's statistic where the caller holds it already, e.g. in LDS)
    const float r = row_rms != nullptr ? *row_rms : pp.inv_rms[(int64_t)b * pp.L + row];
    norm16<DT>(x, r, pp.weight + h * kD + c16 * 16);
  }
  if constexpr (KIND == 3) {
    if (pp.rot != nullptr && row < pp.rot_rows) {
      const float4* m4 = pp.rot + (int64_t)row * (kD / 2) + c16 * 8;
#pragma unroll
      for (int j = 0; j < 8; ++j) comfy_pair<DT>(x[2 * j], x[2 * j + 1], m4[j]);
    }
    return;
  }
  if (pp.freqs != nullptr) {
    const int gh = pp.grid[b][1], gw = pp.grid[b][2];
    const int plane = gh * gw;
    if (row < pp.grid[b][0] * plane) {
      int rem, wi;
      const int f = small_div(row, plane, &rem);
      const int hi = small_div(rem, gw, &wi);
      // one table, three segments; a lane's 8 pairs lie in two of them at most
      auto rotate = [&](const double2* tab, int base_f, int base_h, int base_w) {
        const RopeLaneIndex li = rope_lane_index(c16, base_f, base_h, base_w);
#pragma unroll
        for (int j = 0; j < 8; ++j) rotate_pair<DT>(x[2 * j], x[2 * j + 1], tab[(j < li.split ? li.first : li.second) + j]);
      };
      if (pp.lds_frames > 0 && staged)  // uniform (staged == false: a row outside the rows `rl` was staged for)
        rotate(rl.frame, (f - rl.f0) * kRopeN0,
               (int)(rl.height - rl.frame) + (f * gh + hi - rl.gr0) * kRopeN1 - kRopeSplit0,
               (int)(rl.width - rl.frame) + wi * kRopeN2 - kRopeSplit1);
      else
        rotate(reinterpret_cast<const double2*>(pp.freqs), f * (kD / 2), hi * (kD / 2), wi * (kD / 2));
    }
  }
}

// Dynamic LDS of the kernels that rotate: the staged factors.
extern __shared__ __attribute__((aligned(16))) double2 s_rope_tables[];

template <int PRE>
__device__ __forceinline__ RopeLds maybe_stage_rope(const PrepParams& pp, int b, int row0, int nrows) {
  RopeLds rl{};
  if constexpr (PRE == 1) {
    if (pp.freqs != nullptr && pp.lds_frames > 0) rl = stage_rope(pp, b, row0, nrows, s_rope_tables);
  }
  return rl;
}

// 1 / sqrt(mean(x^2) + eps) of every token row x[b, l, 0 : n8*8].  One wave per row: lane i takes the
// groups of 8 channels i, i+64, i+128, ... in order, adding the 8 squares of each one after the other
// (fp32, squares of half values are exact); the 64 lane sums meet in an adjacent-pair tree.  The order
// is part of the result.  grid = (ceil(L / 4), B), 256 threads.
// the statistic of one row, by one wave (every lane returns it)
template <int DT>
__device__ __forceinline__ float row_inv_rms_of(const uint16_t* base, int n8, float n_channels, float eps, int lane) {
  float acc = 0.0f;
  for (int g = lane; g < n8; g += 64) {
    float v[8];
    widen8<DT>(*reinterpret_cast<const uint4*>(base + g * 8), v);
#pragma unroll
    for (int e = 0; e < 8; ++e) acc = __fmaf_rn(v[e], v[e], acc);
  }
  acc = over_lanes<Sum>(acc);
  // sqrtf, not __fsqrt_rn: the latter is the 1-ulp native instruction in this toolchain, the former is
  // correctly rounded (the build passes -fhip-fp32-correctly-rounded-divide-sqrt)
  return __fdiv_rn(1.0f, sqrtf(__fdiv_rn(acc, n_channels) + eps));
}

template <int DT>
__global__ __launch_bounds__(kThreads) void row_inv_rms_kernel(const uint16_t* __restrict__ x, int64_t sB, int64_t sL,
                                                               int L, int n8, float n_channels, float eps,
                                                               float* __restrict__ inv_rms) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), b = blockIdx.y;
  if (row >= L) return;
  const float r = row_inv_rms_of<DT>(x + b * sB + (int64_t)row * sL, n8, n_channels, eps, lane);
  if (lane == 0) inv_rms[(int64_t)b * L + row] = r;
}

// ---------------------------------------------------------------------------------------
// Column reduction over a chunk of 256 rows.  OP 0: fp32 sum in the frozen order (slot i%32
// sequential over the chunk's 8 row groups, then an adjacent-pair tree over the 32 slots).
// OP 1: max |x| (order free).  OP 2: max |x - centre[d]| over the rows that exist (V smoothing: the
// centre is the channel mean).  grid = (nch, H, B).
// ---------------------------------------------------------------------------------------
template <int DT, int OP, int PRE>
__device__ __forceinline__ void col_partial_chunk(int ch, int h, int b, const uint16_t* __restrict__ x, int64_t sB, int64_t sL,
                                                  int64_t sH, int H, int L_all, int d_in, float* __restrict__ part, int nch,
                                                  const PrepParams& pp, const float* __restrict__ centre) {
  constexpr bool kSum = OP == 0;
  const int t = threadIdx.x, slot = t >> 3, c16 = t & 7;
  const int L = c16 * 16 < d_in ? L_all : 0;  // channels at or past d_in (head size 64) read as zero padding
  const uint16_t* base = x + b * sB + h * sH + c16 * 16;
  const RopeLds rl = maybe_stage_rope<PRE>(pp, b, ch * kMeanChunk, kMeanChunk);
  float acc[16];
  if constexpr (PRE) {
    // all loads first, then the rows one after the other as they arrive (as in quant_k_chunk)
    uint4 raw[kMeanChunk / kSlots][2];
#pragma unroll
    for (int i = 0; i < kMeanChunk / kSlots; ++i) {
      const int row = ch * kMeanChunk + i * kSlots + slot;
      fetch_row16(base + (int64_t)row * sL, row < L, raw[i]);
    }
#pragma unroll
    for (int i = 0; i < kMeanChunk / kSlots; ++i) {
      const int row = ch * kMeanChunk + i * kSlots + slot;
      float x[16];
      widen8<DT>(raw[i][0], x);
      widen8<DT>(raw[i][1], x + 8);
      if (row < L) prep16<DT, PRE>(x, pp, rl, b, row, h, c16);
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        if (i == 0)
          acc[e] = kSum ? x[e] : fabsf(x[e]);
        else
          acc[e] = kSum ? acc[e] + x[e] : fmaxf(acc[e], fabsf(x[e]));
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  } else {
    // all sixteen loads of the lane are issued first and stay in flight as 16-bit values; they are widened and
    // folded in row order as they arrive (keeping them as fp32 costs twice the registers and a wave per SIMD)
    uint4 raw[kMeanChunk / kSlots][2];
#pragma unroll
    for (int i = 0; i < kMeanChunk / kSlots; ++i) {
      const int row = ch * kMeanChunk + i * kSlots + slot;
      raw[i][0] = raw[i][1] = make_uint4(0, 0, 0, 0);
      if (row < L) {
        raw[i][0] = *reinterpret_cast<const uint4*>(base + (int64_t)row * sL);
        raw[i][1] = *reinterpret_cast<const uint4*>(base + (int64_t)row * sL + 8);
      }
    }
    float cen[16];
    if constexpr (OP == 2) {
#pragma unroll
      for (int e = 0; e < 16; ++e) cen[e] = centre[((int64_t)b * H + h) * kD + c16 * 16 + e];
    }
#pragma unroll
    for (int i = 0; i < kMeanChunk / kSlots; ++i) {
      const int row = ch * kMeanChunk + i * kSlots + slot;
      float x[16];
      widen8<DT>(raw[i][0], x);
      widen8<DT>(raw[i][1], x + 8);
      if constexpr (OP == 2) {
        if (row < L) {
#pragma unroll
          for (int e = 0; e < 16; ++e) x[e] = x[e] - cen[e];
        }
      }
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        if (i == 0)
          acc[e] = kSum ? x[e] : fabsf(x[e]);
        else
          acc[e] = kSum ? acc[e] + x[e] : fmaxf(acc[e], fabsf(x[e]));
      }
    }
  }
  __shared__ __attribute__((aligned(16))) float s_w[4][kD];
  const int wave = t >> 6, lane = t & 63;
  store_slots16(over_slots16<typename std::conditional<kSum, Sum, Max>::type>(acc), lane, s_w[wave]);
  __syncthreads();
  if (t < kD) {
    const float lo = kSum ? s_w[0][t] + s_w[1][t] : fmaxf(s_w[0][t], s_w[1][t]);
    const float hi = kSum ? s_w[2][t] + s_w[3][t] : fmaxf(s_w[2][t], s_w[3][t]);
    part[(((int64_t)b * H + h) * nch + ch) * kD + t] = kSum ? lo + hi : fmaxf(lo, hi);
  }
}

template <int DT, int OP, int PRE>
__global__ __launch_bounds__(kThreads) void col_partial_kernel(const uint16_t* __restrict__ x, int64_t sB, int64_t sL,
                                                               int64_t sH, int H, int L_all, int d_in, float* __restrict__ part,
                                                               int nch, const PrepParams pp,
                                                               const float* __restrict__ centre) {
  col_partial_chunk<DT, OP, PRE>(blockIdx.x, blockIdx.y, blockIdx.z, x, sB, sL, sH, H, L_all, d_in, part, nch, pp, centre);
}

// Finalisation of the column reductions.  grid = B*H, 1024 threads.  All chunk partials of the
// head are first pulled into LDS with independent, coalesced loads (the naive form - one
// dependent global load per chunk - costs a memory latency per chunk); 128 threads then combine
// them in increasing chunk order, which for the sum is part of the specification.
constexpr int kFinThreads = 1024;
constexpr int kFinMaxChunks = 96;  // partials staged per pass: 96 x 128 floats = 48 KiB of LDS

template <int OP>
__device__ __forceinline__ float combine_partials(const float* __restrict__ part, int nch, float* s_part) {
  const int d = threadIdx.x & (kD - 1);
  float acc = 0.0f;
  bool first = true;
  for (int c0 = 0; c0 < nch; c0 += kFinMaxChunks) {
    const int n = min(kFinMaxChunks, nch - c0);
    __syncthreads();
    // 96 x 128 floats by 1024 threads: twelve independent loads each, all in flight together
    float v[kFinMaxChunks * kD / kFinThreads];
#pragma unroll
    for (int j = 0; j < kFinMaxChunks * kD / kFinThreads; ++j) {
      const int idx = (int)threadIdx.x + kFinThreads * j;
      v[j] = idx < n * kD ? part[(int64_t)c0 * kD + idx] : 0.0f;
    }
#pragma unroll
    for (int j = 0; j < kFinMaxChunks * kD / kFinThreads; ++j) s_part[(int)threadIdx.x + kFinThreads * j] = v[j];
    __syncthreads();
    if (threadIdx.x < kD) {
      int c = 0;
      if (first) {
        acc = s_part[d];
        first = false;
        c = 1;
      }
      // chunk order is part of the specification for the sum; batches of 16 keep the LDS reads ahead of the adds
      for (; c + 16 <= n; c += 16) {
        float w[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) w[i] = s_part[(c + i) * kD + d];
#pragma unroll
        for (int i = 0; i < 16; ++i) acc = OP == 0 ? acc + w[i] : fmaxf(acc, w[i]);
      }
      for (; c < n; ++c) acc = OP == 0 ? acc + s_part[c * kD + d] : fmaxf(acc, s_part[c * kD + d]);
    }
  }
  return acc;
}

// The numbers of the attention's blocks (kBatchStarts), by one wave of a workgroup of its own, the launch's first: the others'
// work hides it (as the last one it was 0.2 us of a first stage of 5.8).
__host__ __device__ __forceinline__ int numbers_batch(const BatchNumbers& n) { return n.starts != nullptr ? 1 : 0; }
__device__ __forceinline__ void number_batch(const BatchNumbers& n) {
  if (threadIdx.x >= 64) return;
  int rows, keys;
  const int mine = batch_number(n, threadIdx.x, rows, keys);
  if (threadIdx.x < kBatchStarts) n.starts[threadIdx.x] = mine;
}

// chunk sums -> mean rounded to the input dtype, stored widened
__global__ __launch_bounds__(kFinThreads) void k_mean_finalize_kernel(const float* __restrict__ part, int nch, int L,
                                                                      int dtype, int smooth,
                                                                      float* __restrict__ k_mean, int* status, const BatchNumbers numbers) {
  __shared__ float s_part[kFinMaxChunks * kD];
  const int more = numbers_batch(numbers);
  if ((int)blockIdx.x < more) return number_batch(numbers);
  const int bh = blockIdx.x - more;
  if (status != nullptr && bh == 0 && threadIdx.x == 0) *status = 0;  // this path has no wait that could expire
  const float tot = combine_partials<0>(part + (int64_t)bh * nch * kD, nch, s_part);
  if (threadIdx.x < kD) {
    const float mean = __fdiv_rn(tot, (float)L);
    k_mean[bh * kD + threadIdx.x] = smooth ? round_to_half_dtype(mean, dtype) : 0.0f;
  }
}

// chunk abs-max -> scale and its inverse; `zero_mean` (optional) is the mean slot to clear when V is not smoothed
__global__ __launch_bounds__(kFinThreads) void v_scale_finalize_kernel(const float* __restrict__ part, int nch,
                                                                       float* __restrict__ v_scale,
                                                                       float* __restrict__ v_inv,
                                                                       float* __restrict__ zero_mean, int* status) {
  __shared__ float s_part[kFinMaxChunks * kD];
  const int bh = blockIdx.x;
  if (status != nullptr && bh == 0 && threadIdx.x == 0) *status = 0;
  const float amax = combine_partials<1>(part + (int64_t)bh * nch * kD, nch, s_part);
  if (threadIdx.x < kD) {
    const bool nz = amax > 0.0f;
    v_scale[bh * kD + threadIdx.x] = nz ? __fdiv_rn(amax, 448.0f) : 0.0f;
    v_inv[bh * kD + threadIdx.x] = nz ? __fdiv_rn(448.0f, amax) : 0.0f;
    if (zero_mean != nullptr) zero_mean[bh * kD + threadIdx.x] = 0.0f;
  }
}

// max over the workgroup of a non-negative per-thread value
__device__ __forceinline__ float block_max(float v, float* s_red) {
  v = over_lanes<Max>(v);
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) s_red[wave] = v;
  __syncthreads();
  return fmaxf(fmaxf(s_red[0], s_red[1]), fmaxf(s_red[2], s_red[3]));
}

// Block mean from per-thread partial sums (thread = row slot x 16 channels; a slot has added its rows in increasing
// order): the 32 slots meet in an adjacent-pair tree - three steps inside a wave, the four waves through LDS - the sum
// is divided by the number of rows that exist and rounded to the half type.  The frozen order of the block averages
// (block_mean_kernel); the quantizers that take a block's average along use the same code, hence give the same bits.
template <int DT>
__device__ __forceinline__ void store_block_mean(float (&acc)[16], int t, float n_rows, uint16_t* __restrict__ out_row,
                                                 float (*s_w)[kD]) {
  const int wave = t >> 6, lane = t & 63;
  store_slots16(over_slots16<Sum>(acc), lane, s_w[wave]);
  __syncthreads();
  if (t < kD) {
    const float sum = (s_w[0][t] + s_w[1][t]) + (s_w[2][t] + s_w[3][t]);
    const float mean = __fdiv_rn(sum, n_rows);
    uint16_t bits;
    if constexpr (DT == KSANA_SAGE_BF16) {
      bits = __builtin_bit_cast(uint16_t, (__bf16)mean);
    } else {
      bits = __builtin_bit_cast(uint16_t, (_Float16)mean);
    }
    out_row[t] = bits;
  }
}

// a row of Q from its lanes' channels: transform, premul_lane = premul * fwht_lane_sign(c16), scale and codes
__device__ __forceinline__ void quant_q_row(float* x, int c16, float premul_lane, float* scale, int8_t* codes) {
  fwht128(x, c16);
  float amax = 0.0f;
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    x[e] = x[e] * premul_lane;
    amax = fmaxf(amax, fabsf(x[e]));
  }
  amax = fmaxf(amax, lane_xor<1>(amax));
  amax = fmaxf(amax, lane_xor<2>(amax));
  amax = fmaxf(amax, lane_xor<4>(amax));
  const Int8Scale r = int8_scale(amax);
  if (c16 == 0) *scale = r.scale;
  store_out16(codes + c16 * 16, pack_int8x16(x, r.inv));
}

// ---------------------------------------------------------------------------------------
// Q: Hadamard transform, fold sm_scale*log2(e)/128, one int8 scale per query row.  One
// workgroup handles 128 rows (4 per row slot).  grid = (lq_pad/128, H, B).  Output row-major
// int8 [B, H, lq_pad, 128] and fp32 [B, H, lq_pad]; rows at or beyond L come out as zeros.
// ---------------------------------------------------------------------------------------
// POOL: the workgroup's 128 rows are one block of the sparse-linear backend's block map; their average (of the input
// as it is) goes to pooled[b, h, blk, :] - what block_mean_kernel would read q a second time for.
template <int DT, int PRE, bool POOL>
__device__ __forceinline__ void quant_q_block(int blk, int h, int b, const uint16_t* __restrict__ q, int64_t sB, int64_t sL,
                                              int64_t sH, int H, int L_all, int d_in, int lq_pad, float premul,
                                              int8_t* __restrict__ q_i8, float* __restrict__ q_scale, const PrepParams& pp,
                                              uint16_t* __restrict__ pooled) {
  static_assert(!(POOL && PRE), "block averages are taken of the tensor as it is");
  const int t = threadIdx.x, slot = t >> 3, c16 = t & 7;
  const int L = c16 * 16 < d_in ? L_all : 0;  // channels at or past d_in (head size 64) read as zero padding
  const uint16_t* base = q + b * sB + h * sH + c16 * 16;
  constexpr int kRowsPerWg = 128, R = kRowsPerWg / kSlots;
  const int64_t bh = (int64_t)b * H + h;
  const RopeLds rl = maybe_stage_rope<PRE>(pp, b, blk * kRowsPerWg, kRowsPerWg);
  const float premul_lane = premul * fwht_lane_sign(c16);
  auto finish_row = [&](float* xr, int row) {
    quant_q_row(xr, c16, premul_lane, q_scale + bh * lq_pad + row, q_i8 + (bh * lq_pad + row) * kD);
  };
  if constexpr (PRE) {
    // The norm and the rotation are arithmetic-heavy (vector fp64): one row at a time with only the next row's two
    // loads in flight keeps the kernel at half the registers of "load all, then work", i.e. at twice the waves.
    uint4 nxt[2];
    fetch_row16(base + (int64_t)(blk * kRowsPerWg + slot) * sL, blk * kRowsPerWg + slot < L, nxt);
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int row = blk * kRowsPerWg + i * kSlots + slot;
      const uint4 cur0 = nxt[0], cur1 = nxt[1];
      if (i + 1 < R) fetch_row16(base + (int64_t)(row + kSlots) * sL, row + kSlots < L, nxt);
      float xr[16];
      widen8<DT>(cur0, xr);
      widen8<DT>(cur1, xr + 8);
      if (row < L) prep16<DT, PRE>(xr, pp, rl, b, row, h, c16);
      finish_row(xr, row);
      __builtin_amdgcn_sched_barrier(0);
    }
  } else {
    float x[R][16];
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int row = blk * kRowsPerWg + i * kSlots + slot;
      load_row16<DT>(base + (int64_t)row * sL, row < L, x[i]);
    }
    if constexpr (POOL) {
      float acc[16];
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[e] = ((x[0][e] + x[1][e]) + x[2][e]) + x[3][e];
      static_assert(R == 4, "four rows per slot");
      __shared__ __attribute__((aligned(16))) float s_w[4][kD];
      store_block_mean<DT>(acc, t, (float)min(kRowsPerWg, L_all - blk * kRowsPerWg),
                           pooled + (bh * (lq_pad / kRowsPerWg) + blk) * kD, s_w);
    }
#pragma unroll
    for (int i = 0; i < R; ++i) finish_row(x[i], blk * kRowsPerWg + i * kSlots + slot);
  }
}

template <int DT, int PRE, bool POOL = false>
__global__ __launch_bounds__(kThreads) void quant_q_kernel(const uint16_t* __restrict__ q, int64_t sB, int64_t sL,
                                                           int64_t sH, int H, int L_all, int d_in, int lq_pad, float premul,
                                                           int8_t* __restrict__ q_i8, float* __restrict__ q_scale,
                                                           const PrepParams pp, uint16_t* __restrict__ pooled = nullptr) {
  quant_q_block<DT, PRE, POOL>(blockIdx.x, blockIdx.y, blockIdx.z, q, sB, sL, sH, H, L_all, d_in, lq_pad, premul, q_i8, q_scale,
                               pp, pooled);
}

// ---------------------------------------------------------------------------------------
// Q with a norm over the whole token row folded in (Wan), from ONE pass over HBM.  A workgroup takes 8 whole token
// rows, all heads.  First their statistics, as row_inv_rms_kernel takes them (one wave per row, two rows per wave,
// both at a time) - and, where the caller passes k, the statistics of the same rows of k, whose own quantizer then
// needs no statistic pass of its own.  Then the heads, four at a time: a row slot is (row, one of four heads), 8 lanes
// x 16 channels each, the next four heads' loads in flight while these are normed, rotated, transformed and packed.
// The rows are read a second time there, microseconds after the first: from the caches, not from HBM.  Small
// workgroups on purpose: several generations of them pass through a compute unit, so the memory-bound statistics of
// some run next to the arithmetic-bound heads of others.
// grid = (ceil(max(lq_pad, k_L) / 8), B).
// ---------------------------------------------------------------------------------------
constexpr int kRowsQ = 8;                   // token rows per workgroup
constexpr int kHeadsQ = kSlots / kRowsQ;    // heads in work at a time: 4
struct RowStatOf {  // the rows of another tensor whose statistic the kernel takes along (ptr == nullptr: none)
  const uint16_t* ptr;
  int64_t sB, sL;
  int L, n8;
  float n_channels;
  float* inv_rms;  // [B, L]
};

template <int DT, int KIND>
__global__ __launch_bounds__(kThreads) void quant_q_rows_kernel(const uint16_t* __restrict__ q, int64_t sB, int64_t sL,
                                                                int64_t sH, int H, int L, int lq_pad, float premul,
                                                                float eps, int8_t* __restrict__ q_i8,
                                                                float* __restrict__ q_scale, const PrepParams pp,
                                                                float* __restrict__ rms_out, const RowStatOf ks,
                                                                int* __restrict__ clear, int n_clear) {
  const int r0 = blockIdx.x * kRowsQ, b = blockIdx.y;
  const int t = threadIdx.x, slot = t >> 3, c16 = t & 7;
  if (b == 0)  // the counters of the launch that follows
    for (int i = blockIdx.x * kThreads + t; i < n_clear; i += gridDim.x * kThreads) clear[i] = 0;
  const int wave = t >> 6, lane = t & 63;
  __shared__ float s_rms[kRowsQ];
  // ---- the rows' statistics: wave w takes rows 2 w and 2 w + 1 together (every row's sum adds its groups of 8
  // channels in the order of row_inv_rms_of) -------------------------------------------------------------------
  auto stats = [&](const uint16_t* x, int64_t xsB, int64_t xsL, int xL, int n8, float n_channels, float* out, bool keep) {
    constexpr int R = kRowsQ / 4;
    const int first = r0 + wave * R;
    if (first >= xL) return;  // wave-uniform
    const uint16_t* rbase = x + b * xsB + (int64_t)first * xsL;
    float acc[R];
#pragma unroll
    for (int i = 0; i < R; ++i) acc[i] = 0.0f;
#pragma unroll 4
    for (int g = lane; g < n8; g += 64) {
      uint4 raw[R];
#pragma unroll
      for (int i = 0; i < R; ++i)
        raw[i] = first + i < xL ? *reinterpret_cast<const uint4*>(rbase + i * xsL + g * 8) : make_uint4(0, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < R; ++i) {
        float v[8];
        widen8<DT>(raw[i], v);
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[i] = __fmaf_rn(v[e], v[e], acc[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const float a = over_lanes<Sum>(acc[i]);
      const float r = __fdiv_rn(1.0f, sqrtf(__fdiv_rn(a, n_channels) + eps));
      if (lane == 0 && first + i < xL) {
        out[(int64_t)b * xL + first + i] = r;
        if (keep) s_rms[wave * R + i] = r;
      }
    }
  };
  stats(q, sB, sL, L, H * (kD / 8), (float)(H * kD), rms_out, true);
  if (ks.ptr != nullptr) stats(ks.ptr, ks.sB, ks.sL, ks.L, ks.n8, ks.n_channels, ks.inv_rms, false);
  if (r0 >= lq_pad) return;  // rows that exist only in k
  __syncthreads();
  // ---- the heads, four at a time ------------------------------------------------------------------------------
  const int rloc = slot & (kRowsQ - 1), h0 = slot / kRowsQ;
  const int row = r0 + rloc;
  const bool live = row < L;
  // A token's rotation is the same for every head: the lane's 8 factors (pairs 8 * c16 + j of its row) are fetched
  // once, straight from the model's table (1 MiB, cache resident), and stay in registers for the whole head walk.
  bool rotates = false;
  double2 cs[KIND == 1 ? 8 : 1];
  float4 rm[KIND == 3 ? 8 : 1];
  if constexpr (KIND == 1) {
    if (pp.freqs != nullptr && live) {
      const int gh = pp.grid[b][1], gw = pp.grid[b][2], plane = gh * gw;
      if (row < pp.grid[b][0] * plane) {
        rotates = true;
        int rem, wi;
        const int f = small_div(row, plane, &rem);
        const int hi = small_div(rem, gw, &wi);
        const RopeLaneIndex li = rope_lane_index(c16, f * (kD / 2), hi * (kD / 2), wi * (kD / 2));
        const double2* tab = reinterpret_cast<const double2*>(pp.freqs);
#pragma unroll
        for (int j = 0; j < 8; ++j) cs[j] = tab[(j < li.split ? li.first : li.second) + j];
      }
    }
  } else {
    if (pp.rot != nullptr && live && row < pp.rot_rows) {
      rotates = true;
      const float4* m4 = pp.rot + (int64_t)row * (kD / 2) + c16 * 8;
#pragma unroll
      for (int j = 0; j < 8; ++j) rm[j] = m4[j];
    }
  }
  const float rinv = s_rms[rloc];
  const uint16_t* base = q + b * sB + (int64_t)row * sL + c16 * 16;
  const float premul_lane = premul * fwht_lane_sign(c16);
  uint4 nxt[2];
  fetch_row16(base + (int64_t)h0 * sH, live && h0 < H, nxt);
  for (int h = h0; h < H; h += kHeadsQ) {
    const uint4 cur0 = nxt[0], cur1 = nxt[1];
    if (h + kHeadsQ < H) fetch_row16(base + (int64_t)(h + kHeadsQ) * sH, live, nxt);
    float xr[16];
    widen8<DT>(cur0, xr);
    widen8<DT>(cur1, xr + 8);
    if (live) {
      norm16<DT>(xr, rinv, pp.weight + h * kD + c16 * 16);
      if (rotates) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          if constexpr (KIND == 1) rotate_pair<DT>(xr[2 * j], xr[2 * j + 1], cs[j]);
          else comfy_pair<DT>(xr[2 * j], xr[2 * j + 1], rm[j]);
        }
      }
    }
    fwht128(xr, c16);
    float amax = 0.0f;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      xr[e] = xr[e] * premul_lane;
      amax = fmaxf(amax, fabsf(xr[e]));
    }
    amax = fmaxf(amax, lane_xor<1>(amax));
    amax = fmaxf(amax, lane_xor<2>(amax));
    amax = fmaxf(amax, lane_xor<4>(amax));
    const Int8Scale r = int8_scale(amax);
    const int64_t bh = (int64_t)b * H + h;
    if (c16 == 0) q_scale[bh * lq_pad + row] = r.scale;
    store_out16(q_i8 + (bh * lq_pad + row) * kD + c16 * 16, pack_int8x16(xr, r.inv));
    __builtin_amdgcn_sched_barrier(0);
  }
}

// ---------------------------------------------------------------------------------------
// K: subtract the channel mean, Hadamard transform, one int8 scale per 64-row block = one
// workgroup.  grid = (nkb, H, B).  The tile is written in the order
// the attention kernel's int8 MFMA consumes it: fragment (t = row/32, s = 32-channel step)
// is 64 lanes x 16 bytes, lane = 32*(16-channel half within the step) + row%32.
// ---------------------------------------------------------------------------------------
// POOL: the workgroup's 64 rows are one key block of the sparse-linear backend's block map; the average of
// k - mean(k), each difference rounded to the tensor's half type first as the reference forms it, goes to
// pooled[b, h, blk, :] - what block_mean_kernel would read k a third time for.
// `mean`: where the head's channel means are found (128 floats, global memory or LDS) - called once the rows are on
// their way.
template <int DT, int PRE, bool POOL, typename Mean>
__device__ __forceinline__ void quant_k_block(int blk, int h, int b, const uint16_t* __restrict__ k, int64_t sB, int64_t sL,
                                              int64_t sH, int H, int L_all, int d_in, int nkb, Mean&& mean,
                                              int8_t* __restrict__ k_tiles, float* __restrict__ k_scale, const PrepParams& pp,
                                              uint16_t* __restrict__ pooled) {
  static_assert(!(POOL && PRE), "block averages are taken of the tensor as it is");
  const int t = threadIdx.x, slot = t >> 3, c16 = t & 7;
  const int L = c16 * 16 < d_in ? L_all : 0;  // channels at or past d_in (head size 64) read as zero padding
  const int64_t bh = (int64_t)b * H + h;
  const uint16_t* base = k + b * sB + h * sH + c16 * 16;
  constexpr int R = kBlkK / kSlots;
  uint4 raw[R][2];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int row = blk * kBlkK + i * kSlots + slot;
    fetch_row16(base + (int64_t)row * sL, row < L, raw[i]);
  }
  const float* k_mean = mean();
  float km[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) km[e] = k_mean[c16 * 16 + e];
  const RopeLds rl = maybe_stage_rope<PRE>(pp, b, blk * kBlkK, kBlkK);
  float x[R][16];
  float amax = 0.0f;
  [[maybe_unused]] float pool_acc[16];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int row = blk * kBlkK + i * kSlots + slot;
    const bool valid = row < L;
    widen8<DT>(raw[i][0], x[i]);
    widen8<DT>(raw[i][1], x[i] + 8);
    if constexpr (PRE) {
      if (valid) prep16<DT, PRE>(x[i], pp, rl, b, row, h, c16);
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      x[i][e] = valid ? x[i][e] - km[e] : 0.0f;
    }
    if constexpr (POOL) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const float d = valid ? through_half<DT>(x[i][e]) : 0.0f;
        pool_acc[e] = i == 0 ? d : pool_acc[e] + d;
      }
    }
    fwht128(x[i], c16);
#pragma unroll
    for (int e = 0; e < 16; ++e) amax = fmaxf(amax, fabsf(x[i][e]));
  }
  if constexpr (POOL) {
    __shared__ __attribute__((aligned(16))) float s_w[4][kD];
    store_block_mean<DT>(pool_acc, t, (float)min(kBlkK, L_all - blk * kBlkK), pooled + (bh * nkb + blk) * kD, s_w);
  }
  __shared__ float s_red[4];
  amax = block_max(amax, s_red);
  const Int8Scale r = int8_scale(amax);
  const float inv_lane = r.inv * fwht_lane_sign(c16);  // the transform left this lane's values times that sign
  if (t == 0) k_scale[bh * nkb + blk] = r.scale;
  int8_t* tile = k_tiles + (bh * nkb + blk) * (int64_t)kTileBytes;
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int frag = i * 4 + (c16 >> 1);
    const int lane = (c16 & 1) * 32 + slot;
    store_out16(tile + (frag * 64 + lane) * 16, pack_int8x16(x[i], inv_lane));
  }
}

template <int DT, int PRE, bool POOL = false>
__global__ __launch_bounds__(kThreads) void quant_k_kernel(const uint16_t* __restrict__ k, int64_t sB, int64_t sL,
                                                           int64_t sH, int H, int L_all, int d_in, int nkb,
                                                           const float* __restrict__ k_mean,
                                                           int8_t* __restrict__ k_tiles, float* __restrict__ k_scale,
                                                           const PrepParams pp, uint16_t* __restrict__ pooled = nullptr) {
  // Heads and batch entries from the last one down: this pass follows the column-sum pass over the same tensor, which
  // went upwards, so what that pass touched last - and the last-level cache may still hold - is read first.
  const int h = (int)gridDim.y - 1 - (int)blockIdx.y, b = (int)gridDim.z - 1 - (int)blockIdx.z;
  quant_k_block<DT, PRE, POOL>(blockIdx.x, h, b, k, sB, sL, sH, H, L_all, d_in, nkb,
                               [&] { return k_mean + ((int64_t)b * H + h) * kD; }, k_tiles, k_scale, pp, pooled);
}

// ---------------------------------------------------------------------------------------
// V: one workgroup per 64-row block.  grid = (nkb, H, B).  Scales with 448/amax[d], converts
// to e4m3fn, transposes through LDS and writes the V^T tile in the order the fp8 MFMA
// consumes it: chunk (dt = d/32, tt = half of the 64 rows) is 64 lanes x 16 bytes,
// lane = 32*hh + d%32, byte r <-> row 32*tt + 8*(r/4) + 4*hh + r%4.
// ---------------------------------------------------------------------------------------
// `factors`: where the head's 128 factors 448 / amax are found - called once the rows are on their way.
template <int DT, bool CENTRE, typename Factors>
__device__ __forceinline__ void quant_v_block(int blk, int h, int b, const uint16_t* __restrict__ v, int64_t sB, int64_t sL,
                                              int64_t sH, int H, int L_all, int d_in, int nkb, Factors&& factors,
                                              const float* __restrict__ v_mean, uint8_t* __restrict__ v_tiles) {
  const int t = threadIdx.x, slot = t >> 3, c16 = t & 7;
  const int L = c16 * 16 < d_in ? L_all : 0;  // channels at or past d_in (head size 64) read as zero padding
  const int64_t bh = (int64_t)b * H + h;
  const uint16_t* base = v + b * sB + h * sH + c16 * 16;
  constexpr int kStride = kD + 16;  // LDS row pitch in bytes
  __shared__ __attribute__((aligned(16))) uint8_t s_v[kBlkK * kStride];
  uint4 raw[kBlkK / kSlots][2];
#pragma unroll
  for (int i = 0; i < kBlkK / kSlots; ++i) {
    const int row = blk * kBlkK + i * kSlots + slot;
    fetch_row16(base + (int64_t)row * sL, row < L, raw[i]);
  }
  const float* v_inv = factors();
  float inv[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) inv[e] = v_inv[c16 * 16 + e];
  float mean[16];
  if constexpr (CENTRE) {
#pragma unroll
    for (int e = 0; e < 16; ++e) mean[e] = v_mean[bh * kD + c16 * 16 + e];
  }
#pragma unroll
  for (int i = 0; i < kBlkK / kSlots; ++i) {
    const int r = i * kSlots + slot;
    [[maybe_unused]] const int row = blk * kBlkK + r;
    float x[16];
    widen8<DT>(raw[i][0], x);
    widen8<DT>(raw[i][1], x + 8);
    if constexpr (CENTRE) {  // rows past the end stay zero
      if (row < L) {
#pragma unroll
        for (int e = 0; e < 16; ++e) x[e] = x[e] - mean[e];
      }
    }
    uint32_t w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = fminf(fmaxf(x[4 * j + e] * inv[4 * j + e], -448.0f), 448.0f);
      int packed = 0;
      packed = __builtin_amdgcn_cvt_pk_fp8_f32(y[0], y[1], packed, false);
      packed = __builtin_amdgcn_cvt_pk_fp8_f32(y[2], y[3], packed, true);
      w[j] = (uint32_t)packed;
    }
    *reinterpret_cast<uint4*>(&s_v[r * kStride + c16 * 16]) = make_uint4(w[0], w[1], w[2], w[3]);
  }
  __syncthreads();
  uint8_t* tile = v_tiles + (bh * nkb + blk) * (int64_t)kTileBytes;
#pragma unroll
  for (int i = 0; i < kTileBytes / 16 / kThreads; ++i) {
    const int oc = i * kThreads + t;
    const int dt = oc >> 7, tt = (oc >> 6) & 1, lane = oc & 63;
    const int hh = lane >> 5, d = dt * 32 + (lane & 31);
    uint32_t w[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      uint32_t acc = 0;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int row = 32 * tt + 8 * g + 4 * hh + c;
        acc |= (uint32_t)s_v[row * kStride + d] << (8 * c);
      }
      w[g] = acc;
    }
    store_out16(tile + oc * 16, make_uint4(w[0], w[1], w[2], w[3]));
  }
}

template <int DT, bool CENTRE>
__global__ __launch_bounds__(kThreads) void quant_v_kernel(const uint16_t* __restrict__ v, int64_t sB, int64_t sL,
                                                           int64_t sH, int H, int L_all, int d_in, int nkb,
                                                           const float* __restrict__ v_inv,
                                                           const float* __restrict__ v_mean,
                                                           uint8_t* __restrict__ v_tiles) {
  // (heads and batch entries from the last one down, like quant_k_kernel: the abs-max pass went upwards)
  const int h = (int)gridDim.y - 1 - (int)blockIdx.y, b = (int)gridDim.z - 1 - (int)blockIdx.z;
  quant_v_block<DT, CENTRE>(blockIdx.x, h, b, v, sB, sL, sH, H, L_all, d_in, nkb,
                            [&] { return v_inv + ((int64_t)b * H + h) * kD; }, v_mean, v_tiles);
}

// ---------------------------------------------------------------------------------------
// One-read quantizers for K and V.
//
// The two-kernel form above reads K (and V) twice: once for the column statistic of the whole
// sequence, once to quantize.  Here a workgroup keeps its 256-row chunk in registers (as the 16-bit
// values it loaded: 64 registers per lane) across the point where the statistic of its head becomes
// known, so every input byte crosses the memory bus once:
//   1. load the chunk, reduce its columns, publish the chunk's partial result;
//   2. count the chunk in on its head's counter; the workgroup that finds itself last combines the
//      partial results (K: in chunk order, which is part of the specification; V: the maximum needs
//      no order and is taken with an atomic) and raises the head's ready flag;
//   3. every other workgroup of the head waits for the flag, then all of them quantize from registers.
// Waiting is safe because workgroups are dispatched in index order: a waiting workgroup only waits for
// workgroups with indices of the same head, all of which have been dispatched or are next in line on
// their part of the chip, and the launcher only picks this form when a head's chunks are a fraction
// of the workgroups the chip holds at once.  The wait is bounded by a wall-clock limit all the same (a device
// shared with other work may hold fewer workgroups than the launcher counted on): on expiry the workgroup
// records it in `status` and takes the head's statistic from the input itself - every chunk of the head, in the
// specified order - so every wave ends and the result is the same bits, only later.
// ---------------------------------------------------------------------------------------
constexpr int kChunkRowsPerSlot = kMeanChunk / kSlots;  // 8

// Opaque use+def: what was derived from the 16-bit values before this point (their fp32 forms) is not carried
// across it; only the 16-bit values themselves stay in registers.
__device__ __forceinline__ void forget_derived(uint4 (&raw)[kChunkRowsPerSlot][2]) {
#pragma unroll
  for (int i = 0; i < kChunkRowsPerSlot; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
      asm volatile("" : "+v"(raw[i][j].x), "+v"(raw[i][j].y), "+v"(raw[i][j].z), "+v"(raw[i][j].w));
}

template <int DT>
__device__ __forceinline__ uint4 narrow8(const float* x) {
  uint32_t w[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (DT == KSANA_SAGE_BF16) {
      // the values are exactly representable (they went through the half type): truncation is exact
      w[i] = (__float_as_uint(x[2 * i]) >> 16) | (__float_as_uint(x[2 * i + 1]) & 0xffff0000u);
    } else {
      typedef _Float16 h2 __attribute__((ext_vector_type(2)));
      h2 p = {(_Float16)x[2 * i], (_Float16)x[2 * i + 1]};
      w[i] = __builtin_bit_cast(uint32_t, p);
    }
  }
  return make_uint4(w[0], w[1], w[2], w[3]);
}

// Communication between workgroups (which may sit behind different L2 caches) goes through accesses that are
// coherent at device scope by themselves - relaxed device-scope atomics: stores write through, loads are served
// from the point of coherence - ordered by waiting for their completion (a workgroup-scope fence is that wait
// plus a compiler barrier).  Device-scope acquire / release fences are avoided on purpose: each one writes back or
// invalidates a whole L2, and a polling loop built on them starves the loads of every other workgroup.
__device__ __forceinline__ int load_shared_i32(const int* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float load_shared_f32(const float* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void publish_f32(float* p, float v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// every memory access this wave has issued has completed - for the write-through stores and the atomics above:
// has reached the point of coherence - and the compiler moves no access across
__device__ __forceinline__ void complete_accesses() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory"); }

struct HeadSync {
  int* counter;      // [B*H][kSyncStride] chunks counted in (one word per head, each in a cache line of its own)
  int* ready;        // [B*H][kSyncStride] set once the head's statistic is published
  int* status;       // [1]   set to 1 when a wait ran into its time limit
  long long limit;   // wall-clock ticks (100 MHz) a workgroup waits at most; 0 and negative: see QuantOptions
  int* host_word;    // nullptr, or a word in host memory the device can write: set to 1 when a bound > 0 expires
};

// Thread 0 waits until the head's ready flag is up (or the time limit passes), then the workgroup meets.  Returns
// true (to every thread) when the workgroup has to take the statistic from the input itself: the limit passed first,
// or the limit is negative, which means "do not even look".
__device__ __forceinline__ bool wait_for_head(const int* flag, const HeadSync& sy) {
  __shared__ int s_gave_up;
  if (threadIdx.x == 0) {
    int gave_up = 0;
    if (sy.limit < 0) {
      gave_up = 1;
    } else if (load_shared_i32(flag) < 1) {
      const long long t0 = wall_clock64();
      while (load_shared_i32(flag) < 1) {
        __builtin_amdgcn_s_sleep(16);  // ~0.5 us between polls
        if (wall_clock64() - t0 > sy.limit) {
          gave_up = 1;
          break;
        }
      }
    }
    if (gave_up) {
      __hip_atomic_store(sy.status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (sy.limit > 0 && sy.host_word != nullptr)
        __hip_atomic_store(sy.host_word, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    s_gave_up = gave_up;
    complete_accesses();
  }
  __syncthreads();
  return s_gave_up != 0;
}

// Staging of one head's chunk partials for the workgroup that combines them: kFinStage chunks per
// pass (16 KiB of LDS), fetched with loads that are all in flight together; the next pass is fetched while this one
// is combined.
constexpr int kFinStage = 32;
constexpr int kFinLoads = kFinStage * kD / kThreads;  // per thread and pass: 32

__device__ __forceinline__ void fetch_partials(const float* hp, int c0, int nch, float (&v)[kFinLoads]) {
  const int n = (min(kFinStage, nch - c0)) * kD;
#pragma unroll
  for (int j = 0; j < kFinLoads; ++j) {
    const int idx = (int)threadIdx.x + kThreads * j;
    v[j] = idx < n ? load_shared_f32(hp + (int64_t)c0 * kD + idx) : 0.0f;
  }
}
__device__ __forceinline__ void stage_partials(const float (&v)[kFinLoads], float* s_part) {
#pragma unroll
  for (int j = 0; j < kFinLoads; ++j) s_part[(int)threadIdx.x + kThreads * j] = v[j];
}

// The large LDS buffer of a chunk, one for K's and V's code where a kernel holds both (and asks for the same size)
constexpr int kChunkLdsK = kFinStage * kD * 4, kChunkLdsV = 2 * kBlkK * (kD + 16);
static_assert(kChunkLdsV >= kChunkLdsK, "V's is the size for both");
template <int kBytes>
__device__ __forceinline__ uint8_t* chunk_lds() {
  __shared__ __attribute__((aligned(16))) uint8_t s[kBytes];
  return s;
}

// SOLO: the head is this one chunk (at most 256 rows), so its sums are the head's and nobody is waited for.
// n_use: the head's tiles that are wanted, at most nkb; a chunk without any leaves once its sums are counted in.
template <int DT, int PRE, bool SOLO, int kBytes = kChunkLdsV>
__device__ __forceinline__ void quant_k_chunk(int bh, int ch, const uint16_t* __restrict__ k, int64_t sB, int64_t sL,
                                              int64_t sH, int H, int L_all, int d_in, int nkb, int nch,
                                              float* __restrict__ part, float* k_mean, int dtype, int smooth,
                                              int8_t* __restrict__ k_tiles, float* __restrict__ k_scale,
                                              const PrepParams& pp, const HeadSync& sy, int n_use) {
  const int b = bh / H, h = bh - b * H;
  const int t = threadIdx.x, slot = t >> 3, c16 = t & 7;
  const int L = c16 * 16 < d_in ? L_all : 0;  // channels at or past d_in (head size 64) read as zero padding
  const int wave = t >> 6, lane = t & 63;
  const uint16_t* base = k + b * sB + h * sH + c16 * 16;
  const RopeLds rl = maybe_stage_rope<PRE>(pp, b, ch * kMeanChunk, kMeanChunk);
  __shared__ __attribute__((aligned(16))) float s_w[4][kD];
  __shared__ float s_mean[kD];
  __shared__ float s_red[4][4];
  __shared__ int s_last;
  float* s_part = reinterpret_cast<float*>(chunk_lds<kBytes>());

  // ---- 1. the chunk, and its column sums in the specified order -------------------------------
  // every load of the chunk goes out first (the rows stay in registers as 16-bit values until the end anyway): 16 KiB
  // per wave in flight; with the norm / rotation step each row is then worked on in place as it arrives
  uint4 raw[kChunkRowsPerSlot][2];
  float acc[16];
#pragma unroll
  for (int i = 0; i < kChunkRowsPerSlot; ++i) {
    const int row = ch * kMeanChunk + i * kSlots + slot;
    raw[i][0] = raw[i][1] = make_uint4(0, 0, 0, 0);
    if (row < L) {
      raw[i][0] = *reinterpret_cast<const uint4*>(base + (int64_t)row * sL);
      raw[i][1] = *reinterpret_cast<const uint4*>(base + (int64_t)row * sL + 8);
    }
  }
#pragma unroll
  for (int i = 0; i < kChunkRowsPerSlot; ++i) {
    const int row = ch * kMeanChunk + i * kSlots + slot;
    float x[16];
    widen8<DT>(raw[i][0], x);
    widen8<DT>(raw[i][1], x + 8);
    if constexpr (PRE) {
      if (row < L) prep16<DT, PRE, SOLO>(x, pp, rl, b, row, h, c16);
      raw[i][0] = narrow8<DT>(x);
      raw[i][1] = narrow8<DT>(x + 8);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = i == 0 ? x[e] : acc[e] + x[e];
  }
  forget_derived(raw);
  const float4 sums = over_slots16<Sum>(acc);
  if (!smooth) {  // uniform: nothing is taken off, nothing to wait for
    if (t < kD) {
      s_mean[t] = 0.0f;
      if (ch == 0) k_mean[bh * kD + t] = 0.0f;
    }
    __syncthreads();
  } else {
  store_slots16(sums, lane, s_w[wave]);
  __syncthreads();
  if constexpr (SOLO) {
    if (t < kD) {
      const float mean = round_to_half_dtype(__fdiv_rn((s_w[0][t] + s_w[1][t]) + (s_w[2][t] + s_w[3][t]), (float)L_all), dtype);
      s_mean[t] = mean;
      k_mean[bh * kD + t] = mean;
    }
    __syncthreads();
  } else {
  if (t < kD) {
    publish_f32(part + ((int64_t)bh * nch + ch) * kD + t, (s_w[0][t] + s_w[1][t]) + (s_w[2][t] + s_w[3][t]));
    complete_accesses();  // the partial result is visible chip-wide before this chunk is counted in
  }
  __syncthreads();
  // ---- 2. count the chunk in; the last one of the head publishes the mean -----------------------
  if (t == 0) {
    const int before = __hip_atomic_fetch_add(sy.counter + bh * kSyncStride, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = before == nch - 1;
    complete_accesses();
  }
  __syncthreads();
  if (s_last) {  // uniform
    const float* hp = part + (int64_t)bh * nch * kD;
    float tot = 0.0f;
    float nxt[kFinLoads];
    fetch_partials(hp, 0, nch, nxt);
    for (int c0 = 0; c0 < nch; c0 += kFinStage) {
      const int n = min(kFinStage, nch - c0);
      __syncthreads();  // the previous pass has been read
      stage_partials(nxt, s_part);
      if (c0 + kFinStage < nch) fetch_partials(hp, c0 + kFinStage, nch, nxt);
      __syncthreads();
      if (t < kD) {
        // chunk order is part of the specification
        if (n == kFinStage) {
#pragma unroll 16
          for (int c = 0; c < kFinStage; ++c) tot = (c0 == 0 && c == 0) ? s_part[t] : tot + s_part[c * kD + t];
        } else {
          for (int c = 0; c < n; ++c) tot = (c0 == 0 && c == 0) ? s_part[t] : tot + s_part[c * kD + t];
        }
      }
    }
    if (t < kD) {
      const float mean = round_to_half_dtype(__fdiv_rn(tot, (float)L_all), dtype);
      s_mean[t] = mean;
      publish_f32(k_mean + bh * kD + t, mean);
      complete_accesses();
    }
    __syncthreads();
    if (t == 0) __hip_atomic_store(sy.ready + bh * kSyncStride, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  } else {
    // ---- 3. everybody else waits for it -----------------------------------------------------------
    if (ch * (kMeanChunk / kBlkK) >= n_use) return;  // uniform
    if (!wait_for_head(sy.ready + bh * kSyncStride, sy)) {
      if (t < kD) s_mean[t] = load_shared_f32(k_mean + bh * kD + t);
      __syncthreads();
    } else {
      // Uniform, and not taken on a device this call has to itself: the head's mean from the input, every chunk
      // summed and the chunks added up exactly as steps 1 and 2 do it.  (Rotation factors come from the table in
      // global memory: the staged ones cover this workgroup's own rows.)
      float tot = 0.0f;
      for (int c = 0; c < nch; ++c) {
        float a16[16];
#pragma unroll 1
        for (int i = 0; i < kChunkRowsPerSlot; ++i) {
          const int row = c * kMeanChunk + i * kSlots + slot;
          uint4 r[2];
          fetch_row16(base + (int64_t)row * sL, row < L, r);
          float x[16];
          widen8<DT>(r[0], x);
          widen8<DT>(r[1], x + 8);
          if constexpr (PRE) {
            if (row < L) prep16<DT, PRE, SOLO>(x, pp, rl, b, row, h, c16, false);
          }
#pragma unroll
          for (int e = 0; e < 16; ++e) a16[e] = i == 0 ? x[e] : a16[e] + x[e];
        }
        const float4 part16 = over_slots16<Sum>(a16);
        __syncthreads();  // s_w of the chunk before has been read
        store_slots16(part16, lane, s_w[wave]);
        __syncthreads();
        if (t < kD) {
          const float pc = (s_w[0][t] + s_w[1][t]) + (s_w[2][t] + s_w[3][t]);
          tot = c == 0 ? pc : tot + pc;
        }
      }
      if (t < kD) s_mean[t] = round_to_half_dtype(__fdiv_rn(tot, (float)L_all), dtype);
      __syncthreads();
    }
  }
  }
  }
  // ---- 4. quantize the four 64-row tiles of the chunk from registers -----------------------------
#pragma unroll
  for (int tt = 0; tt < kMeanChunk / kBlkK; ++tt) {
    const int blk = ch * (kMeanChunk / kBlkK) + tt;
    if (blk >= n_use) break;  // uniform: the chunk's tail lies beyond the sequence
    float x[2][16];
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int row = blk * kBlkK + i * kSlots + slot;
      widen8<DT>(raw[2 * tt + i][0], x[i]);
      widen8<DT>(raw[2 * tt + i][1], x[i] + 8);
#pragma unroll
      for (int e = 0; e < 16; ++e) x[i][e] = row < L ? x[i][e] - s_mean[c16 * 16 + e] : 0.0f;
      fwht128(x[i], c16);
#pragma unroll
      for (int e = 0; e < 16; ++e) amax = fmaxf(amax, fabsf(x[i][e]));
    }
    amax = over_lanes<Max>(amax);
    if (lane == 0) s_red[tt][wave] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(s_red[tt][0], s_red[tt][1]), fmaxf(s_red[tt][2], s_red[tt][3]));
    const Int8Scale r = int8_scale(amax);
    const float inv_lane = r.inv * fwht_lane_sign(c16);  // the transform left this lane's values times that sign
    if (t == 0) k_scale[(int64_t)bh * nkb + blk] = r.scale;
    int8_t* tile = k_tiles + ((int64_t)bh * nkb + blk) * (int64_t)kTileBytes;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int frag = i * 4 + (c16 >> 1);
      const int ln = (c16 & 1) * 32 + slot;
      store_out16(tile + (frag * 64 + ln) * 16, pack_int8x16(x[i], inv_lane));
    }
  }
}

// With the Wan step folded in the kernel is asked to fit three waves per SIMD (168 registers; it spills ten of them):
// a workgroup idles while it waits for its head's mean, and with two workgroups per compute unit instead of three
// the kernel measured 23 % slower.
template <int DT, int PRE>
__global__ __launch_bounds__(kThreads, PRE == 1 ? 3 : 1) void quant_k_fused_kernel(const uint16_t* __restrict__ k, int64_t sB, int64_t sL,
                                                                 int64_t sH, int H, int L_all, int d_in, int nkb, int nch,
                                                                 float* __restrict__ part, float* k_mean, int dtype,
                                                                 int smooth, int8_t* __restrict__ k_tiles,
                                                                 float* __restrict__ k_scale, const PrepParams pp,
                                                                 const HeadSync sy) {
  const int bh = blockIdx.x / nch;
  quant_k_chunk<DT, PRE, false, kChunkLdsK>(bh, blockIdx.x - bh * nch, k, sB, sL, sH, H, L_all, d_in, nkb, nch, part, k_mean, dtype, smooth,
                                k_tiles, k_scale, pp, sy, nkb);
}

// V: column abs-max of the whole sequence (the last workgroup of a head to arrive takes the maximum over the
// chunks' maxima - no order to respect - and publishes the scales), then per-channel e4m3 in the transposed tile
// order of quant_v_kernel.
template <int DT, bool SOLO>
__device__ __forceinline__ void quant_v_chunk(int bh, int ch, const uint16_t* __restrict__ v, int64_t sB, int64_t sL,
                                              int64_t sH, int H, int L_all, int d_in, int nkb, int nch,
                                              float* __restrict__ part, float* v_scale, float* v_inv,
                                              float* __restrict__ v_mean, uint8_t* __restrict__ v_tiles, const HeadSync& sy,
                                              int n_use) {
  const int b = bh / H, h = bh - b * H;
  const int t = threadIdx.x, slot = t >> 3, c16 = t & 7;
  const int L = c16 * 16 < d_in ? L_all : 0;  // channels at or past d_in (head size 64) read as zero padding
  const int wave = t >> 6, lane = t & 63;
  const uint16_t* base = v + b * sB + h * sH + c16 * 16;
  __shared__ __attribute__((aligned(16))) float s_w[4][kD];
  __shared__ float s_inv[kD];
  __shared__ int s_last;
  constexpr int kStride = kD + 16;  // LDS row pitch in bytes
  uint8_t(*s_v)[kBlkK * kStride] = reinterpret_cast<uint8_t(*)[kBlkK * kStride]>(chunk_lds<kChunkLdsV>());

  uint4 raw[kChunkRowsPerSlot][2];
  float acc[16];
#pragma unroll
  for (int i = 0; i < kChunkRowsPerSlot; ++i) {
    const int row = ch * kMeanChunk + i * kSlots + slot;
    raw[i][0] = raw[i][1] = make_uint4(0, 0, 0, 0);
    if (row < L) {
      raw[i][0] = *reinterpret_cast<const uint4*>(base + (int64_t)row * sL);
      raw[i][1] = *reinterpret_cast<const uint4*>(base + (int64_t)row * sL + 8);
    }
    float x[16];
    widen8<DT>(raw[i][0], x);
    widen8<DT>(raw[i][1], x + 8);
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = i == 0 ? fabsf(x[e]) : fmaxf(acc[e], fabsf(x[e]));
  }
  forget_derived(raw);
  store_slots16(over_slots16<Max>(acc), lane, s_w[wave]);
  __syncthreads();
  if constexpr (SOLO) {
    if (t < kD) {
      const float amax = fmaxf(fmaxf(s_w[0][t], s_w[1][t]), fmaxf(s_w[2][t], s_w[3][t]));
      const bool nz = amax > 0.0f;
      const float inv = nz ? __fdiv_rn(448.0f, amax) : 0.0f;
      s_inv[t] = inv;
      v_inv[bh * kD + t] = inv;
      v_scale[bh * kD + t] = nz ? __fdiv_rn(amax, 448.0f) : 0.0f;
      v_mean[bh * kD + t] = 0.0f;
    }
    __syncthreads();
  } else {
  if (t < kD) {
    publish_f32(part + ((int64_t)bh * nch + ch) * kD + t, fmaxf(fmaxf(s_w[0][t], s_w[1][t]), fmaxf(s_w[2][t], s_w[3][t])));
    complete_accesses();  // visible chip-wide before this chunk is counted in
  }
  __syncthreads();
  if (t == 0) {
    const int before = __hip_atomic_fetch_add(sy.counter + bh * kSyncStride, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = before == nch - 1;
    complete_accesses();
  }
  __syncthreads();
  if (s_last) {  // uniform
    // thread t: channel t % 128, chunks of parity t / 128; 32 loads in flight at a time
    const float* hp = part + (int64_t)bh * nch * kD + (t & (kD - 1));
    float m = 0.0f;
    for (int c0 = t >> 7; c0 < nch; c0 += 64) {
      float v32[32];
#pragma unroll
      for (int j = 0; j < 32; ++j) v32[j] = c0 + 2 * j < nch ? load_shared_f32(hp + (int64_t)(c0 + 2 * j) * kD) : 0.0f;
#pragma unroll
      for (int j = 0; j < 32; ++j) m = fmaxf(m, v32[j]);
    }
    __syncthreads();  // s_w was read above by every thread that needed it
    s_w[t >> 7][t & (kD - 1)] = m;
    __syncthreads();
    if (t < kD) {
      const float amax = fmaxf(s_w[0][t], s_w[1][t]);
      const bool nz = amax > 0.0f;
      const float inv = nz ? __fdiv_rn(448.0f, amax) : 0.0f;
      s_inv[t] = inv;
      publish_f32(v_inv + bh * kD + t, inv);
      v_scale[bh * kD + t] = nz ? __fdiv_rn(amax, 448.0f) : 0.0f;
      v_mean[bh * kD + t] = 0.0f;
      complete_accesses();
    }
    __syncthreads();
    if (t == 0) __hip_atomic_store(sy.ready + bh * kSyncStride, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  } else {
    if (ch * (kMeanChunk / kBlkK) >= n_use) return;  // uniform
    if (!wait_for_head(sy.ready + bh * kSyncStride, sy)) {
      if (t < kD) s_inv[t] = load_shared_f32(v_inv + bh * kD + t);
      __syncthreads();
    } else {
      // Uniform, and not taken on a device this call has to itself: the head's column maxima from the input (a
      // maximum needs no order), and from them the factor the last workgroup would have published.
      float m16[16];
#pragma unroll
      for (int e = 0; e < 16; ++e) m16[e] = 0.0f;
      for (int row = slot; row < L; row += kSlots) {
        float x[16];
        widen8<DT>(*reinterpret_cast<const uint4*>(base + (int64_t)row * sL), x);
        widen8<DT>(*reinterpret_cast<const uint4*>(base + (int64_t)row * sL + 8), x + 8);
#pragma unroll
        for (int e = 0; e < 16; ++e) m16[e] = fmaxf(m16[e], fabsf(x[e]));
      }
      const float4 top16 = over_slots16<Max>(m16);
      __syncthreads();  // s_w of step 1 has been read
      store_slots16(top16, lane, s_w[wave]);
      __syncthreads();
      if (t < kD) {
        const float amax = fmaxf(fmaxf(s_w[0][t], s_w[1][t]), fmaxf(s_w[2][t], s_w[3][t]));
        s_inv[t] = amax > 0.0f ? __fdiv_rn(448.0f, amax) : 0.0f;
      }
      __syncthreads();
    }
  }
  }
  float inv[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) inv[e] = s_inv[c16 * 16 + e];
#pragma unroll
  for (int tt = 0; tt < kMeanChunk / kBlkK; ++tt) {
    const int blk = ch * (kMeanChunk / kBlkK) + tt;
    if (blk >= n_use) break;  // uniform
    uint8_t* sv = s_v[tt & 1];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = i * kSlots + slot;
      float x[16];
      widen8<DT>(raw[2 * tt + i][0], x);
      widen8<DT>(raw[2 * tt + i][1], x + 8);
      uint32_t w[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float y[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = fminf(fmaxf(x[4 * j + e] * inv[4 * j + e], -448.0f), 448.0f);
        int packed = 0;
        packed = __builtin_amdgcn_cvt_pk_fp8_f32(y[0], y[1], packed, false);
        packed = __builtin_amdgcn_cvt_pk_fp8_f32(y[2], y[3], packed, true);
        w[j] = (uint32_t)packed;
      }
      *reinterpret_cast<uint4*>(&sv[r * kStride + c16 * 16]) = make_uint4(w[0], w[1], w[2], w[3]);
    }
    __syncthreads();  // two staging buffers: the one written two tiles ago was read before the last barrier
    uint8_t* tile = v_tiles + ((int64_t)bh * nkb + blk) * (int64_t)kTileBytes;
#pragma unroll
    for (int i = 0; i < kTileBytes / 16 / kThreads; ++i) {
      const int oc = i * kThreads + t;
      const int dt = oc >> 7, th = (oc >> 6) & 1, ln = oc & 63;
      const int hh = ln >> 5, d = dt * 32 + (ln & 31);
      uint32_t w[4];
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        uint32_t a = 0;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const int row = 32 * th + 8 * g + 4 * hh + c;
          a |= (uint32_t)sv[row * kStride + d] << (8 * c);
        }
        w[g] = a;
      }
      store_out16(tile + oc * 16, make_uint4(w[0], w[1], w[2], w[3]));
    }
  }
}

template <int DT>
__global__ __launch_bounds__(kThreads) void quant_v_fused_kernel(const uint16_t* __restrict__ v, int64_t sB, int64_t sL,
                                                                 int64_t sH, int H, int L_all, int d_in, int nkb, int nch,
                                                                 float* __restrict__ part, float* v_scale, float* v_inv,
                                                                 float* __restrict__ v_mean,
                                                                 uint8_t* __restrict__ v_tiles, const HeadSync sy) {
  const int bh = blockIdx.x / nch;
  quant_v_chunk<DT, false>(bh, blockIdx.x - bh * nch, v, sB, sL, sH, H, L_all, d_in, nkb, nch, part, v_scale, v_inv, v_mean, v_tiles,
                           sy, nkb);
}

// K with a step folded in and V in one launch: a head's V chunks are neighbours of its K chunks.  What that saves is a launch;
// the two do not run faster together (see kv_in_one_launch_pays).
template <int DT, int PRE>
__global__ __launch_bounds__(kThreads, 3) void quant_kv_meet_kernel(const QkvCall c, const PrepParams pp, const HeadSync sk, const HeadSync sv) {
  const int bh = blockIdx.x / (2 * c.nch), item = blockIdx.x - bh * 2 * c.nch;
  if (item < c.nch)
    quant_k_chunk<DT, PRE, false>(bh, item, c.k.ptr, c.k.sB, c.k.sL, c.k.sH, c.Hkv, c.Lk, c.k.D, c.nkb, c.nch, c.k_part, c.k_mean,
                                  c.k.dtype, c.smooth_k, c.k_tiles, c.k_scale, pp, sk, c.nkb);
  else
    quant_v_chunk<DT, false>(bh, item - c.nch, c.v.ptr, c.v.sB, c.v.sL, c.v.sH, c.Hkv, c.Lk, c.v.D, c.nkb, c.nch, c.v_part, c.v_scale,
                             c.v_inv, c.v_mean, c.v_tiles, sv, c.nkb);
}

// ---------------------------------------------------------------------------------------
// Q, K and V of one call together, in one or two launches.
//
// Separate quantizers are six launches, and below a few thousand tokens each of them is bound by being one: 4-5 us from
// the end of a kernel to the end of the next however little the next does.  Three forms (launch_quant_qkv picks):
//
//   small    at most 256 keys, one chunk per head: the K and V workgroups hold their whole head, one launch does all.
//   stages   stage 1 takes the chunk sums of K, the chunk maxima of V and quantizes Q; stage 2 quantizes K and V, every
//            workgroup forming its head's statistic from the chunks' by itself (the same operations in the same order as
//            the finalisation kernels).  Stage 2 reads its inputs a second time - out of the caches while K and V fit
//            them - and nch * 512 bytes of partial results per workgroup.
//   meet     one launch, every input read once: K's and V's chunks meet per head as in the one-read kernels above.  Calls
//            with a step folded in do not take it (see launch_qkv_kind).
//
// Measured, all quantizer launches of a call, us (separate quantizers / this):  B=2, 64 heads, 32 tokens 27 / 8 small;
// 40 heads, 1560 tokens 43 / 22 stages; 9000 tokens 120 / 106 stages; 14000 tokens 184 / 158 meet; 32760 tokens 392 / 369
// meet (HBM-bound: 9 bytes per element at 4 TB/s).
// ---------------------------------------------------------------------------------------
// channel d's mean of a head of K
__device__ __forceinline__ float head_mean(const QkvCall& c, int bh, int d, bool publish) {
  const float* hp = c.k_part + (int64_t)bh * c.nch * kD + d;
  float tot = 0.0f;
  if (c.smooth_k) {
    for (int c0 = 0; c0 < c.nch; c0 += 16) {  // 16 loads in flight; added in chunk order
      float v[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) v[j] = hp[min(c0 + j, c.nch - 1) * kD];
#pragma unroll
      for (int j = 0; j < 16; ++j)
        if (c0 + j < c.nch) tot = c0 + j == 0 ? v[0] : tot + v[j];
    }
  }
  const float mean = c.smooth_k ? round_to_half_dtype(__fdiv_rn(tot, (float)c.Lk), c.k.dtype) : 0.0f;
  if (publish) c.k_mean[bh * kD + d] = mean;
  return mean;
}

template <int OP>  // 0: K's mean (ordered sum), 1: V's factor 448 / amax
__device__ __forceinline__ void head_statistic(const QkvCall& c, int bh, bool publish, float (*s_stat)[kD]) {
  const int t = threadIdx.x, d = t & (kD - 1);
  const float* hp = (OP == 0 ? c.k_part : c.v_part) + (int64_t)bh * c.nch * kD + d;
  if constexpr (OP == 0) {
    if (t < kD) s_stat[0][d] = head_mean(c, bh, d, publish);
    __syncthreads();
  } else {
    float m = 0.0f;  // a maximum needs no order: the two halves of the workgroup take the even and the odd chunks
    for (int c0 = t >> 7; c0 < c.nch; c0 += 32) {
      float v[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) v[j] = hp[min(c0 + 2 * j, c.nch - 1) * kD];
#pragma unroll
      for (int j = 0; j < 16; ++j) m = fmaxf(m, v[j]);  // (a chunk taken twice changes no maximum)
    }
    s_stat[t >> 7][d] = m;
    __syncthreads();
    const float amax = fmaxf(s_stat[0][d], s_stat[1][d]);
    const bool nz = amax > 0.0f;
    const float inv = nz ? __fdiv_rn(448.0f, amax) : 0.0f;
    __syncthreads();
    if (t < kD) {
      s_stat[0][d] = inv;
      if (publish) {
        c.v_inv[bh * kD + d] = inv;
        c.v_scale[bh * kD + d] = nz ? __fdiv_rn(amax, 448.0f) : 0.0f;
        c.v_mean[bh * kD + d] = 0.0f;  // the attention adds whatever the slot holds
      }
    }
    __syncthreads();
  }
}

// (this form has no wait that could expire)
__device__ __forceinline__ void clear_status(const QkvCall& c) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *c.sync.k_status = 0, *c.sync.v_status = 0;
}

// Key tiles of a batch entry that anybody reads.  The others' second reading and their codes are left out (us per call, entries
// falling off to 45 %: 6 x 24 heads of 520 rows on 10561 keys 456 / 420, of 16 of 1111 on 4311 190 / 178, 3 x 24 of 3001 on
// 4099 195.4 / 193.1); their statistics are not, so the codes that are read stay the same.
__device__ __forceinline__ int tiles_in_use(const QkvCall& c, int b) {
  return c.k_lens == nullptr ? c.nkb : tiles_counted(c.k_lens[b], c.nkb);
}

template <int DT, int KIND>
__device__ __forceinline__ void quant_q_item(int item, const QkvCall& c, const PrepParams& pp) {
  const int bh = item / c.nqb;
  if (c.q_lens != nullptr && (item - bh * c.nqb) * kQPad >= c.q_lens[bh / c.Hq]) return;  // (uniform) no row of it takes part
  quant_q_block<DT, KIND, false>(item - bh * c.nqb, bh % c.Hq, bh / c.Hq, c.q.ptr, c.q.sB, c.q.sL, c.q.sH, c.Hq, c.Lq, c.q.D, c.lq_pad,
                                 c.premul, c.q_i8, c.q_scale, pp, nullptr);
}

// The joint block's items take several heads of the same rows: a lane's norm weights and rotation factors are read once for all of
// them (a row's factors are twice its own bytes, and came out of the L2 for every head).  Bound by vector work, 54-62 % busy:
// 2 x 4352 tokens of 24 heads, stage 1 70 -> 61 us, stage 2 47 -> 45.
constexpr int kJointHeadsQ = 4, kJointHeadsK = 2;

// 32 query rows of kJointHeadsQ heads
template <int DT>
__device__ __forceinline__ void joint_q_item(int item, const QkvCall& c, const PrepParams& pp) {
  const int t = threadIdx.x, slot = t >> 3, c16 = t & 7;
  const int blocks = c.lq_pad / kSlots, groups = (c.Hq + kJointHeadsQ - 1) / kJointHeadsQ;
  const int bg = item / blocks, row = (item - bg * blocks) * kSlots + slot, b = bg / groups, h0 = (bg - b * groups) * kJointHeadsQ;
  const bool valid = row < c.Lq;
  const uint16_t* base = c.q.ptr + b * c.q.sB + (int64_t)row * c.q.sL + c16 * 16;
  const int n = min(kJointHeadsQ, c.Hq - h0);
  uint4 next[2];
  fetch_row16(base + h0 * c.q.sH, valid, next);
  QwenRow f{};
  if (valid) qwen_row(f, pp, row, c16);
  const float premul_lane = c.premul * fwht_lane_sign(c16);
#pragma unroll 1  // (unrolled, the heads' work is pulled together and spills)
  for (int i = 0; i < n; ++i) {
    float x[16];
    widen8<DT>(next[0], x);
    widen8<DT>(next[1], x + 8);
    if (i + 1 < n) fetch_row16(base + (h0 + i + 1) * c.q.sH, valid, next);
    if (valid) prep16_qwen<DT, true>(x, f, pp.eps);
    const int64_t at = ((int64_t)b * c.Hq + h0 + i) * c.lq_pad + row;
    quant_q_row(x, c16, premul_lane, c.q_scale + at, c.q_i8 + at * kD);
  }
}

// the column sums of one chunk of K for kJointHeadsK heads, in the order of col_partial_chunk
template <int DT>
__device__ __forceinline__ void joint_k_sums(int item, const QkvCall& c, const PrepParams& pp) {
  const int t = threadIdx.x, slot = t >> 3, c16 = t & 7;
  const int groups = (c.Hkv + kJointHeadsK - 1) / kJointHeadsK;
  const int bg = item / c.nch, ch = item - bg * c.nch, b = bg / groups, h0 = (bg - b * groups) * kJointHeadsK;
  const uint16_t* base = c.k.ptr + b * c.k.sB + h0 * c.k.sH + c16 * 16;
  float acc[kJointHeadsK][16];
  uint4 next[kJointHeadsK][2];
  auto fetch = [&](int i) {
    const int row = ch * kMeanChunk + i * kSlots + slot;
#pragma unroll
    for (int hh = 0; hh < kJointHeadsK; ++hh) {
      next[hh][0] = next[hh][1] = make_uint4(0, 0, 0, 0);
      if (h0 + hh < c.Hkv) fetch_row16(base + (int64_t)row * c.k.sL + hh * c.k.sH, row < c.Lk, next[hh]);
    }
  };
  auto add_row = [&](int i, bool first) {
    const int row = ch * kMeanChunk + i * kSlots + slot;
    uint4 raw[kJointHeadsK][2];
#pragma unroll
    for (int hh = 0; hh < kJointHeadsK; ++hh) raw[hh][0] = next[hh][0], raw[hh][1] = next[hh][1];
    QwenRow f{};
    if (row < c.Lk) qwen_row(f, pp, row, c16);
    if (i + 1 < kMeanChunk / kSlots) fetch(i + 1);
#pragma unroll
    for (int hh = 0; hh < kJointHeadsK; ++hh) {
      float x[16];
      widen8<DT>(raw[hh][0], x);
      widen8<DT>(raw[hh][1], x + 8);
      if (row < c.Lk) prep16_qwen<DT, true>(x, f, pp.eps);
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[hh][e] = first ? x[e] : acc[hh][e] + x[e];
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  fetch(0);
  add_row(0, true);
#pragma unroll 1  // (unrolled, the rows' work is pulled together and spills)
  for (int i = 1; i < kMeanChunk / kSlots; ++i) add_row(i, false);
  __shared__ __attribute__((aligned(16))) float s_w[kJointHeadsK][4][kD];
  const int wave = t >> 6, lane = t & 63;
#pragma unroll
  for (int hh = 0; hh < kJointHeadsK; ++hh) {
    store_slots16(over_slots16<Sum>(acc[hh]), lane, s_w[hh][wave]);
  }
  __syncthreads();
  static_assert(kJointHeadsK * kD == kThreads, "a thread per head and channel");
  const int hh = t >> 7, d = t & (kD - 1);
  if (h0 + hh < c.Hkv)
    c.k_part[(((int64_t)b * c.Hkv + h0 + hh) * c.nch + ch) * kD + d] =
        (s_w[hh][0][d] + s_w[hh][1][d]) + (s_w[hh][2][d] + s_w[hh][3][d]);
}

// one tile of K for kJointHeadsK heads; the heads' means from the chunk sums
template <int DT>
__device__ __forceinline__ void joint_k_item(int item, const QkvCall& c, const PrepParams& pp) {
  const int t = threadIdx.x, slot = t >> 3, c16 = t & 7;
  const int groups = (c.Hkv + kJointHeadsK - 1) / kJointHeadsK;
  const int bg = item / c.nkb, blk = item - bg * c.nkb, b = bg / groups, h0 = (bg - b * groups) * kJointHeadsK;
  const uint16_t* base = c.k.ptr + b * c.k.sB + h0 * c.k.sH + c16 * 16;
  __shared__ float s_mean[kJointHeadsK][kD];
  __shared__ float s_red[kJointHeadsK][4];
  constexpr int R = kBlkK / kSlots;
  uint4 next[R][2];
  QwenRow f[R]{};
  auto fetch = [&](int hh) {
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int row = blk * kBlkK + i * kSlots + slot;
      fetch_row16(base + (int64_t)row * c.k.sL + hh * c.k.sH, row < c.Lk, next[i]);
    }
  };
  fetch(0);
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int row = blk * kBlkK + i * kSlots + slot;
    if (row < c.Lk) qwen_row(f[i], pp, row, c16);
  }
  {
    const int hh = t >> 7, d = t & (kD - 1), bh = b * c.Hkv + h0 + hh;
    if (h0 + hh < c.Hkv) s_mean[hh][d] = head_mean(c, bh, d, blk == 0);
  }
  __syncthreads();
  const int wave = t >> 6;
  const int n = min(kJointHeadsK, c.Hkv - h0);
#pragma unroll 1
  for (int hh = 0; hh < n; ++hh) {
    float x[R][16], amax = 0.0f;
#pragma unroll
    for (int i = 0; i < R; ++i) {
      widen8<DT>(next[i][0], x[i]);
      widen8<DT>(next[i][1], x[i] + 8);
    }
    if (hh + 1 < n) fetch(hh + 1);
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const bool valid = blk * kBlkK + i * kSlots + slot < c.Lk;
      if (valid) {  // (a row that is not there has been read as zeros and stays so)
        prep16_qwen<DT, true>(x[i], f[i], pp.eps);
#pragma unroll
        for (int e = 0; e < 16; ++e) x[i][e] = x[i][e] - s_mean[hh][c16 * 16 + e];
      }
      fwht128(x[i], c16);
#pragma unroll
      for (int e = 0; e < 16; ++e) amax = fmaxf(amax, fabsf(x[i][e]));
      __builtin_amdgcn_sched_barrier(0);
    }
    amax = over_lanes<Max>(amax);
    if ((t & 63) == 0) s_red[hh][wave] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(s_red[hh][0], s_red[hh][1]), fmaxf(s_red[hh][2], s_red[hh][3]));
    const Int8Scale r = int8_scale(amax);
    const float inv_lane = r.inv * fwht_lane_sign(c16);
    const int64_t at = ((int64_t)b * c.Hkv + h0 + hh) * c.nkb + blk;
    if (t == 0) c.k_scale[at] = r.scale;
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int frag = i * 4 + (c16 >> 1), ln = (c16 & 1) * 32 + slot;
      store_out16(c.k_tiles + at * kTileBytes + (frag * 64 + ln) * 16, pack_int8x16(x[i], inv_lane));
    }
  }
}

// kHeads: the joint block's step with several heads per item (launch_qkv_kind)
template <int DT, int KIND, bool kHeads>
__global__ __launch_bounds__(kThreads, KIND == 0 ? 5 : 4) void quant_qkv_stage1_kernel(const QkvCall c, const PrepParams pq, const PrepParams pk) {
  want(c.q.ptr, c.v.ptr, c.B, c.k_part, c.v_tiles);
  clear_status(c);
  const int more = KIND == 0 ? numbers_batch(c.numbers) : 0;
  if ((int)blockIdx.x < more) return number_batch(c.numbers);
  const int n_v = c.B * c.Hkv * c.nch;
  const int n_k = !c.smooth_k ? 0 : (!kHeads ? n_v : c.B * ((c.Hkv + kJointHeadsK - 1) / kJointHeadsK) * c.nch);
  int item = blockIdx.x - more;
  if (item < n_k) {
    if constexpr (kHeads) {
      joint_k_sums<DT>(item, c, pk);
    } else {
      const int bh = item / c.nch;
      col_partial_chunk<DT, 0, KIND>(item - bh * c.nch, bh % c.Hkv, bh / c.Hkv, c.k.ptr, c.k.sB, c.k.sL, c.k.sH, c.Hkv, c.Lk, c.k.D, c.k_part,
                                  c.nch, pk, nullptr);
    }
    return;
  }
  item -= n_k;
  if (item < n_v) {
    const int bh = item / c.nch;
    col_partial_chunk<DT, 1, 0>(item - bh * c.nch, bh % c.Hkv, bh / c.Hkv, c.v.ptr, c.v.sB, c.v.sL, c.v.sH, c.Hkv, c.Lk, c.v.D, c.v_part,
                                c.nch, pk, nullptr);
    return;
  }
  if constexpr (kHeads)
    joint_q_item<DT>(item - n_v, c, pq);
  else
    quant_q_item<DT, KIND>(item - n_v, c, pq);
}

template <int DT, int KIND, bool kHeads>
__global__ __launch_bounds__(kThreads, KIND == 0 ? 6 : (kHeads ? 4 : 5)) void quant_qkv_stage2_kernel(const QkvCall c, const PrepParams pk) {
  want(c.q.ptr, c.v.ptr, c.B, c.k_part, c.v_tiles);
  __shared__ float s_stat[2][kD];
  const int per_head = (c.nkb + c.tiles_per_wg - 1) / c.tiles_per_wg, n = c.B * c.Hkv * per_head;
  const int n_k = !kHeads ? n : c.B * ((c.Hkv + kJointHeadsK - 1) / kJointHeadsK) * c.nkb;
  const bool is_v = (int)blockIdx.x >= n_k;
  if constexpr (kHeads) {
    if (!is_v) {
      joint_k_item<DT>(blockIdx.x, c, pk);
      return;
    }
  }
  const int item = is_v ? blockIdx.x - n_k : blockIdx.x;
  const int bh = item / per_head, run = item - bh * per_head, b = bh / c.Hkv, h = bh - b * c.Hkv;
  const int first = run * c.tiles_per_wg, last = min(tiles_in_use(c, b), first + c.tiles_per_wg);
  if (first >= last && run != 0) return;  // (uniform) keys that take no part; the head's first workgroup stores its statistics
  auto stat = [&]() -> const float* { return s_stat[0]; };
  if (is_v) {
    head_statistic<1>(c, bh, run == 0, s_stat);
    for (int blk = first; blk < last; ++blk) {
      quant_v_block<DT, false>(blk, h, b, c.v.ptr, c.v.sB, c.v.sL, c.v.sH, c.Hkv, c.Lk, c.v.D, c.nkb, stat, nullptr, c.v_tiles);
      __syncthreads();  // the tile has been read out of LDS
    }
  } else {
    head_statistic<0>(c, bh, run == 0, s_stat);
    for (int blk = first; blk < last; ++blk) {
      quant_k_block<DT, KIND, false>(blk, h, b, c.k.ptr, c.k.sB, c.k.sL, c.k.sH, c.Hkv, c.Lk, c.k.D, c.nkb, stat, c.k_tiles, c.k_scale,
                                     pk, nullptr);
      __syncthreads();
    }
  }
}

// One launch over inputs that are read once: the chunks of K and V meet per head as in the one-read kernels above, and
// the items of a head - its K chunks, its V chunks, the Q blocks of its query heads - are neighbours in the grid, so the
// Q blocks (which wait for nobody) and the V chunks work while K's chunks wait for their mean.
template <int DT>
__global__ __launch_bounds__(kThreads, 4) void quant_qkv_meet_kernel(const QkvCall c, const HeadSync sk, const HeadSync sv) {
  const int more = numbers_batch(c.numbers);
  if ((int)blockIdx.x < more) return number_batch(c.numbers);
  const PrepParams none{};
  const int group = c.Hq / c.Hkv, per_head = 2 * c.nch + group * c.nqb;
  const int block = blockIdx.x - more, bh = block / per_head;
  int item = block - bh * per_head;
  if (item < c.nch) {
    quant_k_chunk<DT, 0, false>(bh, item, c.k.ptr, c.k.sB, c.k.sL, c.k.sH, c.Hkv, c.Lk, c.k.D, c.nkb, c.nch, c.k_part, c.k_mean,
                                c.k.dtype, c.smooth_k, c.k_tiles, c.k_scale, none, sk, tiles_in_use(c, bh / c.Hkv));
    return;
  }
  item -= c.nch;
  if (item < c.nch) {
    quant_v_chunk<DT, false>(bh, item, c.v.ptr, c.v.sB, c.v.sL, c.v.sH, c.Hkv, c.Lk, c.v.D, c.nkb, c.nch, c.v_part, c.v_scale, c.v_inv,
                             c.v_mean, c.v_tiles, sv, tiles_in_use(c, bh / c.Hkv));
    return;
  }
  item -= c.nch;
  const int b = bh / c.Hkv, hk = bh - b * c.Hkv;
  const int hq = hk * group + item / c.nqb;
  quant_q_item<DT, 0>((b * c.Hq + hq) * c.nqb + item % c.nqb, c, none);
}

// at most 256 keys: one launch
// (The joint step's K chunk holds its rows in 163 registers.  With the 128 that four workgroups a unit have, up to 69 went through
// memory, how many depending on the kernel's arguments; three a unit are enough for the grids of this launch.  us per call of 24 heads,
// four / three: 84 tokens 20.0 / 17.4, 256 30.6 / 27.6, 4 x 256 35.8 / 31.5; beside the four with 50 in memory 8 x 120 27.1 / 21.9, 8 x 256
// 44.0 / 39.3, 12 x 256 53.7 / 46.6, 16 x 256, four rounds in place of three, 57.3 / 56.9, 24 x 256 79.9 / 78.9.)
template <int DT, int KIND>
__global__ __launch_bounds__(kThreads, KIND == 2 ? 3 : 4) void quant_qkv_small_kernel(const QkvCall c, const PrepParams pq, const PrepParams pk) {
  want(c.q.ptr, c.v.ptr, c.B, c.k_part, c.v_tiles);
  clear_status(c);
  const int more = KIND == 0 ? numbers_batch(c.numbers) : 0;
  if ((int)blockIdx.x < more) return number_batch(c.numbers);
  const int n = c.B * c.Hkv;
  const int item = blockIdx.x - more;
  const HeadSync nobody{};
  if (item < n)
    quant_k_chunk<DT, KIND, true>(item, 0, c.k.ptr, c.k.sB, c.k.sL, c.k.sH, c.Hkv, c.Lk, c.k.D, c.nkb, 1, c.k_part, c.k_mean, c.k.dtype,
                                  c.smooth_k, c.k_tiles, c.k_scale, pk, nobody, tiles_in_use(c, item / c.Hkv));
  else if (item < 2 * n)
    quant_v_chunk<DT, true>(item - n, 0, c.v.ptr, c.v.sB, c.v.sL, c.v.sH, c.Hkv, c.Lk, c.v.D, c.nkb, 1, c.v_part, c.v_scale, c.v_inv,
                            c.v_mean, c.v_tiles, nobody, tiles_in_use(c, (item - n) / c.Hkv));
  else
    quant_q_item<DT, KIND>(item - 2 * n, c, pq);
}

// The sparse-linear backend's second launch: the statistics have come with the linear branch's pass over K and V, so K and V are
// quantized (from the last head down: what that pass read last is read first), Q with them, the block averages of Q and K
// are taken along, and the linear branch's matrices are finished.  With the first launch it replaces seven (Q, K's sums, their
// finalisation, K, V with its counters, the linear branch's finalisation) and a third reading of K and a second of V: HBM-bound.
// kReady: a launch in between (sla_finalize_kernel) has finished the heads' statistics and the linear branch's matrices - from
// kSlaReadyChunks on, where the chunk results every workgroup would add up are no longer small next to its rows.
template <int DT, bool kReady>
__global__ __launch_bounds__(kThreads, 4) void quant_sla_kernel(const QkvCall c, const SlaFinal f) {
  __shared__ float s_stat[2][kD];
  int item = blockIdx.x;
  const int n_bh = c.B * c.Hkv;
  if constexpr (!kReady) {
    clear_status(c);
    const int n_fin = n_bh * (kD / kFinRows);
    if (item < n_fin) {
      sla_kv_finalize<DT>(item % (kD / kFinRows), item / (kD / kFinRows), f.part, f.runs, f.proj_w, f.m_frag, f.ksum);
      return;
    }
    item -= n_fin;
  }
  const int per_head = (c.nkb + c.tiles_per_wg - 1) / c.tiles_per_wg;
  if (item < 2 * n_bh * per_head) {
    const int up = item / (2 * per_head), bh = n_bh - 1 - up, b = bh / c.Hkv, h = bh - b * c.Hkv;
    int run = item - up * (2 * per_head);
    const bool is_v = run >= per_head;
    if (is_v) run -= per_head;
    const int first = run * c.tiles_per_wg, last = min(c.nkb, first + c.tiles_per_wg);
    auto stat = [&]() -> const float* { return kReady ? (is_v ? c.v_inv : c.k_mean) + bh * kD : s_stat[0]; };
    const PrepParams none{};
    if (is_v) {
      if constexpr (!kReady) head_statistic<1>(c, bh, run == 0, s_stat);
      for (int blk = first; blk < last; ++blk) {
        quant_v_block<DT, false>(blk, h, b, c.v.ptr, c.v.sB, c.v.sL, c.v.sH, c.Hkv, c.Lk, c.v.D, c.nkb, stat, nullptr, c.v_tiles);
        __syncthreads();  // the tile has been read out of LDS
      }
    } else {
      if constexpr (!kReady) head_statistic<0>(c, bh, run == 0, s_stat);
      for (int blk = first; blk < last; ++blk) {
        quant_k_block<DT, 0, true>(blk, h, b, c.k.ptr, c.k.sB, c.k.sL, c.k.sH, c.Hkv, c.Lk, c.k.D, c.nkb, stat, c.k_tiles, c.k_scale,
                                   none, f.pooled_k);
        __syncthreads();
      }
    }
    return;
  }
  item -= 2 * n_bh * per_head;
  const PrepParams none{};
  const int bh = item / c.nqb;
  quant_q_block<DT, 0, true>(item - bh * c.nqb, bh % c.Hq, bh / c.Hq, c.q.ptr, c.q.sB, c.q.sL, c.q.sH, c.Hq, c.Lq, c.q.D, c.lq_pad,
                             c.premul, c.q_i8, c.q_scale, none, f.pooled_q);
}

// the heads' statistics and the linear branch's matrices: grid = B * H * (8 + 2)
template <int DT>
__global__ __launch_bounds__(kThreads) void sla_finalize_kernel(const QkvCall c, const SlaFinal f) {
  __shared__ float s_stat[2][kD];
  clear_status(c);
  const int n_bh = c.B * c.Hkv, n_fin = n_bh * (kD / kFinRows), item = blockIdx.x;
  if (item < n_bh)
    head_statistic<0>(c, item, true, s_stat);
  else if (item < 2 * n_bh)
    head_statistic<1>(c, item - n_bh, true, s_stat);
  else if (item < 2 * n_bh + n_fin)
    sla_kv_finalize<DT>((item - 2 * n_bh) % (kD / kFinRows), (item - 2 * n_bh) / (kD / kFinRows), f.part, f.runs, f.proj_w, f.m_frag, f.ksum);
}

// ---------------------------------------------------------------------------------------
// Block means: out[b, h, blk, d] = mean over the rows [blk * rows, min((blk + 1) * rows, L)) of x[b, :, h, d],
// optionally of x - centre[b, h, d] with each difference rounded to the tensor's half type first (the reference
// forms `k - mean(k)` as a half tensor before it pools it).  fp32 sum in a frozen order - row r of the block goes to
// slot r % 32, a slot adds its rows in increasing order, the 32 slots meet in an adjacent-pair tree - divided by the
// number of rows that exist and rounded to the half type.  One workgroup per block; rows <= 256, a multiple of 32.
// grid = (nblk, H, B).
// ---------------------------------------------------------------------------------------
template <int DT>
__global__ __launch_bounds__(kThreads) void block_mean_kernel(const uint16_t* __restrict__ x, int64_t sB, int64_t sL,
                                                              int64_t sH, int H, int L, int rows,
                                                              const float* __restrict__ centre,
                                                              uint16_t* __restrict__ out) {
  const int blk = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int t = threadIdx.x, slot = t >> 3, c16 = t & 7;
  const uint16_t* base = x + b * sB + h * sH + c16 * 16;
  const int64_t bh = (int64_t)b * H + h;
  float cen[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) cen[e] = centre != nullptr ? centre[bh * kD + c16 * 16 + e] : 0.0f;
  float acc[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[e] = 0.0f;
  for (int i = 0; i < rows / kSlots; ++i) {
    const int row = blk * rows + i * kSlots + slot;
    float v[16];
    load_row16<DT>(base + (int64_t)row * sL, row < L, v);
    if (centre != nullptr && row < L) {
#pragma unroll
      for (int e = 0; e < 16; ++e) v[e] = through_half<DT>(v[e] - cen[e]);
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = i == 0 ? v[e] : acc[e] + v[e];
  }
  __shared__ __attribute__((aligned(16))) float s_w[4][kD];
  store_block_mean<DT>(acc, t, (float)min(rows, L - blk * rows), out + (bh * gridDim.x + blk) * kD, s_w);
}

__global__ void clear_ints_kernel(int* p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

}  // namespace

#define KSANA_DISPATCH_DT(dtype, ...)            \
  do {                                           \
    if ((dtype) == KSANA_SAGE_BF16) {            \
      constexpr int DT = KSANA_SAGE_BF16;        \
      __VA_ARGS__;                               \
    } else {                                     \
      constexpr int DT = KSANA_SAGE_FP16;        \
      __VA_ARGS__;                               \
    }                                            \
  } while (0)

// KIND as a compile-time constant for the three variants of the folded step (PrepParams::kind)
#define KSANA_DISPATCH_KIND(kind, ...)  \
  do {                                  \
    if ((kind) == 1) {                  \
      constexpr int KIND = 1;           \
      __VA_ARGS__;                      \
    } else if ((kind) == 2) {           \
      constexpr int KIND = 2;           \
      __VA_ARGS__;                      \
    } else {                            \
      constexpr int KIND = 3;           \
      __VA_ARGS__;                      \
    }                                   \
  } while (0)

// Sizes the LDS copy of the rotation factors for kernels that give `rows_per_wg` consecutive rows to
// a workgroup; returns the dynamic LDS bytes (0: the kernel reads the table directly).
static size_t plan_rope_lds(PrepParams* pp, int B, int rows_per_wg) {
  pp->lds_frames = pp->lds_heights = pp->lds_widths = 0;
  if (pp->kind == 2 || pp->freqs == nullptr) return 0;
  int nf = 0, nh = 0, nw = 0;
  for (int b = 0; b < B; ++b) {
    const int gh = pp->grid[b][1], gw = pp->grid[b][2];
    nf = max(nf, (rows_per_wg - 1) / (gh * gw) + 2);
    nh = max(nh, (rows_per_wg - 1) / gw + 2);
    nw = max(nw, gw);
  }
  const size_t bytes = ((size_t)nf * kRopeN0 + (size_t)nh * kRopeN1 + (size_t)nw * kRopeN2) * sizeof(double2);
  if (bytes > 48 * 1024) return 0;  // unusual grids (very wide, or planes of a few tokens): direct reads
  pp->lds_frames = nf, pp->lds_heights = nh, pp->lds_widths = nw;
  return bytes;
}

hipError_t launch_row_inv_rms(const InTensor& x, int B, int H, int L, float eps, float* inv_rms, hipStream_t s) {
  const dim3 grid((L + 3) / 4, B), block(kThreads);
  KSANA_DISPATCH_DT(x.dtype, (row_inv_rms_kernel<DT><<<grid, block, 0, s>>>(x.ptr, x.sB, x.sL, L, H * kD / 8,
                                                                            (float)(H * kD), eps, inv_rms)));
  return hipGetLastError();
}

hipError_t launch_col_partial(const InTensor& x, int B, int H, int L, int op, float* part, int nch, hipStream_t s,
                              const PrepParams* prep, const float* centre) {
  const dim3 grid(nch, H, B), block(kThreads);
  const PrepParams none{};
  KSANA_DISPATCH_DT(x.dtype, {
    if (op == 2)
      col_partial_kernel<DT, 2, 0><<<grid, block, 0, s>>>(x.ptr, x.sB, x.sL, x.sH, H, L, x.D, part, nch, none, centre);
    else if (op == 1)
      col_partial_kernel<DT, 1, 0><<<grid, block, 0, s>>>(x.ptr, x.sB, x.sL, x.sH, H, L, x.D, part, nch, none, nullptr);
    else if (prep == nullptr)
      col_partial_kernel<DT, 0, 0><<<grid, block, 0, s>>>(x.ptr, x.sB, x.sL, x.sH, H, L, x.D, part, nch, none, nullptr);
    else {
      PrepParams pp = *prep;
      const size_t lds = plan_rope_lds(&pp, B, kMeanChunk);
      KSANA_DISPATCH_KIND(pp.kind, (col_partial_kernel<DT, 0, KIND><<<grid, block, lds, s>>>(x.ptr, x.sB, x.sL, x.sH, H, L, x.D, part,
                                                                                        nch, pp, nullptr)));
    }
  });
  return hipGetLastError();
}

hipError_t launch_k_mean_finalize(const float* part, int BH, int nch, int L, int dtype, int smooth, float* k_mean,
                                  hipStream_t s, int* status, const BatchNumbers& numbers) {
  k_mean_finalize_kernel<<<dim3(BH + numbers_batch(numbers)), dim3(kFinThreads), 0, s>>>(part, nch, L, dtype, smooth, k_mean, status, numbers);
  return hipGetLastError();
}

hipError_t launch_v_scale_finalize(const float* part, int BH, int nch, float* v_scale, float* v_inv, float* zero_mean,
                                   hipStream_t s, int* status) {
  v_scale_finalize_kernel<<<dim3(BH), dim3(kFinThreads), 0, s>>>(part, nch, v_scale, v_inv, zero_mean, status);
  return hipGetLastError();
}

hipError_t launch_quant_q(const InTensor& q, int B, int H, int L, int lq_pad, float premul, int8_t* q_i8,
                          float* q_scale, hipStream_t s, const PrepParams* prep, uint16_t* pooled) {
  const dim3 grid(lq_pad / 128, H, B), block(kThreads);
  const PrepParams none{};
  if (pooled != nullptr && (prep != nullptr || q.D != kD)) return hipErrorInvalidValue;
  KSANA_DISPATCH_DT(q.dtype, {
    if (pooled != nullptr)
      quant_q_kernel<DT, 0, true><<<grid, block, 0, s>>>(q.ptr, q.sB, q.sL, q.sH, H, L, q.D, lq_pad, premul, q_i8,
                                                              q_scale, none, pooled);
    else if (prep == nullptr)
      quant_q_kernel<DT, 0><<<grid, block, 0, s>>>(q.ptr, q.sB, q.sL, q.sH, H, L, q.D, lq_pad, premul, q_i8, q_scale,
                                                        none);
    else {
      PrepParams pp = *prep;
      const size_t lds = plan_rope_lds(&pp, B, 128);
      KSANA_DISPATCH_KIND(pp.kind, (quant_q_kernel<DT, KIND><<<grid, block, lds, s>>>(q.ptr, q.sB, q.sL, q.sH, H, L, q.D, lq_pad,
                                                                                 premul, q_i8, q_scale, pp)));
    }
  });
  return hipGetLastError();
}

hipError_t launch_quant_q_rows(const InTensor& q, int B, int H, int L, int lq_pad, float premul, float eps,
                               int8_t* q_i8, float* q_scale, hipStream_t s, const PrepParams& prep,
                               const InTensor* k_rows, int k_H, int k_L, float* k_rms, int* clear, int n_clear) {
  RowStatOf ks{};
  if (k_rows != nullptr)
    ks = RowStatOf{k_rows->ptr, k_rows->sB, k_rows->sL, k_L, k_H * (kD / 8), (float)(k_H * kD), k_rms};
  const int rows = max(lq_pad, k_rows != nullptr ? k_L : 0);
  const dim3 grid((rows + kRowsQ - 1) / kRowsQ, B), block(kThreads);
  PrepParams pp = prep;
  float* rms_out = const_cast<float*>(pp.inv_rms);  // the caller's statistic area: written here, read by nobody else in this launch
  const size_t lds = 0;  // the rotation factors of a token are held in registers across its heads: nothing is staged
  KSANA_DISPATCH_DT(q.dtype, {
    if (pp.kind == 3)
      quant_q_rows_kernel<DT, 3><<<grid, block, lds, s>>>(q.ptr, q.sB, q.sL, q.sH, H, L, lq_pad, premul, eps, q_i8, q_scale, pp, rms_out, ks, clear, n_clear);
    else
      quant_q_rows_kernel<DT, 1><<<grid, block, lds, s>>>(q.ptr, q.sB, q.sL, q.sH, H, L, lq_pad, premul, eps, q_i8, q_scale, pp, rms_out, ks, clear, n_clear);
  });
  return hipGetLastError();
}

hipError_t launch_quant_k(const InTensor& k, int B, int H, int L, int nkb, const float* k_mean, int8_t* k_tiles,
                          float* k_scale, hipStream_t s, const PrepParams* prep, uint16_t* pooled) {
  const dim3 grid(nkb, H, B), block(kThreads);
  const PrepParams none{};
  if (pooled != nullptr && (prep != nullptr || k.D != kD)) return hipErrorInvalidValue;
  KSANA_DISPATCH_DT(k.dtype, {
    if (pooled != nullptr)
      quant_k_kernel<DT, 0, true><<<grid, block, 0, s>>>(k.ptr, k.sB, k.sL, k.sH, H, L, k.D, nkb, k_mean, k_tiles,
                                                              k_scale, none, pooled);
    else if (prep == nullptr)
      quant_k_kernel<DT, 0><<<grid, block, 0, s>>>(k.ptr, k.sB, k.sL, k.sH, H, L, k.D, nkb, k_mean, k_tiles, k_scale,
                                                        none);
    else {
      PrepParams pp = *prep;
      const size_t lds = plan_rope_lds(&pp, B, kBlkK);
      KSANA_DISPATCH_KIND(pp.kind, (quant_k_kernel<DT, KIND><<<grid, block, lds, s>>>(k.ptr, k.sB, k.sL, k.sH, H, L, k.D, nkb,
                                                                                 k_mean, k_tiles, k_scale, pp)));
    }
  });
  return hipGetLastError();
}

namespace {
constexpr int kMaxDevices = 64;

// Resident-workgroup counts the launchers have asked the runtime for, kept per (device, kernel address): every
// instantiation of a kernel template has its own register and LDS footprint, and all instantiations of one
// template share one function-pointer TYPE, so the address is the key.
class OccupancyCache {
 public:
  int find(int dev, const void* kernel) {
    std::lock_guard<std::mutex> lock(m_);
    for (int i = 0; i < n_; ++i)
      if (e_[i].dev == dev && e_[i].kernel == kernel) return e_[i].workgroups;
    return -1;
  }
  void put(int dev, const void* kernel, int workgroups) {
    std::lock_guard<std::mutex> lock(m_);
    for (int i = 0; i < n_; ++i)
      if (e_[i].dev == dev && e_[i].kernel == kernel) {
        e_[i].workgroups = workgroups;
        return;
      }
    if (n_ < kEntries) e_[n_++] = Entry{dev, kernel, workgroups};  // full: the answer is simply asked for again
  }

 private:
  struct Entry {
    int dev;
    const void* kernel;
    int workgroups;
  };
  static constexpr int kEntries = 256;
  std::mutex m_;
  Entry e_[kEntries];
  int n_ = 0;
};
OccupancyCache g_occupancy;

// Workgroups of `kernel` (256 threads, `lds` bytes of dynamic LDS) the current device holds at once.
// (0 when the runtime cannot tell: the caller then takes the two-pass kernels.)  The answer for a launch
// without dynamic LDS is kept per device and kernel.
template <typename K>
int resident_workgroups(K kernel, size_t lds) {
  int per_cu = 0, dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return 0;
  const void* key = reinterpret_cast<const void*>(kernel);
  if (lds == 0) {
    const int c = g_occupancy.find(dev, key);
    if (c > 0) return c;
  }
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kThreads, lds) != hipSuccess) return 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
  if (lds == 0 && per_cu * cus > 0) g_occupancy.put(dev, key, per_cu * cus);
  return per_cu * cus;
}

// ---- process-wide settings (see QuantOptions) ----------------------------------------------------------------
std::mutex g_opt_mutex;
bool g_opt_ready = false;
QuantOptions g_opt{false, true, kDefaultWaitTicks};

void parse_stages(const char* stages, QuantOptions* o) {
  o->one_read_k = strchr(stages, 'k') != nullptr;
  o->one_read_v = strchr(stages, 'v') != nullptr;
}
void options_from_environment_locked() {
  if (g_opt_ready) return;
  g_opt_ready = true;
  const char* e = getenv("KSANA_SAGE_ONE_READ");
  parse_stages(e ? e : "v", &g_opt);
  const char* w = getenv("KSANA_SAGE_WAIT_TICKS");
  if (w != nullptr && *w != 0) {
    char* end = nullptr;
    const long long v = strtoll(w, &end, 10);
    if (end != w) g_opt.wait_ticks = v;
  }
}

// One word of host memory per device that the device can write (pinned, mapped): a kernel whose wait expires sets it,
// the launchers read it as plain host memory - no copy, no synchronisation.  Allocated when a one-read kernel is first
// launched on the device by a caller that may allocate, and kept until the process ends.
struct HostWord {
  int* host = nullptr;
  int* dev = nullptr;
};
HostWord g_host_word[kMaxDevices];
std::mutex g_host_word_mutex;

HostWord host_word(bool may_allocate) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return HostWord{};
  std::lock_guard<std::mutex> lock(g_host_word_mutex);
  HostWord& w = g_host_word[dev];
  if (w.host == nullptr && may_allocate) {
    void* h = nullptr;
    void* d = nullptr;
    if (hipHostMalloc(&h, 64, hipHostMallocMapped) == hipSuccess) {
      *static_cast<volatile int*>(h) = 0;
      if (hipHostGetDevicePointer(&d, h, 0) == hipSuccess) {
        w.host = static_cast<int*>(h);
        w.dev = static_cast<int*>(d);
      } else {
        (void)hipGetLastError();
        (void)hipHostFree(h);
      }
    } else {
      (void)hipGetLastError();  // no word, no reports: the kernels still end and still give the same bits
    }
  }
  return w;
}

}  // namespace

QuantOptions quant_options() {
  std::lock_guard<std::mutex> lock(g_opt_mutex);
  options_from_environment_locked();
  return g_opt;
}

void configure_quant(const char* stages, long long wait_ticks, bool keep_ticks) {
  {
    std::lock_guard<std::mutex> lock(g_opt_mutex);
    options_from_environment_locked();
    if (stages != nullptr) parse_stages(stages, &g_opt);
    if (!keep_ticks) g_opt.wait_ticks = wait_ticks;
  }
  std::lock_guard<std::mutex> lock(g_host_word_mutex);
  for (HostWord& w : g_host_word)
    if (w.host != nullptr) *static_cast<volatile int*>(w.host) = 0;
}

bool one_read_demoted(bool may_allocate) {
  const HostWord w = host_word(may_allocate);
  return w.host != nullptr && *static_cast<volatile int*>(w.host) != 0;
}

int selftest_occupancy_cache() {
  OccupancyCache c;
  const void* a = reinterpret_cast<const void*>(&quant_k_fused_kernel<KSANA_SAGE_BF16, 1>);
  const void* b = reinterpret_cast<const void*>(&quant_k_fused_kernel<KSANA_SAGE_BF16, 2>);
  if (a == b) return 1;
  if (c.find(0, a) != -1) return 2;
  c.put(0, a, 768);
  if (c.find(0, a) != 768 || c.find(0, b) != -1 || c.find(1, a) != -1) return 3;
  c.put(0, b, 1024);
  c.put(1, a, 512);
  if (c.find(0, a) != 768 || c.find(0, b) != 1024 || c.find(1, a) != 512) return 4;
  c.put(0, a, 256);
  return c.find(0, a) == 256 && c.find(0, b) == 1024 ? 0 : 5;
}

hipError_t launch_block_means(const InTensor& x, int B, int H, int L, int rows, const float* centre, uint16_t* out,
                              hipStream_t s) {
  const dim3 grid((L + rows - 1) / rows, H, B), block(kThreads);
  KSANA_DISPATCH_DT(x.dtype, (block_mean_kernel<DT><<<grid, block, 0, s>>>(x.ptr, x.sB, x.sL, x.sH, H, L, rows, centre, out)));
  return hipGetLastError();
}

hipError_t launch_clear_ints(int* p, int n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  clear_ints_kernel<<<dim3((n + 255) / 256), dim3(256), 0, s>>>(p, n);
  return hipGetLastError();
}

// The one-read forms are used when a head's chunks are at most half of what the chip holds at once (see the
// comment above the kernels); *used tells the caller whether anything was launched.
hipError_t launch_quant_k_fused(const InTensor& k, int B, int H, int L, int nkb, int nch, int smooth, float* part,
                                float* k_mean, int8_t* k_tiles, float* k_scale, const QuantSync& sync, hipStream_t s,
                                const PrepParams* prep, bool* used, bool may_allocate) {
  *used = false;
  if ((int64_t)B * H * nch > INT32_MAX) return hipSuccess;
  if (one_read_demoted(may_allocate)) return hipSuccess;
  const dim3 grid(B * H * nch), block(kThreads);
  const HeadSync sy{sync.k_counter, sync.k_ready, sync.k_status, quant_options().wait_ticks, host_word(false).dev};
  const PrepParams none{};
  hipError_t e = hipSuccess;
  KSANA_DISPATCH_DT(k.dtype, {
    if (prep == nullptr) {
      const int resident = resident_workgroups(quant_k_fused_kernel<DT, 0>, 0);
      if (2 * nch <= resident) {
        quant_k_fused_kernel<DT, 0><<<grid, block, 0, s>>>(k.ptr, k.sB, k.sL, k.sH, H, L, k.D, nkb, nch, part, k_mean,
                                                                k.dtype, smooth, k_tiles, k_scale, none, sy);
        *used = true;
      }
    } else {
      PrepParams pp = *prep;
      const size_t lds = plan_rope_lds(&pp, B, kMeanChunk);
      KSANA_DISPATCH_KIND(pp.kind, {
        // lds != 0 only for kind 1; the cached answer (lds == 0) is kept per kernel address
        if (2 * nch <= resident_workgroups(quant_k_fused_kernel<DT, KIND>, lds)) {
          quant_k_fused_kernel<DT, KIND><<<grid, block, lds, s>>>(k.ptr, k.sB, k.sL, k.sH, H, L, k.D, nkb, nch, part, k_mean,
                                                                   k.dtype, smooth, k_tiles, k_scale, pp, sy);
          *used = true;
        }
      });
    }
  });
  if (*used) e = hipGetLastError();
  return e;
}

// K with the Wan step and V, a launch each or one for both, by the rounds of the chip that one launch takes (`slots` workgroups at
// once, 768 where the grid's factors take up to 30 KB of LDS).  One launch has a gap less (3 us) and fills up its last round once
// and not twice, but V's chunks run three to a compute unit where they would run four.  us per call, a launch each / one, in calls none
// of whose query rows count (what they do besides is the same), at 12, 24 and 40 heads of one entry and 24 and 40 of two:
//   under 1.5 rounds     0.7-0.9: 83.6 / 75.7, 80.6 / 72.3, 80.0 / 68.2; 1.3-1.45: 99.4 / 96.0, 94.7 / 91.7, 108.1 / 101.0
//   1.5 .. 2: slower     112.1 / 116.3, 115.3 / 118.2, 126.1 / 131.0, 120.2 / 130.5, 110.1 / 114.9 (24 of 25 sizes)
//   2 .. 7 rounds        2.7: 192.3 / 175.6, 193.2 / 180.8, 170.8 / 164.5; 4.5: 308.6 / 299.5, 290.3 / 281.3, 289.2 / 281.8; 6.2-6.5:
//                        430.4 / 436.7, 393.7 / 389.9, 395.5 / 387.7, 382.8 / 381.0, 387.9 / 381.8; 6.9: +1.2, +2.7, -3.1, -3.2, -4.0
//   beyond 7: slower     7.1: 462.3 / 464.9, 424.3 / 434.0, 427.9 / 430.4, 413.2 / 414.8, 418.1 / 419.6; up to 14 rounds -1 to +3 %
static bool kv_in_one_launch_pays(int64_t workgroups, int64_t slots) {
  return 2 * workgroups < 3 * slots || (workgroups > 2 * slots && workgroups <= 7 * slots);
}

hipError_t launch_quant_kv_meet(const QkvCall& c, const PrepParams& prep, hipStream_t s, bool* used) {
  *used = false;
  const int64_t grid = 2 * (int64_t)c.B * c.Hkv * c.nch;
  if (grid > INT32_MAX || (prep.kind != 1 && prep.kind != 3) || one_read_demoted()) return hipSuccess;
  const QuantSync& y = c.sync;
  const long long ticks = quant_options().wait_ticks;
  int* host = host_word(false).dev;
  const HeadSync sk{y.k_counter, y.k_ready, y.k_status, ticks, host}, sv{y.v_counter, y.v_ready, y.v_status, ticks, host};
  PrepParams pp = prep;
  const size_t lds = plan_rope_lds(&pp, c.B, kMeanChunk);
  auto go = [&](auto kernel) {
    const int slots = resident_workgroups(kernel, lds);
    if (2 * c.nch > slots || !kv_in_one_launch_pays(grid, slots)) return;
    kernel<<<dim3((unsigned)grid), dim3(kThreads), lds, s>>>(c, pp, sk, sv);
    *used = true;
  };
  KSANA_DISPATCH_DT(c.k.dtype, {
    if (pp.kind == 1) go(quant_kv_meet_kernel<DT, 1>);
    else go(quant_kv_meet_kernel<DT, 3>);
  });
  return *used ? hipGetLastError() : hipSuccess;
}

hipError_t launch_quant_v_fused(const InTensor& v, int B, int H, int L, int nkb, int nch, float* part, float* v_scale,
                                float* v_inv, float* v_mean, uint8_t* v_tiles, const QuantSync& sync, hipStream_t s,
                                bool* used) {
  *used = false;
  if ((int64_t)B * H * nch > INT32_MAX) return hipSuccess;
  if (one_read_demoted()) return hipSuccess;
  const dim3 grid(B * H * nch), block(kThreads);
  const HeadSync sy{sync.v_counter, sync.v_ready, sync.v_status, quant_options().wait_ticks, host_word(false).dev};
  hipError_t e = hipSuccess;
  KSANA_DISPATCH_DT(v.dtype, {
    const int resident = resident_workgroups(quant_v_fused_kernel<DT>, 0);
    if (2 * nch <= resident) {
      quant_v_fused_kernel<DT><<<grid, block, 0, s>>>(v.ptr, v.sB, v.sL, v.sH, H, L, v.D, nkb, nch, part, v_scale, v_inv,
                                                       v_mean, v_tiles, sy);
      *used = true;
    }
  });
  if (*used) e = hipGetLastError();
  return e;
}

// Two stages while a head's partial results stay small next to the rows a workgroup of stage 2 quantizes (64 chunks are
// 32 KiB, the rows 16-32 KiB) and the second reading of K and V comes from the last-level cache (256 MB).  Beyond that
// calls without a folded step take the meeting launch.  us, stages / meeting / separate kernels:
//   40 heads of 9000 tokens (176 MB of K and V) 106 / 108 / 120; 24 heads of 17000 (199 MB) 125 / 122 / 135, two entries of
//   8500 122 / 117 / 131; 40 heads of 14000 (273 MB) 192 / 158 / 184; 8 heads of 20000 (78 MB, 79 chunks) 46 / 49 / 56.
constexpr int kStageMaxChunks = 64;
constexpr int64_t kStageMaxBytes = 192ll << 20;
// The joint block's calls beyond it take the separate kernels (K from one read, the step done once): stages / separate, whole
// calls of 24 heads, one entry of 15512 tokens (191 MB) 1604 / 1608, four of 3856 (190 MB) 572.5 / 574.5, of 7056 (347 MB) 1552 /
// 1533, one of 16256 (200 MB) 1708 / 1700, two of 10512 (258 MB) 1578 / 1567.  A meeting launch with the step in it is no gain over them.
// Joint block, several heads per item or one: from this many workgroups (of one head, Q's blocks and K's and V's chunks) on the
// items of several heads still fill the chip.  Whole calls, us, one / several: 24 heads of 1024 tokens 42.2 / 48.3, of 2560 (960
// workgroups) 82.2 / 84.8, of 4512 203 / 196; two entries of 1024 54.2 / 58.9, of 1328 (1104) 84.7 / 83.9, of 2056 133 / 128, of
// 4352 360 / 347.5, of 6512 689 / 664.
constexpr int kJointHeadsFrom = 1104;
// Beyond this many chunks a head's first workgroups wait for its last ones longer than a second pass takes (296 chunks:
// the separate quantizers are 3 % faster).
constexpr int kMeetMaxChunks = 160;
// From here on stage 2 has workgroups enough to give each two tiles per statistic it forms.  us, with 1 / 2 / 4 tiles (an
// attention launch without rows, 10-35 us, in each figure): plain, 1024 tiles 18.5 / 20.1 / 20.7, 2048 33.1 / 33.5 / 33.9,
// 3264 45.8 / 45.2 / 46.4, 6528 86.0 / 83.3 / 83.9, 11280 143.0 / 140.1 / 141.0; joint block, 1024 32.2 / 35.2 / 38.5, 3264
// 68.6 / 71.0 / 73.6, 5120 92.6 / 91.3 / 96.7, 6528 125.4 / 124.3 / 127.2.
constexpr int kTwoTilesFrom = 2048, kTwoTilesFromJoint = 4096;

template <int DT, int KIND>
static hipError_t launch_qkv_kind(QkvCall& c, const PrepParams& pq, const PrepParams& pk, hipStream_t s, bool* used) {
  static_assert(KIND == 0 || KIND == 2, "nothing folded in, or the joint block's step");
  const dim3 block(kThreads);
  const int64_t n_q = (int64_t)c.B * c.Hq * c.nqb, n_chunks = (int64_t)c.B * c.Hkv * c.nch;
  const int more = KIND == 0 ? numbers_batch(c.numbers) : 0;
  if (c.nch == 1) {
    quant_qkv_small_kernel<DT, KIND><<<dim3((unsigned)(n_q + 2 * n_chunks + more)), block, 0, s>>>(c, pq, pk);
    *used = true;
  } else if (c.nch <= kStageMaxChunks && 4 * (int64_t)c.B * c.Hkv * c.Lk * c.k.D <= kStageMaxBytes) {
    const int64_t tiles = 2 * (int64_t)c.B * c.Hkv * c.nkb;
    c.tiles_per_wg = tiles >= (KIND == 0 ? kTwoTilesFrom : kTwoTilesFromJoint) ? 2 : 1;
    const int64_t n_v2 = (int64_t)c.B * c.Hkv * ((c.nkb + c.tiles_per_wg - 1) / c.tiles_per_wg);
    if (KIND == 2 && n_q + 2 * n_chunks >= kJointHeadsFrom) {
      const int64_t k_groups = (int64_t)c.B * ((c.Hkv + kJointHeadsK - 1) / kJointHeadsK);
      const int64_t n_rows = c.nqb == 0 ? 0 : (int64_t)c.B * ((c.Hq + kJointHeadsQ - 1) / kJointHeadsQ) * (c.lq_pad / kSlots);
      quant_qkv_stage1_kernel<DT, 2, true><<<dim3((unsigned)(n_rows + n_chunks + (c.smooth_k ? k_groups * c.nch : 0))), block, 0, s>>>(c, pq, pk);
      quant_qkv_stage2_kernel<DT, 2, true><<<dim3((unsigned)(k_groups * c.nkb + n_v2)), block, 0, s>>>(c, pk);
    } else {
      quant_qkv_stage1_kernel<DT, KIND, false><<<dim3((unsigned)(n_q + (c.smooth_k ? 2 : 1) * n_chunks + more)), block, 0, s>>>(c, pq, pk);
      quant_qkv_stage2_kernel<DT, KIND, false><<<dim3((unsigned)(2 * n_v2)), block, 0, s>>>(c, pk);
    }
    *used = true;
  } else if (KIND == 0 && c.nch <= kMeetMaxChunks) {
    const QuantOptions opt = quant_options();
    // (V's one-read setting stands for both here: K's letter concerns its separate kernel, see ksana_sage_configure)
    if (!opt.one_read_v || one_read_demoted()) return hipSuccess;
    if (2 * c.nch > resident_workgroups(quant_qkv_meet_kernel<DT>, 0)) return hipSuccess;
    int* host = host_word(false).dev;
    const QuantSync& y = c.sync;
    const int n_words = (int)(y.v_status - y.k_counter) + kSyncStride;
    const hipError_t e = launch_clear_ints(y.k_counter, n_words, s);
    if (e != hipSuccess) return e;
    const HeadSync sk{y.k_counter, y.k_ready, y.k_status, opt.wait_ticks, host}, sv{y.v_counter, y.v_ready, y.v_status, opt.wait_ticks, host};
    quant_qkv_meet_kernel<DT><<<dim3((unsigned)(n_q + 2 * n_chunks + more)), block, 0, s>>>(c, sk, sv);
    *used = true;
  }
  return hipGetLastError();
}

hipError_t launch_quant_qkv(const QkvCall& call, const PrepParams* pq, const PrepParams* pk, hipStream_t s, bool* used) {
  *used = false;
  QkvCall c = call;
  const int kind = pq != nullptr ? pq->kind : (pk != nullptr ? pk->kind : 0);
  if (kind != 0 && kind != 2) return hipSuccess;
  if ((int64_t)c.B * c.Hq * c.nqb + 2 * (int64_t)c.B * c.Hkv * c.nkb >= INT32_MAX) return hipSuccess;
  // (a side without anything to apply runs with every step of its parameters switched off)
  PrepParams off{};
  off.kind = kind;
  const PrepParams &a = pq != nullptr ? *pq : off, &b = pk != nullptr ? *pk : off;
  hipError_t e = hipSuccess;
  KSANA_DISPATCH_DT(c.q.dtype, { e = kind == 0 ? launch_qkv_kind<DT, 0>(c, a, b, s, used) : launch_qkv_kind<DT, 2>(c, a, b, s, used); });
  return e;
}

// us per call, every workgroup by itself / a launch in between: 40 heads of 3000 tokens (12 chunks) 122 / 131, of 6867 (27) 272 / 281, of
// 12000 (47) 483 / 486, of 32760 (128) 2006 / 1938; 12 heads of 16000 (63) 234 / 247.
constexpr int kSlaReadyChunks = 64;

hipError_t launch_quant_sla(const QkvCall& call, const SlaFinal& f, hipStream_t s) {
  QkvCall c = call;
  c.tiles_per_wg = 2 * (int64_t)c.B * c.Hkv * c.nkb >= kTwoTilesFrom ? 2 : 1;
  const bool ready = c.nch >= kSlaReadyChunks;
  if (ready) c.tiles_per_wg = 1;
  const int64_t n_bh = (int64_t)c.B * c.Hkv;
  const int64_t n = 2 * n_bh * ((c.nkb + c.tiles_per_wg - 1) / c.tiles_per_wg) + (int64_t)c.B * c.Hq * c.nqb;
  const int64_t n_fin = n_bh * (kD / kFinRows);
  if (n + n_fin > INT32_MAX) return hipErrorInvalidValue;
  const dim3 block(kThreads);
  KSANA_DISPATCH_DT(c.q.dtype, {
    if (ready) {
      sla_finalize_kernel<DT><<<dim3((unsigned)(2 * n_bh + n_fin)), block, 0, s>>>(c, f);
      quant_sla_kernel<DT, true><<<dim3((unsigned)n), block, 0, s>>>(c, f);
    } else {
      quant_sla_kernel<DT, false><<<dim3((unsigned)(n_fin + n)), block, 0, s>>>(c, f);
    }
  });
  return hipGetLastError();
}

hipError_t launch_quant_v(const InTensor& v, int B, int H, int L, int nkb, const float* v_inv, const float* v_mean,
                          uint8_t* v_tiles, hipStream_t s) {
  const dim3 grid(nkb, H, B), block(kThreads);
  KSANA_DISPATCH_DT(v.dtype, {
    if (v_mean != nullptr)
      quant_v_kernel<DT, true><<<grid, block, 0, s>>>(v.ptr, v.sB, v.sL, v.sH, H, L, v.D, nkb, v_inv, v_mean, v_tiles);
    else
      quant_v_kernel<DT, false><<<grid, block, 0, s>>>(v.ptr, v.sB, v.sL, v.sH, H, L, v.D, nkb, v_inv, nullptr, v_tiles);
  });
  return hipGetLastError();
}

}  // namespace ksana_sage
