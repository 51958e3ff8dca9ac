// The first pass of the sparse-linear backend's linear branch, shared by its own kernels and by the quantizers' launches that
// take it along: phi(k)^T v over runs of rows, and the finalisation per head.
#pragma once

#include "sage_device.h"
#include "sage_kernels.h"

namespace ksana_sage {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

constexpr float kLog2e = 1.4426950408889634f;

template <int DT>
__device__ __forceinline__ v4f mfma16(const uint4& a, const uint4& b, const v4f& c) {
  if constexpr (DT == KSANA_SAGE_BF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), c, 0, 0, 0);
}
template <int DT>
__device__ __forceinline__ v16f mfma32(const uint4& a, const uint4& b, const v16f& c) {
  if constexpr (DT == KSANA_SAGE_BF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), c, 0, 0, 0);
}

// two fp32 values -> one dword of the half type (a in the low half)
template <int DT>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  if constexpr (DT == KSANA_SAGE_BF16) {
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    const b2 p = {(__bf16)a, (__bf16)b};
    return __builtin_bit_cast(uint32_t, p);
  } else {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const h2 p = {(_Float16)a, (_Float16)b};
    return __builtin_bit_cast(uint32_t, p);
  }
}
template <int DT>
__device__ __forceinline__ float round_half(float x) {
  if constexpr (DT == KSANA_SAGE_BF16) return (float)(__bf16)x;
  return (float)(_Float16)x;
}

// value of lane ^ M within the lane's group of 16, M = 1, 2, 4, 8 (DPP: quad permutes, half-row mirror, row rotation)
template <int M>
__device__ __forceinline__ float xor16(float v) {
  const int iv = __float_as_int(v);
  if constexpr (M == 1) return __int_as_float(__builtin_amdgcn_mov_dpp(iv, 0xB1, 0xF, 0xF, true));
  if constexpr (M == 2) return __int_as_float(__builtin_amdgcn_mov_dpp(iv, 0x4E, 0xF, 0xF, true));
  if constexpr (M == 8) return __int_as_float(__builtin_amdgcn_mov_dpp(iv, 0x128, 0xF, 0xF, true));  // row_ror:8
  const int t = __builtin_amdgcn_mov_dpp(iv, 0x141, 0xF, 0xF, true);                                // row_half_mirror
  return __int_as_float(__builtin_amdgcn_mov_dpp(t, 0x1B, 0xF, 0xF, true));                         // quad_perm [3,2,1,0]
}
__device__ __forceinline__ float max16(float v) {
  v = fmaxf(v, xor16<1>(v));
  v = fmaxf(v, xor16<2>(v));
  v = fmaxf(v, xor16<4>(v));
  return fmaxf(v, xor16<8>(v));
}
__device__ __forceinline__ float sum16(float v) {
  v += xor16<1>(v);
  v += xor16<2>(v);
  v += xor16<4>(v);
  return v + xor16<8>(v);
}

// ---------------------------------------------------------------------------------------------------------------
// kv and ksum over one run of rows of one head, by a workgroup of 256 threads.
//
// A workgroup walks its rows 256 at a time, in two halves of 32 rows per wave.  Lane (j = lane % 16, g = lane / 16) of wave w
// loads the rows 8 w + 4 hs + g + 32 i of half hs, i = 0 .. 7, channels 8 j .. 8 j + 7 of k and of v (16 bytes each; a load
// instruction covers four whole 256-byte rows).  The matrix instruction (16x16x32, contraction over 32 rows, whichever) wants,
// per lane, 8 ROWS of one channel: column t of the lane's 8 x 8 block - a matter of picking halves of registers, no data moves
// between lanes.  Tile t of the 128 phi(k) channels is therefore the strided set {8 j + t}, likewise tile u of the v
// channels {8 j + u}; the result is put back in order when it is written.
// The softmax of a row needs its 128 channels: 8 in the lane, the rest across the 16 lanes of its group (DPP).
// Operand fragments go through LDS so that every wave can use the rows of all four: wave w keeps the phi(k) tiles
// 2 w, 2 w + 1 against all eight v tiles (64 accumulator registers) and, against an all-ones operand, their row sums.
//
// kStats: the chunk sums of K and the chunk maxima of |V| are taken along for the quantizers (k_part, v_part as
// col_partial_chunk writes them): with the rows above a lane adds row slot 8 w + 4 hs + g of the specified order by itself,
// and the slots meet pairwise across g, the halves and the waves.
// ---------------------------------------------------------------------------------------------------------------
constexpr int kSlaStepRows = kMeanChunk;
constexpr int kSlaPartFloats = kD * kD + kD;  // one partial: kv, then ksum

template <int DT, bool kStats>
__device__ __forceinline__ void sla_kv_run(int run, int runs, int h, int b, const uint16_t* __restrict__ k, int64_t ksB, int64_t ksL,
                                           int64_t ksH, const uint16_t* __restrict__ v, int64_t vsB, int64_t vsL, int64_t vsH, int H,
                                           int L, int rows_per_run, float* __restrict__ part, float* __restrict__ k_part,
                                           float* __restrict__ v_part, int nch) {
  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int j = lane & 15, g = lane >> 4;
  const int r_begin = run * rows_per_run, r_end = min(L, r_begin + rows_per_run);
  const uint16_t* kb = k + b * ksB + h * ksH + 8 * j;
  const uint16_t* vb = v + b * vsB + h * vsH + 8 * j;
  // fragments in operand order: [wave whose rows][tile][lane] x 16 bytes
  __shared__ uint4 s_a[4 * 8 * 64];
  __shared__ uint4 s_b[4 * 8 * 64];
  [[maybe_unused]] __shared__ float s_stat[kStats ? 2 : 1][4][kStats ? kD : 1];
  v4f acc[2][8], accs[2];
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    accs[m] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < 8; ++u) acc[m][u] = v4f{0.f, 0.f, 0.f, 0.f};
  }
  uint4 ones;
  {
    const uint32_t one2 = DT == KSANA_SAGE_BF16 ? 0x3f803f80u : 0x3c003c00u;
    ones = make_uint4(one2, one2, one2, one2);
  }
  // A half's rows are requested while the half before it is multiplied.  What bounds it is the chain of a half-step - row
  // reductions, conversions, two barriers - in two workgroups per compute unit (LDS and registers allow no third): 40 heads of
  // 32760 rows 162 us, 189 with the statistics (3.6 TB/s; column sums of K and maxima of V on their own took 70 and 50).
  uint4 kx[8], vx[8];
  auto request = [&](int row0) {
    const uint16_t *kr = kb + (int64_t)row0 * ksL, *vr = vb + (int64_t)row0 * vsL;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      // (rows past the run: its last row again, and zeros in its place)
      const int back = min(0, r_end - 1 - (row0 + 32 * i));
      kx[i] = *reinterpret_cast<const uint4*>(kr + (int64_t)(32 * i + back) * ksL);
      vx[i] = *reinterpret_cast<const uint4*>(vr + (int64_t)(32 * i + back) * vsL);
    }
  };
  auto clear_past = [&](int row0) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (row0 + 32 * i >= r_end) kx[i] = vx[i] = make_uint4(0, 0, 0, 0);
  };
  request(r_begin + 8 * w + g);
  [[maybe_unused]] float k_first[8], v_first[8];  // of the half before
  for (int r0 = r_begin, hs = 0; r0 < r_end; r0 += hs * kSlaStepRows, hs ^= 1) {
    [[maybe_unused]] float k_sum[8], v_top[8];
    {
      const int row0 = r0 + 8 * w + 4 * hs + g;
      if (r0 + kSlaStepRows > r_end) clear_past(row0);  // uniform: the run's last rows
      // column t of the lane's 8 x 8 block is its fragment of tile t; v's first, its registers are wanted
      if constexpr (kStats) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          float y[8];
          widen8<DT>(vx[i], y);
#pragma unroll
          for (int e = 0; e < 8; ++e) v_top[e] = i == 0 ? fabsf(y[e]) : fmaxf(v_top[e], fabsf(y[e]));
        }
      }
#pragma unroll
      for (int tt = 0; tt < 8; ++tt) {
        // half (tt & 1) of dword tt / 2 of each row's register
        const uint32_t sel = (tt & 1) ? 0x07060302u : 0x05040100u;  // (high halves | low halves) of (src0, src1)
        auto dw = [&](const uint4& r) { return tt < 2 ? r.x : (tt < 4 ? r.y : (tt < 6 ? r.z : r.w)); };
        s_b[(w * 8 + tt) * 64 + lane] =
            make_uint4(__builtin_amdgcn_perm(dw(vx[1]), dw(vx[0]), sel), __builtin_amdgcn_perm(dw(vx[3]), dw(vx[2]), sel),
                       __builtin_amdgcn_perm(dw(vx[5]), dw(vx[4]), sel), __builtin_amdgcn_perm(dw(vx[7]), dw(vx[6]), sel));
      }
      __builtin_amdgcn_sched_barrier(0);
      // phi(k): softmax over the row's 128 channels, rounded to the half type as it is packed, two rows to a register
      uint32_t f[4][8];
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        float x[2][8];
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          const int i = 2 * m + r;
          widen8<DT>(kx[i], x[r]);
          if constexpr (kStats) {
#pragma unroll
            for (int e = 0; e < 8; ++e) k_sum[e] = i == 0 ? x[r][e] : k_sum[e] + x[r][e];
          }
          float mx = fmaxf(fmaxf(fmaxf(x[r][0], x[r][1]), fmaxf(x[r][2], x[r][3])), fmaxf(fmaxf(x[r][4], x[r][5]), fmaxf(x[r][6], x[r][7])));
          mx = max16(mx);
          const float c = -mx * kLog2e;
          float sum = 0.0f;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            x[r][e] = __builtin_amdgcn_exp2f(__builtin_fmaf(x[r][e], kLog2e, c));
            sum += x[r][e];
          }
          sum = sum16(sum);
          const float inv = row0 + 32 * i < r_end ? __builtin_amdgcn_rcpf(sum) : 0.0f;  // rows past the run contribute nothing
#pragma unroll
          for (int e = 0; e < 8; ++e) x[r][e] *= inv;
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) f[m][e] = pack2<DT>(x[0][e], x[1][e]);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int tt = 0; tt < 8; ++tt) s_a[(w * 8 + tt) * 64 + lane] = make_uint4(f[0][tt], f[1][tt], f[2][tt], f[3][tt]);
      request(hs == 0 ? row0 + 4 : row0 - 4 + kSlaStepRows);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (kStats) {
        // lanes g and g ^ 1 (16 lanes apart), then g ^ 2 (32), then the two halves: the adjacent-pair tree over the wave's slots
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const auto a16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(k_sum[e]), __float_as_uint(k_sum[e]), false, false);
          const float a = __uint_as_float(a16[0]) + __uint_as_float(a16[1]);
          const auto a32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(a), false, false);
          k_sum[e] = __uint_as_float(a32[0]) + __uint_as_float(a32[1]);
        }
        if (hs == 0) {
#pragma unroll
          for (int e = 0; e < 8; ++e) k_first[e] = k_sum[e], v_first[e] = v_top[e];
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            k_sum[e] = k_first[e] + k_sum[e];
            const float m = fmaxf(v_first[e], v_top[e]);
            const auto m16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(m), __float_as_uint(m), false, false);
            const float n = fmaxf(__uint_as_float(m16[0]), __uint_as_float(m16[1]));
            const auto m32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(n), __float_as_uint(n), false, false);
            v_top[e] = fmaxf(__uint_as_float(m32[0]), __uint_as_float(m32[1]));
          }
          if (g == 0) {
#pragma unroll
            for (int e = 0; e < 8; ++e) s_stat[0][w][8 * j + e] = k_sum[e], s_stat[1][w][8 * j + e] = v_top[e];
          }
        }
      }
      __syncthreads();
      if constexpr (kStats) {
        if (hs == 1) {
          const int d = t & (kD - 1);
          const int64_t at = (((int64_t)b * H + h) * nch + r0 / kMeanChunk) * kD + d;
          if (t < kD)
            k_part[at] = (s_stat[0][0][d] + s_stat[0][1][d]) + (s_stat[0][2][d] + s_stat[0][3][d]);
          else
            v_part[at] = fmaxf(fmaxf(s_stat[1][0][d], s_stat[1][1][d]), fmaxf(s_stat[1][2][d], s_stat[1][3][d]));
        }
      }
      // the 32 rows wave ks brought, ks = 0 .. 3; the operands of the next four are read while four are multiplied
      uint4 fa[2], fb[2][4];
      auto read_b = [&](int n) {
#pragma unroll
        for (int u = 0; u < 4; ++u) fb[n & 1][u] = s_b[((n >> 1) * 8 + 4 * (n & 1) + u) * 64 + lane];
      };
      read_b(0);
#pragma unroll
      for (int n = 0; n < 8; ++n) {
        if ((n & 1) == 0) fa[0] = s_a[((n >> 1) * 8 + 2 * w) * 64 + lane], fa[1] = s_a[((n >> 1) * 8 + 2 * w + 1) * 64 + lane];
        if (n + 1 < 8) read_b(n + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int at = 4 * (n & 1) + u;
          acc[0][at] = mfma16<DT>(fa[0], fb[n & 1][u], acc[0][at]);
          acc[1][at] = mfma16<DT>(fa[1], fb[n & 1][u], acc[1][at]);
        }
        if ((n & 1) == 1) accs[0] = mfma16<DT>(fa[0], ones, accs[0]), accs[1] = mfma16<DT>(fa[1], ones, accs[1]);
        __builtin_amdgcn_sched_barrier(0);
      }
      __syncthreads();  // the fragments have been read: the next half may overwrite them
    }
  }
  // accumulator register r of tile (m, u): phi(k) channel 8 * (4 g + r) + (2 w + m), v channel 8 * j + u
  float* out = part + (((int64_t)b * H + h) * runs + run) * kSlaPartFloats;
#pragma unroll
  for (int m = 0; m < 2; ++m) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int ck = 8 * (4 * g + r) + 2 * w + m;
      float* orow = out + ck * kD + 8 * j;
      *reinterpret_cast<float4*>(orow) = make_float4(acc[m][0][r], acc[m][1][r], acc[m][2][r], acc[m][3][r]);
      *reinterpret_cast<float4*>(orow + 4) = make_float4(acc[m][4][r], acc[m][5][r], acc[m][6][r], acc[m][7][r]);
      if (j == 0) out[kD * kD + ck] = accs[m][r];  // every column of the all-ones product holds the row sum
    }
  }
}

// ---------------------------------------------------------------------------------------------------------------
// Per head: the runs' partial results added in run order; kv and ksum rounded to the half type (they are tensors of
// that type in the reference); then M = kv W^T (fp32 accumulation) where a projection is folded in, M = kv otherwise.
// M is stored for sla_apply_kernel's A operand: fragment (nt, s) = 64 lanes x 8 halves, lane (n = lane % 32,
// g = lane / 32) holding M[16 s + 8 g + i][32 nt + n], i = 0 .. 7.  16 rows of kv (slice of 8) per workgroup of 256 threads.
// ---------------------------------------------------------------------------------------------------------------
constexpr int kSlaThreads = 256;
constexpr int kFinRows = 16;  // rows of kv per workgroup

template <int DT>
__device__ __forceinline__ void sla_kv_finalize(int slice, int bh, const float* __restrict__ part, int runs,
                                                const float* __restrict__ proj_w, uint16_t* __restrict__ m_frag,
                                                float* __restrict__ ksum) {
  const int d0 = slice * kFinRows, t = threadIdx.x;
  __shared__ __attribute__((aligned(16))) float s_kv[kFinRows * kD];
  const float* p = part + (int64_t)bh * runs * kSlaPartFloats;
  // Bound by latency: the runs are added in order, but read four at a time, both of the thread's quadruples together (one
  // value of one run at a time, 12 runs were 96 memory latencies one after the other: 40 heads 39 -> 16 us).
  constexpr int kQuads = kFinRows * kD / 4 / kSlaThreads, kAtOnce = 4;
  float4 sum[kQuads];
#pragma unroll
  for (int i = 0; i < kQuads; ++i) sum[i] = make_float4(0.f, 0.f, 0.f, 0.f);
  float sum1 = 0.0f;
  for (int r0 = 0; r0 < runs; r0 += kAtOnce) {
    float4 x[kAtOnce][kQuads];
    float y[kAtOnce];
#pragma unroll
    for (int c = 0; c < kAtOnce; ++c) {
      const float* pr = p + (int64_t)min(r0 + c, runs - 1) * kSlaPartFloats;
#pragma unroll
      for (int i = 0; i < kQuads; ++i) x[c][i] = *reinterpret_cast<const float4*>(pr + d0 * kD + 4 * (i * kSlaThreads + t));
      y[c] = pr[kD * kD + d0 + (t & (kFinRows - 1))];
    }
#pragma unroll
    for (int c = 0; c < kAtOnce; ++c) {
      if (r0 + c >= runs) break;  // uniform
#pragma unroll
      for (int i = 0; i < kQuads; ++i) sum[i].x += x[c][i].x, sum[i].y += x[c][i].y, sum[i].z += x[c][i].z, sum[i].w += x[c][i].w;
      sum1 += y[c];
    }
  }
#pragma unroll
  for (int i = 0; i < kQuads; ++i)
    *reinterpret_cast<float4*>(s_kv + 4 * (i * kSlaThreads + t)) =
        make_float4(round_half<DT>(sum[i].x), round_half<DT>(sum[i].y), round_half<DT>(sum[i].z), round_half<DT>(sum[i].w));
  if (t < kFinRows) ksum[bh * kD + d0 + t] = round_half<DT>(sum1);
  __syncthreads();
  // thread t: output column n = t % 128 for the rows d0 + (t / 128), d0 + (t / 128) + 2, ...
  const int n = t & (kD - 1);
  float m[kFinRows / 2];
  if (proj_w != nullptr) {
#pragma unroll
    for (int i = 0; i < kFinRows / 2; ++i) m[i] = 0.0f;
    const float4* wr = reinterpret_cast<const float4*>(proj_w + n * kD);  // W[n][c]
#pragma unroll 8
    for (int c4 = 0; c4 < kD / 4; ++c4) {
      const float4 wv = wr[c4];
#pragma unroll
      for (int i = 0; i < kFinRows / 2; ++i) {
        const float* kr = s_kv + ((t >> 7) + 2 * i) * kD + 4 * c4;  // the same address in every lane: a broadcast
        m[i] = __builtin_fmaf(kr[0], wv.x, m[i]);
        m[i] = __builtin_fmaf(kr[1], wv.y, m[i]);
        m[i] = __builtin_fmaf(kr[2], wv.z, m[i]);
        m[i] = __builtin_fmaf(kr[3], wv.w, m[i]);
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < kFinRows / 2; ++i) m[i] = s_kv[((t >> 7) + 2 * i) * kD + n];
  }
#pragma unroll
  for (int i = 0; i < kFinRows / 2; ++i) {
    const int d = d0 + (t >> 7) + 2 * i;
    const int nt = n >> 5, s = d >> 4, g = (d >> 3) & 1, e = d & 7, lane = 32 * g + (n & 31);
    uint16_t bits;
    if constexpr (DT == KSANA_SAGE_BF16)
      bits = __builtin_bit_cast(uint16_t, (__bf16)m[i]);
    else
      bits = __builtin_bit_cast(uint16_t, (_Float16)m[i]);
    m_frag[(int64_t)bh * kD * kD + ((nt * 8 + s) * 64 + lane) * 8 + e] = bits;
  }
}

// ---- the second pass, one row per pair of lanes (row = lane % 32 of the wave, g = lane / 32): out = phi(q) M / (1e-5 +
// phi(q) . ksum) ---------------------------------------------------------------------------------------------------
// raw[s]: the channels 16 s + 8 g .. + 7 of the lane's row, s = 0 .. 7 - half of the row, and its B operands of the
// 32x32x16 instruction; the other half sits in lane + 32.  x: the exponentials of its channels; returns 1 / their row sum.
template <int DT>
__device__ __forceinline__ float sla_row_exps(const uint4 (&raw)[8], float (&x)[8][8]) {
  float mx = -INFINITY;
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    widen8<DT>(raw[s], x[s]);
#pragma unroll
    for (int e = 0; e < 8; ++e) mx = fmaxf(mx, x[s][e]);
  }
  mx = over_halves<Max>(mx);
  const float c = -mx * kLog2e;
  float sum = 0.0f;
#pragma unroll
  for (int s = 0; s < 8; ++s)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      x[s][e] = __builtin_amdgcn_exp2f(__builtin_fmaf(x[s][e], kLog2e, c));
      sum += x[s][e];
    }
  sum = over_halves<Sum>(sum);
  return __builtin_amdgcn_rcpf(sum);
}
// the operands fq (phi in the half type) and 1 / (1e-5 + phi . ksum); s_ks: ksum of the head, in LDS
template <int DT>
__device__ __forceinline__ float sla_row_scale(const float (&x)[8][8], float inv, const float* s_ks, int g, uint4 (&fq)[8]) {
  float den = 0.0f;
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    uint32_t pw[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float f0 = x[s][2 * e] * inv, f1 = x[s][2 * e + 1] * inv;
      pw[e] = pack2<DT>(f0, f1);
      den = __builtin_fmaf(f0, s_ks[16 * s + 8 * g + 2 * e], den);
      den = __builtin_fmaf(f1, s_ks[16 * s + 8 * g + 2 * e + 1], den);
    }
    fq[s] = make_uint4(pw[0], pw[1], pw[2], pw[3]);
  }
  den = over_halves<Sum>(den);
  return __builtin_amdgcn_rcpf(1e-5f + den);
}
// Output channels 32 nt .. + 31 of the lane's row, transposed (out^T = M^T phi(q)^T): register r is channel
// 32 nt + 8 (r / 4) + 4 g + r % 4.  s_m: M in operand order, in LDS.
template <int DT>
__device__ __forceinline__ v16f sla_row_product(const uint4* s_m, const uint4 (&fq)[8], int nt, int lane) {
  v16f acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
#pragma unroll
  for (int s = 0; s < 8; ++s) acc = mfma32<DT>(s_m[(nt * 8 + s) * 64 + lane], fq[s], acc);
  return acc;
}

}  // namespace ksana_sage
