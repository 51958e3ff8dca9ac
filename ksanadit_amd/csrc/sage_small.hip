// Short calls in one launch: quantize K, V and Q and attend, everything between the inputs and the result in registers
// and LDS.  For at most 256 keys (one chunk of the K statistic: a workgroup sees its head's whole key sequence), where the
// two launches of the general path cost more than their work.
//
// A workgroup is 8 waves = 256 query rows of one (batch, head).  Waves 0-3 first quantize the head's K and waves 4-7 its V, in
// the quantizers' thread mapping (32 row slots x 8 lanes x 16 channels), into LDS tiles of the attention kernel's operand
// order; then every wave walks them for its 32 rows.  Operations, orders and roundings are those of the quantizers and of
// the general kernel, so the result is the same bits.
//
// Bound by the length of its instruction stream: a wave alone on its SIMD issues one every five cycles.  32 tokens take 18 000
// cycles: 2 900 up to the loads, 2 400 for the statistics, 3 400 quantizing, 2 100 turning V, 4 000 for the one tile, 2 400 on
// the way out.  us per call, issued one after the other, two launches / this: 32 tokens of 2 x 64 heads 15.1 / 9.8, 65 of 4 x 24
// 19.3 / 12.3, 156 of 8 (64 channels, causal) 21.0 / 12.1, 250 of 40 24.6 / 17.7, 256 of 4 x 64 38 / 27; 8 000 queries on 200
// keys, 8 heads 34 / 24.
#include "sage_attn_device.h"

#include <atomic>

#include "../../include/ksana_sage_hip.h"

namespace ksana_sage {
namespace {

constexpr int kComputeUnits = 256;
constexpr int kThreads = 512, kHalf = 256, kSlots = 32, kMaxTiles = kMeanChunk / kBlkK;
constexpr int kChunkRows = kMeanChunk / kSlots;  // rows per slot
constexpr int kVPitch = kD + 16;                 // bytes per row of V's codes before they are turned
constexpr int kOutPitch = 2 * kD + 16;           // bytes per result row on its way out
constexpr int kSmallFloats = 8 * kD + 3 * kD + kMaxTiles + 4 * kMaxTiles;

// LDS: K tiles, V^T tiles; V's codes row by row, later (read by then) the result rows; small things
constexpr int turn_bytes(int n, int rows_wg) { return n * kBlkK * kVPitch > rows_wg * kOutPitch ? n * kBlkK * kVPitch : rows_wg * kOutPitch; }
constexpr size_t small_lds(int n, int rows_wg) { return 2 * n * kTileBytes + turn_bytes(n, rows_wg) + kSmallFloats * 4; }

struct Sum {
  static __device__ __forceinline__ float of(float a, float b) { return a + b; }
};
struct Max {
  static __device__ __forceinline__ float of(float a, float b) { return fmaxf(a, b); }
};
// v of this lane and of lane ^ 8, ^ 16, ^ 32 in turn: the adjacent-pair tree over a wave's eight row slots
template <typename Op>
__device__ __forceinline__ float over_slots(float v) {
  v = Op::of(v, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x128, 0xF, 0xF, true)));  // row_ror:8
  const auto r16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = Op::of(__uint_as_float(r16[0]), __uint_as_float(r16[1]));
  const auto r32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return Op::of(__uint_as_float(r32[0]), __uint_as_float(r32[1]));
}

// kG: 32-channel groups that hold data, as in the general kernel
template <int DT, int kG>
__global__ __launch_bounds__(kThreads) void sage_small_kernel(const SmallCall c, int n_qwg, int rows_wg) {
  want(c.q.ptr, c.k.sL, c.o.ptr, c.B, c.k_lens);
  constexpr int kMagicBits = kG == 4 ? kMagicI : kMagicI2;
  constexpr float kMagicVal = kG == 4 ? kMagicF : kMagicF2;
  const int bh = blockIdx.x / n_qwg, qwg = blockIdx.x - bh * n_qwg;
  const int b = bh / c.Hq, h = bh - b * c.Hq, hk = h / (c.Hq / c.Hkv);
  const int t = threadIdx.x & (kHalf - 1), slot = t >> 3, c16 = t & 7, lane = t & 63, l32 = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), w4 = wave & 3;
  const bool on_k = wave < 4;  // this wave's half of the workgroup quantizes K, the other one V
  // (the half with V, which has less to do, takes the first 128 query rows)
  const bool my_rows = (wave ^ 4) * 32 < rows_wg;
  const int q0 = qwg * rows_wg + (wave ^ 4) * 32, row = q0 + l32;
  int lq = c.Lq, lk = c.Lk;  // rows and keys that take part
  take_counts(c.q_lens, c.k_lens, b, lq, lk);
  if (lk == 0 || qwg * rows_wg >= lq) {  // uniform: softmax over no key, or no row that takes part
    if (my_rows && row < c.Lq && 64 * hh < c.d_out) {
      uint4* orow = reinterpret_cast<uint4*>(c.o.ptr + b * c.o.sB + (int64_t)row * c.o.sL + h * c.o.sH + 64 * hh);
#pragma unroll
      for (int i = 0; i < 8; ++i) orow[i] = make_uint4(0, 0, 0, 0);
    }
    return;
  }
  const bool active = my_rows && q0 < lq;  // wave-uniform
  const int n_tiles = (lk + kBlkK - 1) / kBlkK;

  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int n_lds = (c.Lk + kBlkK - 1) / kBlkK;
  uint8_t* k_tiles = smem;
  uint8_t* v_tiles = k_tiles + n_lds * kTileBytes;
  uint8_t* v_rows = v_tiles + n_lds * kTileBytes;
  float(*s_k)[kD] = reinterpret_cast<float(*)[kD]>(v_rows + turn_bytes(n_lds, rows_wg));
  float(*s_v)[kD] = s_k + 4;
  float* s_mean = s_v[4];
  float* s_inv = s_mean + kD;
  float* s_vs = s_inv + kD;
  float* s_ks = s_vs + kD;
  float(*s_red)[4] = reinterpret_cast<float(*)[4]>(s_ks + kMaxTiles);

  // ---- everything the workgroup reads is requested together -----------------------------------------
  uint4 raw[kChunkRows][2], qr[8];
  const bool has = c16 * 16 < c.k.D;  // (head size 64: the upper channels are zeros)
  const uint16_t* base = (on_k ? c.k.ptr + b * c.k.sB + hk * c.k.sH : c.v.ptr + b * c.v.sB + hk * c.v.sH) + c16 * 16;
  const int64_t sL = on_k ? c.k.sL : c.v.sL;  // (rows are walked with one 64-bit step)
  base += slot * sL;
#pragma unroll
  for (int i = 0; i < kChunkRows; ++i) {
    raw[i][0] = raw[i][1] = make_uint4(0, 0, 0, 0);
    if (i * kSlots < c.Lk) fetch_row16(base + i * (kSlots * sL), has && i * kSlots + slot < c.Lk, raw[i]);
  }
  const uint16_t* qrow = c.q.ptr + b * c.q.sB + (int64_t)row * c.q.sL + h * c.q.sH + 16 * hh;
#pragma unroll
  for (int s = 0; s < kG; ++s) {
    qr[2 * s] = qr[2 * s + 1] = make_uint4(0, 0, 0, 0);
    if (active && row < c.Lq && 32 * s < c.q.D) {
      qr[2 * s] = *reinterpret_cast<const uint4*>(qrow + 32 * s);
      qr[2 * s + 1] = *reinterpret_cast<const uint4*>(qrow + 32 * s + 8);
    }
  }

  // ---- the head's statistics: K's channel means, V's channel maxima ---------------------------------
  {
    float acc[16];
    if (on_k) {
#pragma unroll
      for (int i = 0; i < kChunkRows; ++i) {
        if (i != 0 && i * kSlots >= c.Lk) continue;  // uniform: rows of zeros
        float x[16];
        widen8<DT>(raw[i][0], x);
        widen8<DT>(raw[i][1], x + 8);
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[e] = i == 0 ? x[e] : acc[e] + x[e];
      }
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[e] = over_slots<Sum>(acc[e]);
    } else {
#pragma unroll
      for (int i = 0; i < kChunkRows; ++i) {
        if (i != 0 && i * kSlots >= c.Lk) continue;
        float x[16];
        widen8<DT>(raw[i][0], x);
        widen8<DT>(raw[i][1], x + 8);
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[e] = i == 0 ? fabsf(x[e]) : fmaxf(acc[e], fabsf(x[e]));
      }
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[e] = over_slots<Max>(acc[e]);
    }
    if (lane < 8) {
#pragma unroll
      for (int e = 0; e < 16; ++e) (on_k ? s_k : s_v)[w4][c16 * 16 + e] = acc[e];
    }
  }
  __syncthreads();
  if (t < kD) {
    if (on_k) {
      const float mean = __fdiv_rn((s_k[0][t] + s_k[1][t]) + (s_k[2][t] + s_k[3][t]), (float)c.Lk);
      s_mean[t] = c.smooth_k ? round_to_half_dtype(mean, DT) : 0.0f;
    } else {
      const float top = fmaxf(fmaxf(s_v[0][t], s_v[1][t]), fmaxf(s_v[2][t], s_v[3][t]));
      const bool nz = top > 0.0f;
      s_inv[t] = nz ? __fdiv_rn(448.0f, top) : 0.0f;
      s_vs[t] = nz ? __fdiv_rn(top, 448.0f) : 0.0f;
    }
  }
  __syncthreads();

  // ---- each wave's own query rows; V: codes to LDS row by row; K: transform, and the tiles' maxima --------
  // (Q in the attention kernel's mapping, one row per lane: 800 instructions for a wave's 32 rows.  In the quantizers' mapping
  // they are 250 for every eight, shared by waves that have no rows of their own: no faster.)
  v4i qf[4];
  float qs = 0.0f;
#pragma unroll
  for (int s = 0; s < 4; ++s) qf[s] = v4i{0, 0, 0, 0};
  if (active) quant_q_rows<DT, kG>(qr, c.premul, qf, qs);
  float x[kMaxTiles][2][16];
  float stat[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) stat[e] = (on_k ? s_mean : s_inv)[c16 * 16 + e];
  if (on_k) {
#pragma unroll
    for (int tt = 0; tt < kMaxTiles; ++tt) {
      if (tt >= n_tiles) continue;  // uniform
      float amax = 0.0f;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if ((2 * tt + i) * kSlots >= c.Lk) {  // uniform
#pragma unroll
          for (int e = 0; e < 16; ++e) x[tt][i][e] = 0.0f;
          continue;
        }
        widen8<DT>(raw[2 * tt + i][0], x[tt][i]);
        widen8<DT>(raw[2 * tt + i][1], x[tt][i] + 8);
        const bool valid = has && (2 * tt + i) * kSlots + slot < c.Lk;
#pragma unroll
        for (int e = 0; e < 16; ++e) x[tt][i][e] = valid ? x[tt][i][e] - stat[e] : 0.0f;
        fwht128(x[tt][i], c16);
#pragma unroll
        for (int e = 0; e < 16; ++e) amax = fmaxf(amax, fabsf(x[tt][i][e]));
      }
      amax = fmaxf(amax, lane_xor<1>(amax));
      amax = fmaxf(amax, lane_xor<2>(amax));
      amax = fmaxf(amax, lane_xor<4>(amax));
      amax = over_slots<Max>(amax);
      if (lane == 0) s_red[tt][w4] = amax;
    }
  } else {
#pragma unroll
    for (int i = 0; i < kChunkRows; ++i) {
      if (i >= 2 * n_tiles) continue;  // uniform
      float y[16];
      widen8<DT>(raw[i][0], y);
      widen8<DT>(raw[i][1], y + 8);
      uint32_t w[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float z[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) z[e] = fminf(fmaxf(y[4 * j + e] * stat[4 * j + e], -448.0f), 448.0f);
        int packed = 0;
        packed = __builtin_amdgcn_cvt_pk_fp8_f32(z[0], z[1], packed, false);
        packed = __builtin_amdgcn_cvt_pk_fp8_f32(z[2], z[3], packed, true);
        w[j] = (uint32_t)packed;
      }
      *reinterpret_cast<uint4*>(v_rows + (i * kSlots + slot) * kVPitch + c16 * 16) = make_uint4(w[0], w[1], w[2], w[3]);
    }
  }
  __syncthreads();
  // ---- K's tiles, and V's turned out of the rows by the whole workgroup (the order of quant_v_block) ----
#pragma unroll
  for (int tt = 0; tt < kMaxTiles; ++tt) {
    if (tt >= n_tiles) continue;
    const uint8_t* rows = v_rows + tt * kBlkK * kVPitch;
    const int oc = threadIdx.x, dt = oc >> 7, th = (oc >> 6) & 1, d = dt * 32 + l32;
    uint32_t w[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      uint32_t a = 0;
#pragma unroll
      for (int k = 0; k < 4; ++k) a |= (uint32_t)rows[(32 * th + 8 * g + 4 * hh + k) * kVPitch + d] << (8 * k);
      w[g] = a;
    }
    *reinterpret_cast<uint4*>(v_tiles + tt * kTileBytes + oc * 16) = make_uint4(w[0], w[1], w[2], w[3]);
  }
  static_assert(kThreads * 16 == kTileBytes, "one piece of a tile per thread");
  if (on_k) {
#pragma unroll
    for (int tt = 0; tt < kMaxTiles; ++tt) {
      if (tt >= n_tiles) continue;
      const float amax = fmaxf(fmaxf(s_red[tt][0], s_red[tt][1]), fmaxf(s_red[tt][2], s_red[tt][3]));
      const bool nz = amax > 0.0f;
      const float inv_lane = (nz ? __fdiv_rn(127.0f, amax) : 0.0f) * fwht_lane_sign(c16);
      if (t == 0) s_ks[tt] = nz ? __fdiv_rn(amax, 127.0f) : 0.0f;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int frag = i * 4 + (c16 >> 1), ln = (c16 & 1) * 32 + slot;
        *reinterpret_cast<uint4*>(k_tiles + tt * kTileBytes + (frag * 64 + ln) * 16) = pack_int8x16(x[tt][i], inv_lane);
      }
    }
  }
  __syncthreads();

  // ---- attention, tile by tile (the general kernel's steps without its pipeline) ----------------------
  v16f oacc[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) oacc[dt][r] = 0.0f;
  v4f lacc = {0.0f, 0.0f, 0.0f, 0.0f};  // row sums, see the general kernel for the operand of ones
  if (active) {
    v8i ones;
    v16i magic;
#pragma unroll
    for (int r = 0; r < 8; ++r) ones[r] = ((lane >> 2) & 1) == ((lane >> 4) & 1) ? 0x38383838 : 0;
#pragma unroll
    for (int r = 0; r < 16; ++r) magic[r] = kMagicBits;
    float m_run = -INFINITY, x_base = -INFINITY, x_limit = -INFINITY;
    const int n_mine = c.causal ? min(n_tiles, (q0 >> 6) + 1) : n_tiles;
    for (int j = 0; j < n_mine; ++j) {
      v16i s[2];
      qk_tile<kG>(k_tiles + j * kTileBytes, lane, qf, magic, s);
      // keys [0, allowed) of the tile count for this row
      const int allowed = min(kBlkK, (c.causal ? min(lk, row + 1) : lk) - j * kBlkK);
      const bool whole = __all(allowed == kBlkK);
      if (!whole) blank_scores<kMagicBits>(s, hh, allowed);
      int top = s[0][0];
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int r = 0; r < 16; ++r) top = max(top, s[u][r]);
      float sc = qs * s_ks[j], mneg = -kMagicVal * sc;
      const float alpha = move_point(top, sc, mneg, qs, m_run, x_base, x_limit);
      if (j == 0 ? __any(alpha != alpha) : __any(alpha != 1.0f)) {
#pragma unroll
        for (int dt = 0; dt < kG; ++dt)
#pragma unroll
          for (int r = 0; r < 16; ++r) oacc[dt][r] *= alpha;
        lacc[0] *= alpha;
      }
      v8i pf = tile_probs(s, sc, x_base + mneg);
      if (!whole) blank_probs(pf, hh, allowed);
      const uint8_t* vt = v_tiles + j * kTileBytes;
#pragma unroll
      for (int dt = 0; dt < kG; ++dt) {
        const v4i lo = *reinterpret_cast<const v4i*>(vt + ((dt * 2 + 0) * 64 + lane) * 16);
        const v4i hi = *reinterpret_cast<const v4i*>(vt + ((dt * 2 + 1) * 64 + lane) * 16);
        const v8i vf = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        oacc[dt] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(vf, pf, oacc[dt], 0, 0, 0, 0, 0, 0);
      }
      lacc = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(ones, pf, lacc, 0, 0, 0, 0, 0, 0);
    }
  }

  // ---- O = O^T / rowsum * v_scale, whole rows out through LDS -----------------------------------------
  // (a dense row always has a sum; causal rows: as the general kernel has it)
  const float inv_l = !c.causal || lacc[0] > 0.0f ? 1.0f / lacc[0] : 0.0f;
  float4 s4[16];
#pragma unroll
  for (int i = 0; i < 4 * kG; ++i) s4[i] = reinterpret_cast<const float4*>(s_vs)[(32 * (i >> 2) + 8 * (i & 3) + 4 * hh) >> 2];
  uint8_t* stage = v_rows + (wave ^ 4) * (32 * kOutPitch);
  if (!my_rows) return;
#pragma unroll
  for (int i = 0; i < 4 * kG; ++i) {
    const int dt = i >> 2, g = i & 3;
    *reinterpret_cast<uint2*>(stage + l32 * kOutPitch + 2 * (32 * dt + 8 * g + 4 * hh)) =
        half4<DT>(oacc[dt][4 * g + 0] * inv_l * s4[i].x, oacc[dt][4 * g + 1] * inv_l * s4[i].y,
                  oacc[dt][4 * g + 2] * inv_l * s4[i].z, oacc[dt][4 * g + 3] * inv_l * s4[i].w);
  }
  uint16_t* obase = c.o.ptr + b * c.o.sB + h * c.o.sH;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int idx = i * 64 + lane, r = idx >> 4, piece = idx & 15;
    const uint4 w = *reinterpret_cast<const uint4*>(stage + r * kOutPitch + 16 * piece);
    if (q0 + r < c.Lq && 8 * piece < c.d_out && 8 * piece < 32 * kG) *reinterpret_cast<uint4*>(obase + (int64_t)(q0 + r) * c.o.sL + 8 * piece) = w;
  }
  // Rows that do not count become zeros, whatever their q, or v, holds.  (By the threads that have just written them and not
  // in their stead: a branch ahead of the stores holds up the last instructions of every call, 9.9 -> 10.1 us at 32 tokens.)
  if (q0 + 32 > lq) {
#pragma unroll 1
    for (int i = 0; i < 8; ++i) {
      const int idx = i * 64 + lane, r = idx >> 4, piece = idx & 15;
      if (q0 + r >= lq && q0 + r < c.Lq && 8 * piece < c.d_out)
        *reinterpret_cast<uint4*>(obase + (int64_t)(q0 + r) * c.o.sL + 8 * piece) = make_uint4(0, 0, 0, 0);
    }
  }
}

template <int DT, int kG>
hipError_t launch(const SmallCall& c, int n_qwg, int rows_wg, hipStream_t s) {
  // more than 64 KiB of dynamic LDS has to be requested per kernel, once per device
  constexpr int kMaxDevices = 64;
  static std::atomic<bool> requested[kMaxDevices];
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  if (!requested[dev].load(std::memory_order_acquire)) {
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(&sage_small_kernel<DT, kG>), hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)small_lds(kMaxTiles, 256));
    if (e != hipSuccess) return e;
    requested[dev].store(true, std::memory_order_release);
  }
  const int n = (c.Lk + kBlkK - 1) / kBlkK;
  sage_small_kernel<DT, kG><<<dim3(c.B * c.Hq * n_qwg), dim3(kThreads), small_lds(n, rows_wg), s>>>(c, n_qwg, rows_wg);
  return hipGetLastError();
}

}  // namespace

// One round of the chip: every workgroup quantizes its head's K and V by itself, and beyond that the general path, which does
// it once, is ahead (us, two launches / this: 280 workgroups of 256 keys 34 / 42, 504 of 250 keys 45 / 46; 256 of 200 keys 34 / 24).
bool small_call_suits(int B, int Hq, int Lq, int Lk) { return Lk <= kMeanChunk && (int64_t)B * Hq * ((Lq + 255) / 256) <= kComputeUnits; }

hipError_t launch_small(const SmallCall& c, hipStream_t s) {
  // 128 rows a workgroup while there is a compute unit for each: the attention then has its SIMDs to itself, one wave on each
  // (250 tokens of 40 heads 21.8 / 18.0 us with 256 / 128)
  const int rows_wg = c.B * c.Hq * ((c.Lq + 127) / 128) <= kComputeUnits ? 128 : 256;
  const int n_qwg = (c.Lq + rows_wg - 1) / rows_wg;
  const bool bf16 = c.o.dtype == KSANA_SAGE_BF16;
  if (c.d_out <= 64) return bf16 ? launch<KSANA_SAGE_BF16, 2>(c, n_qwg, rows_wg, s) : launch<KSANA_SAGE_FP16, 2>(c, n_qwg, rows_wg, s);
  return bf16 ? launch<KSANA_SAGE_BF16, 4>(c, n_qwg, rows_wg, s) : launch<KSANA_SAGE_FP16, 4>(c, n_qwg, rows_wg, s);
}

}  // namespace ksana_sage
