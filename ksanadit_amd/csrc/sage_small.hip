// Short calls in one launch: quantize K, V and Q and attend, everything between the inputs and the result in registers
// and LDS.  For at most 256 keys (one chunk of the K statistic: a workgroup sees its head's whole key sequence), where the
// two launches of the general path cost more than their work.
//
// A workgroup is 8 waves and 32 to 256 query rows of one (batch, head).  Waves 0-3 first quantize the head's K and waves 4-7
// its V, in the quantizers' thread mapping (32 row slots x 8 lanes x 16 channels), into LDS tiles of the attention kernel's
// operand order; Q follows, and then the waves walk the tiles, 32 rows each - or several for the same rows with a share of the
// output channels each.  Operations, orders and roundings are those of the quantizers and of the general kernel, so the
// result is the same bits.
//
// Bound by the length of its instruction stream: a wave alone on its SIMD issues one every five cycles.  Hence as many waves as
// there are on everything: up to 64 rows are quantized eight to a wave, and up to 128 leave several waves to each 32 rows.
// GPU time in us of calls replayed from a graph, one wave for each 32 rows from their quantization to the result / this:
// 32 tokens of 2 x 64 heads 9.2 / 5.8, 65 of 4 x 24 12.0 / 9.6, 100 of 16 12.3 / 9.2, 156 of 8 (64 channels, causal) 12.0 / 10.2,
// 200 of 2 x 32 (64 channels) 15.4 / 13.9, 250 of 40 17.5 / 16.4, 256 of 4 x 64 26.6 / 26.4; 8 000 queries on 200 keys, 8 heads
// 23.2 / 22.1.  (The two launches of the general path: 32 tokens of 2 x 64 heads 15.1, 250 of 40 24.6, 256 of 4 x 64 38.)
#include "sage_attn_device.h"

#include <atomic>
#include <type_traits>

#include "../../include/ksana_sage_hip.h"

namespace ksana_sage {
namespace {

constexpr int kComputeUnits = 256;
constexpr int kThreads = 512, kHalf = 256, kSlots = 32, kMaxTiles = kMeanChunk / kBlkK;
constexpr int kChunkRows = kMeanChunk / kSlots;  // rows per slot
constexpr int kVPitch = kD + 16;                 // bytes per row of V's codes before they are turned
constexpr int kSmallFloats = 8 * kD + 3 * kD + kMaxTiles + 4 * kMaxTiles;

// LDS: K tiles, V^T tiles; V's codes row by row; Q's operands and scales; small things
constexpr size_t small_lds(int n, int rows_wg) { return 2 * n * kTileBytes + n * kBlkK * kVPitch + rows_wg * (kD + 4) + kSmallFloats * 4; }

// kG: 32-channel groups that hold data, as in the general kernel.  kRows: query rows of a workgroup.
template <int DT, int kG, int kRows>
__global__ __launch_bounds__(kThreads) void sage_small_kernel(const SmallCall c) {
  want(c.q.ptr, c.k.sL, c.o.ptr, c.B, c.k_lens);
  constexpr int kMagicBits = kG == 4 ? kMagicI : kMagicI2;
  constexpr float kMagicVal = kG == 4 ? kMagicF : kMagicF2;
  // waves per 32 rows, each with kDt 32-channel groups of their result (the scores and probabilities each works out by itself)
  constexpr int kRowGroups = kRows / 32, kShare = kG < 8 / kRowGroups ? kG : 8 / kRowGroups, kDt = kG / kShare;
  constexpr bool kQSlots = kRows <= 64;             // Q by V's waves in the quantizers' mapping; else 32 rows by one wave
  constexpr bool kQHanded = !kQSlots && kShare > 1;  // ... which hands its operand to the waves it shares them with
  const int qwg = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int hk = c.group == 1 ? h : (int)__umulhi((unsigned)h, c.group_magic);  // h / group
  const int t = threadIdx.x & (kHalf - 1), slot = t >> 3, c16 = t & 7, lane = t & 63, l32 = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), w4 = wave & 3;
  const bool on_k = wave < 4;  // this wave's half of the workgroup quantizes K, the other one V
  // (the half with V, which has less to do, comes first)
  const int row_group = (wave ^ 4) % kRowGroups, share = (wave ^ 4) / kRowGroups;
  const int q0 = qwg * kRows + row_group * 32, row = q0 + l32;
  int lq = c.Lq, lk = c.Lk;  // rows and keys that take part
  take_counts(c.q_lens, c.k_lens, b, lq, lk);
  uint16_t* obase = c.o.ptr + b * c.o.sB + h * c.o.sH;
  if (lk == 0 || qwg * kRows >= lq) {  // uniform: softmax over no key, or no row that takes part
    const int piece = threadIdx.x & 15;
    for (int r = qwg * kRows + (threadIdx.x >> 4); r < min(c.Lq, (qwg + 1) * kRows); r += kThreads / 16)
      if (8 * piece < c.d_out) *reinterpret_cast<uint4*>(obase + (int64_t)r * c.o.sL + 8 * piece) = make_uint4(0, 0, 0, 0);
    return;
  }
  const bool active = share < kShare && q0 < lq;  // wave-uniform
  const int n_tiles = (lk + kBlkK - 1) / kBlkK;

  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int n_lds = (c.Lk + kBlkK - 1) / kBlkK;
  uint8_t* k_tiles = smem;
  uint8_t* v_tiles = k_tiles + n_lds * kTileBytes;
  uint8_t* v_rows = v_tiles + n_lds * kTileBytes;
  uint8_t* q_ops = v_rows + n_lds * kBlkK * kVPitch;
  float* s_qs = reinterpret_cast<float*>(q_ops + kRows * kD);
  float(*s_k)[kD] = reinterpret_cast<float(*)[kD]>(s_qs + kRows);
  float(*s_v)[kD] = s_k + 4;
  float* s_mean = s_v[4];
  float* s_inv = s_mean + kD;
  float* s_vs = s_inv + kD;
  float* s_ks = s_vs + kD;
  float(*s_red)[4] = reinterpret_cast<float(*)[4]>(s_ks + kMaxTiles);

  // ---- everything the workgroup reads is requested together -----------------------------------------
  // (blocks of 32 keys beyond the last one are not looked at again, hence left as they are)
  uint4 raw[kChunkRows][2], qr[8];
  const bool has = c16 * 16 < c.k.D;  // (head size 64: the upper channels are zeros)
  const uint16_t* base = (on_k ? c.k.ptr + b * c.k.sB + hk * c.k.sH : c.v.ptr + b * c.v.sB + hk * c.v.sH) + c16 * 16;
  const int64_t sL = on_k ? c.k.sL : c.v.sL;  // (rows are walked with one 64-bit step)
  base += slot * sL;
#pragma unroll
  for (int i = 0; i < kChunkRows; ++i) {
    if (i * kSlots >= c.Lk) break;  // uniform
    fetch_row16(base + i * (kSlots * sL), has && i * kSlots + slot < c.Lk, raw[i]);
  }
  if constexpr (kQSlots) {
    if (!on_k) {
      const uint16_t* qrow = c.q.ptr + b * c.q.sB + (int64_t)(qwg * kRows + slot) * c.q.sL + h * c.q.sH + 16 * c16;
#pragma unroll
      for (int g = 0; g < kRowGroups; ++g) {
        uint4 two[2];
        fetch_row16(qrow + g * (kSlots * c.q.sL), has && qwg * kRows + g * kSlots + slot < c.Lq, two);
        qr[2 * g] = two[0], qr[2 * g + 1] = two[1];
      }
    }
  } else if (active && share == 0) {
    const uint16_t* qrow = c.q.ptr + b * c.q.sB + (int64_t)row * c.q.sL + h * c.q.sH + 16 * hh;
#pragma unroll
    for (int s = 0; s < kG; ++s) {
      qr[2 * s] = qr[2 * s + 1] = make_uint4(0, 0, 0, 0);
      if (row < c.Lq && 32 * s < c.q.D) {
        qr[2 * s] = *reinterpret_cast<const uint4*>(qrow + 32 * s);
        qr[2 * s + 1] = *reinterpret_cast<const uint4*>(qrow + 32 * s + 8);
      }
    }
  }

  // ---- the head's statistics: K's channel means, V's channel maxima ---------------------------------
  {
    float acc[16];
    float4 part;
    if (on_k) {
#pragma unroll
      for (int i = 0; i < kChunkRows; ++i) {
        if (i != 0 && i * kSlots >= c.Lk) break;  // uniform: no rows
        float x[16];
        widen8<DT>(raw[i][0], x);
        widen8<DT>(raw[i][1], x + 8);
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[e] = i == 0 ? x[e] : acc[e] + x[e];
      }
      part = over_slots16<Sum>(acc);
    } else {
#pragma unroll
      for (int i = 0; i < kChunkRows; ++i) {
        if (i != 0 && i * kSlots >= c.Lk) break;
        float x[16];
        widen8<DT>(raw[i][0], x);
        widen8<DT>(raw[i][1], x + 8);
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[e] = i == 0 ? fabsf(x[e]) : fmaxf(acc[e], fabsf(x[e]));
      }
      part = over_slots16<Max>(acc);
    }
    store_slots16(part, lane, (on_k ? s_k : s_v)[w4]);
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

  // ---- V: codes to LDS row by row; K: transform, and the tiles' maxima; Q --------------------------------
  v4i qf[4];
  float qs = 0.0f;
#pragma unroll
  for (int s = 0; s < 4; ++s) qf[s] = v4i{0, 0, 0, 0};
  if constexpr (!kQSlots) {
    if (active && share == 0) {
      quant_q_rows<DT, kG>(qr, c.premul, qf, qs);
      if constexpr (kQHanded) {
#pragma unroll
        for (int s = 0; s < kG; ++s) *reinterpret_cast<v4i*>(q_ops + ((row_group * 4 + s) * 64 + lane) * 16) = qf[s];
        if (hh == 0) s_qs[row_group * 32 + l32] = qs;
      }
    }
  }
  float x[kMaxTiles][2][16];
  float stat[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) stat[e] = (on_k ? s_mean : s_inv)[c16 * 16 + e];
  if (on_k) {
#pragma unroll
    for (int tt = 0; tt < kMaxTiles; ++tt) {
      if (tt >= n_tiles) break;  // uniform
      float amax = 0.0f;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if ((2 * tt + i) * kSlots >= c.Lk) break;  // uniform: half a tile without keys, which nobody reads
        widen8<DT>(raw[2 * tt + i][0], x[tt][i]);
        widen8<DT>(raw[2 * tt + i][1], x[tt][i] + 8);
        const bool valid = has && (2 * tt + i) * kSlots + slot < c.Lk;
#pragma unroll
        for (int e = 0; e < 16; ++e) x[tt][i][e] = valid ? x[tt][i][e] - stat[e] : 0.0f;
        fwht128(x[tt][i], c16);
#pragma unroll
        for (int e = 0; e < 16; ++e) amax = fmaxf(amax, fabsf(x[tt][i][e]));
      }
      amax = over_lanes<Max>(amax);
      if (lane == 0) s_red[tt][w4] = amax;
    }
  } else {
#pragma unroll
    for (int i = 0; i < kChunkRows; ++i) {
      if (i >= 2 * n_tiles || i * kSlots >= c.Lk) break;  // uniform
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
    if constexpr (kQSlots) {
      // 250 instructions for every eight rows, where one wave needs 800 for 32 in its operand's own mapping
#pragma unroll
      for (int g = 0; g < kRowGroups; ++g) {
        float y[16];
        widen8<DT>(qr[2 * g], y);
        widen8<DT>(qr[2 * g + 1], y + 8);
        fwht128(y, c16);
        float amax = 0.0f;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          y[e] = y[e] * c.premul;
          amax = fmaxf(amax, fabsf(y[e]));
        }
        amax = fmaxf(amax, lane_xor<1>(amax));
        amax = fmaxf(amax, lane_xor<2>(amax));
        amax = fmaxf(amax, lane_xor<4>(amax));
        const Int8Scale r = int8_scale(amax);
        const float inv_lane = r.inv * fwht_lane_sign(c16);
        *reinterpret_cast<uint4*>(q_ops + ((g * 4 + (c16 >> 1)) * 64 + (c16 & 1) * 32 + slot) * 16) = pack_int8x16(y, inv_lane);
        if (c16 == 0) s_qs[g * kSlots + slot] = r.scale;
      }
    }
  }
  __syncthreads();
  // ---- K's tiles, and V's turned out of the rows by the whole workgroup (the order of quant_v_block) ----
#pragma unroll
  for (int tt = 0; tt < kMaxTiles; ++tt) {
    if (tt >= n_tiles) break;
    const uint8_t* rows = v_rows + tt * kBlkK * kVPitch;
    const int oc = threadIdx.x, dt = oc >> 7, th = wave & 1, d = dt * 32 + l32;
    uint32_t w[4] = {0, 0, 0, 0};
    if (tt * kBlkK + 32 * th < c.Lk) {  // uniform; keys that are not there: zeros (their probabilities are, too)
#pragma unroll
      for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int k = 0; k < 4; ++k) w[g] |= (uint32_t)rows[(32 * th + 8 * g + 4 * hh + k) * kVPitch + d] << (8 * k);
    }
    *reinterpret_cast<uint4*>(v_tiles + tt * kTileBytes + oc * 16) = make_uint4(w[0], w[1], w[2], w[3]);
  }
  static_assert(kThreads * 16 == kTileBytes, "one piece of a tile per thread");
  if (on_k) {
#pragma unroll
    for (int tt = 0; tt < kMaxTiles; ++tt) {
      if (tt >= n_tiles) break;
      const float amax = fmaxf(fmaxf(s_red[tt][0], s_red[tt][1]), fmaxf(s_red[tt][2], s_red[tt][3]));
      const Int8Scale r = int8_scale(amax);
      const float inv_lane = r.inv * fwht_lane_sign(c16);
      if (t == 0) s_ks[tt] = r.scale;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if ((2 * tt + i) * kSlots >= c.Lk) break;
        const int frag = i * 4 + (c16 >> 1), ln = (c16 & 1) * 32 + slot;
        *reinterpret_cast<uint4*>(k_tiles + tt * kTileBytes + (frag * 64 + ln) * 16) = pack_int8x16(x[tt][i], inv_lane);
      }
    }
  }
  __syncthreads();
  if (share >= kShare) return;

  // ---- attention, tile by tile (the general kernel's steps without its pipeline) ----------------------
  v16f oacc[kDt];
#pragma unroll
  for (int dt = 0; dt < kDt; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) oacc[dt][r] = 0.0f;
  v4f lacc = {0.0f, 0.0f, 0.0f, 0.0f};  // row sums, see the general kernel for the operand of ones
  if (active) {
    if constexpr (kQSlots || kQHanded) {
#pragma unroll
      for (int s = 0; s < kG; ++s) qf[s] = *reinterpret_cast<const v4i*>(q_ops + ((row_group * 4 + s) * 64 + lane) * 16);
      qs = s_qs[row_group * 32 + l32];
    }
    v8i ones;
    v16i magic;
#pragma unroll
    for (int r = 0; r < 8; ++r) ones[r] = ((lane >> 2) & 1) == ((lane >> 4) & 1) ? 0x38383838 : 0;
#pragma unroll
    for (int r = 0; r < 16; ++r) magic[r] = kMagicBits;
    float m_run = -INFINITY, x_base = -INFINITY, x_limit = -INFINITY;
    const int n_mine = c.causal ? min(n_tiles, (q0 >> 6) + 1) : n_tiles;
    // one tile; half: it holds at most 32 keys, and its second half is left out
    auto tile = [&](int j, auto half) {
      constexpr int kHalves = decltype(half)::value ? 1 : 2;
      const uint8_t* kt = k_tiles + j * kTileBytes + lane * 16;
      v16i s[2] = {magic, magic};
#pragma unroll
      for (int i = 0; i < kG; ++i)
#pragma unroll
        for (int u = 0; u < kHalves; ++u)
          s[u] = __builtin_amdgcn_mfma_i32_32x32x32_i8(*reinterpret_cast<const v4i*>(kt + (u * 4 + i) * 1024), qf[i], s[u], 0, 0, 0);
      // keys [0, allowed) of the tile count for this row
      const int allowed = min(kBlkK, (c.causal ? min(lk, row + 1) : lk) - j * kBlkK);
      const bool whole = __all(allowed >= 32 * kHalves);
      if (!whole) blank_scores<kMagicBits, kHalves>(s, hh, allowed);
      int top = s[0][0];
#pragma unroll
      for (int u = 0; u < kHalves; ++u)
#pragma unroll
        for (int r = 0; r < 16; ++r) top = max(top, s[u][r]);
      float sc = qs * s_ks[j], mneg = -kMagicVal * sc;
      const float alpha = move_point(top, sc, mneg, qs, m_run, x_base, x_limit);
      if (j == 0 ? __any(alpha != alpha) : __any(alpha != 1.0f)) {
#pragma unroll
        for (int dt = 0; dt < kDt; ++dt)
#pragma unroll
          for (int r = 0; r < 16; ++r) oacc[dt][r] *= alpha;
        lacc[0] *= alpha;
      }
      v8i pf = tile_probs<kHalves>(s, sc, x_base + mneg);
      if (!whole) blank_probs<kHalves>(pf, hh, allowed);
      const uint8_t* vt = v_tiles + j * kTileBytes + (share * kDt * 2 * 64 + lane) * 16;
#pragma unroll
      for (int dt = 0; dt < kDt; ++dt) {
        const v4i lo = *reinterpret_cast<const v4i*>(vt + (dt * 2 + 0) * 1024);
        const v4i hi = *reinterpret_cast<const v4i*>(vt + (dt * 2 + 1) * 1024);
        const v8i vf = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        oacc[dt] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(vf, pf, oacc[dt], 0, 0, 0, 0, 0, 0);
      }
      lacc = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(ones, pf, lacc, 0, 0, 0, 0, 0, 0);
    };
    for (int j = 0; j < n_mine; ++j) {
      if (lk - j * kBlkK > 32) tile(j, std::false_type{});
      else tile(j, std::true_type{});
    }
  }

  // ---- O = O^T / rowsum * v_scale, written from the registers -------------------------------------------
  // (a dense row always has a sum; causal rows: as the general kernel has it)
  const float inv_l = !c.causal || lacc[0] > 0.0f ? 1.0f / lacc[0] : 0.0f;
  const float4* s4 = reinterpret_cast<const float4*>(s_vs) + share * kDt * 8 + hh;
  uint16_t* orow = obase + (int64_t)row * c.o.sL + share * kDt * 32 + 8 * hh;
#pragma unroll
  for (int dt = 0; dt < kDt; ++dt)
#pragma unroll
    for (int g = 0; g < 4; g += 2) {
      uint2 w[2];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const float4 s = s4[8 * dt + 2 * (g + e)];
        const int r = 4 * (g + e);
        w[e] = half4<DT>(oacc[dt][r] * inv_l * s.x, oacc[dt][r + 1] * inv_l * s.y, oacc[dt][r + 2] * inv_l * s.z, oacc[dt][r + 3] * inv_l * s.w);
        // rows that do not count become zeros, whatever their q, or v, holds
        if (row >= lq) w[e] = make_uint2(0, 0);
      }
      // lanes l and l + 32 trade every second four channels, so that each stores eight in a row
      const auto lo = __builtin_amdgcn_permlane32_swap(w[0].x, w[1].x, false, false);
      const auto hi = __builtin_amdgcn_permlane32_swap(w[0].y, w[1].y, false, false);
      if (row < c.Lq) *reinterpret_cast<uint4*>(orow + 32 * dt + 8 * g) = make_uint4(lo[0], hi[0], lo[1], hi[1]);
    }
}

template <int DT, int kG, int kRows>
hipError_t launch(const SmallCall& c, hipStream_t s) {
  // more than 64 KiB of dynamic LDS has to be requested per kernel, once per device
  constexpr int kMaxDevices = 64;
  static std::atomic<bool> requested[kMaxDevices];
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  if (!requested[dev].load(std::memory_order_acquire)) {
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(&sage_small_kernel<DT, kG, kRows>), hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)small_lds(kMaxTiles, kRows));
    if (e != hipSuccess) return e;
    requested[dev].store(true, std::memory_order_release);
  }
  const int n = (c.Lk + kBlkK - 1) / kBlkK;
  sage_small_kernel<DT, kG, kRows><<<dim3((c.Lq + kRows - 1) / kRows, c.Hq, c.B), dim3(kThreads), small_lds(n, kRows), s>>>(c);
  return hipGetLastError();
}

template <int DT, int kG>
hipError_t launch_rows(const SmallCall& c, hipStream_t s) {
  // The fewest rows a workgroup with which there is a compute unit for each: they quantize the same K and V side by side, and
  // what follows is shorter.  us, at least 32 / 64 / 128 / 256 rows: 32 tokens of 2 x 64 heads 5.8 / 6.5 / 7.2 / 7.6, 100 of 16
  // 9.2 / 10.4 / 11.7 / 11.6, 250 of 40 16.4 / 16.5 / 17.3 / 20.5, 200 of 2 x 32 (64 channels) 13.7 / 13.8 / 14.4 / 15.4.
  const auto fits = [&](int rows) { return (int64_t)c.B * c.Hq * ((c.Lq + rows - 1) / rows) <= kComputeUnits; };
  if (fits(32)) return launch<DT, kG, 32>(c, s);
  if (fits(64)) return launch<DT, kG, 64>(c, s);
  if (fits(128)) return launch<DT, kG, 128>(c, s);
  return launch<DT, kG, 256>(c, s);
}

}  // namespace

// One round of the chip: every workgroup quantizes its head's K and V by itself, and beyond that the general path, which does
// it once, is ahead.  us replayed from a graph, general / one launch, on 64, 128, 256 keys: 256 workgroups (64 heads of 1000 rows)
// 18.5 / 15.0, 22.2 / 18.5, 30.0 / 26.8; 264 22.6 / 25.2, 26.2 / 30.8, 34.5 / 44.1; 384 (96 of 1000) 25.1 / 26.3, 28.7 / 33.1, 37.3 / 46.5.
// Two kinds of call beyond the line would still gain, and take the general path: entries of one block each (8 x 64 heads of 250
// rows, 512 workgroups, 35.8 / 29.7, 41.4 / 36.8, 56.0 / 54.9) and 64 channels on few keys (264: 19.3 / 16.9, 21.5 / 21.6, 27.8 / 33.2).
bool small_call_suits(int B, int Hq, int Lq, int Lk) { return Lk <= kMeanChunk && (int64_t)B * Hq * ((Lq + 255) / 256) <= kComputeUnits; }

hipError_t launch_small(const SmallCall& call, hipStream_t s) {
  SmallCall c = call;
  c.group = c.Hq / c.Hkv;
  c.group_magic = c.group > 1 ? (unsigned)(((1ull << 32) + c.group - 1) / c.group) : 0;  // exact below 2^32 / group
  const bool bf16 = c.o.dtype == KSANA_SAGE_BF16;
  if (c.d_out <= 64) return bf16 ? launch_rows<KSANA_SAGE_BF16, 2>(c, s) : launch_rows<KSANA_SAGE_FP16, 2>(c, s);
  return bf16 ? launch_rows<KSANA_SAGE_BF16, 4>(c, s) : launch_rows<KSANA_SAGE_FP16, 4>(c, s);
}

}  // namespace ksana_sage
