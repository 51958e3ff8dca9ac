// Few keys, many query rows (video tokens on a prompt): the head's quantized K and V^T stay in LDS, 16 KiB per 64 keys, and
// the query rows stream past them.
//
// One workgroup per compute unit, 8 waves.  It brings in a head's tiles once and takes a part of the head's blocks of 32 query
// rows; its waves take the part's blocks in turn - each quantizes its rows, walks the tiles, writes its results - and never
// meet again.  Nothing is copied or awaited in a block but its own rows, which are requested while the block before ends.
//
// The general kernel spends 8.6 of a workgroup's 18.3 us at 512 keys on its set-up - rows, tiles, Q's transform - with one
// other workgroup on the unit to hide it.  Here the waves of a SIMD drift apart and hide each other's; bound by the vector
// instructions of the softmax and of Q's transform.
//
// Operations, orders and roundings are the general kernel's, and so are the bits.
#include "sage_attn_device.h"

#include <algorithm>
#include <atomic>
#include <type_traits>

#include "../../include/ksana_sage_hip.h"

namespace ksana_sage {
namespace {

constexpr int kComputeUnits = 256;  // a workgroup each
constexpr int kWaves = 8, kMaxTiles = 8, kRows = 32;
constexpr int kScalesAt = 2 * kMaxTiles * kTileBytes;              // V scales, V means (128 floats each), K scales
constexpr int kLds = kScalesAt + (2 * kD + kMaxTiles + 4) * 4;     // .. and the next block's number: 132 144 bytes

// a wave-uniform address, in scalar registers wherever it was worked out
__device__ __forceinline__ const uint8_t* scalar(const uint8_t* at) {
  const uint64_t a = reinterpret_cast<uint64_t>(at);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a), hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
  return reinterpret_cast<const uint8_t*>((uint64_t)hi << 32 | lo);
}

// A place in LDS of this lane's own as one register, to which only constants are added: in 128 KiB the tiles lie beyond the 64 KiB
// that an instruction's offset reaches, and left to itself the compiler keeps an address for every constant (39 registers, 18 of
// them in scratch memory, read back behind the next block's rows, and eight additions per two steps).  us, before / with it: 40
// heads of 32760 rows on 512 keys 305.1 / 303.5, of 75600 677.9 / 672.2, 2 x 24 of 20000 on 333 203.5 / 201.4.
typedef const __attribute__((address_space(3))) uint8_t* LdsBytes;
__device__ __forceinline__ LdsBytes own_place(const uint8_t* at) {
  LdsBytes lds = (LdsBytes)at;
  pin(lds);
  return lds;
}
template <typename T>
__device__ __forceinline__ T lds_read(LdsBytes at) {
  return *reinterpret_cast<const __attribute__((address_space(3))) T*>(at);
}

// n_blk: blocks of 32 rows per (batch, head); parts: workgroups per (batch, head)
template <int DT, int kG>
__global__ __launch_bounds__(kWaves * 64, 1) void sage_resident_kernel(const AttnParams p, int n_blk, int parts, int n_wg) {
  want(p.q_rows.ptr, p.k_tiles, p.o.sH, p.k_lens, n_blk);
  constexpr int kMagicBits = kG == 4 ? kMagicI : kMagicI2;
  constexpr float kMagicVal = kG == 4 ? kMagicF : kMagicF2;
  // consecutive workgroups land on consecutive XCDs: each XCD gets a run of them, whose heads share its L2
  const int wg = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  if (wg >= n_wg) return;
  const int bh = __builtin_amdgcn_readfirstlane(wg / parts), part = wg - bh * parts;
  const int per = n_blk / parts, more = n_blk - per * parts;  // the first `more` parts have one block more
  const int blk0 = part * per + min(part, more), n_here = per + (part < more ? 1 : 0);

  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  float* s_vs = reinterpret_cast<float*>(smem + kScalesAt);
  float* s_ks = s_vs + 2 * kD;
  int* s_next = reinterpret_cast<int*>(s_ks + kMaxTiles);
  const LdsBytes my_k = own_place(smem + lane * 16);                           // this lane's pieces of K tile 0 ..
  const LdsBytes my_v = own_place(smem + kMaxTiles * kTileBytes + lane * 16);  // .. and of V^T tile 0

  const int b = __builtin_amdgcn_readfirstlane(bh / p.Hq), h = bh - b * p.Hq;
  const int bhk = __builtin_amdgcn_readfirstlane(b * p.Hkv + h / (p.Hq / p.Hkv));
  const int n_tiles = (p.Lk + kBlkK - 1) / kBlkK;
  const int n_last = p.Lk & (kBlkK - 1), tail = n_last != 0 ? n_tiles - 1 : -1;  // a ragged last tile: its keys, its number
  uint16_t* obase = p.o.ptr + b * p.o.sB + h * p.o.sH + 8 * hh;

  const uint16_t* qbase = p.q_rows.ptr + b * p.q_rows.sB + h * p.q_rows.sH + 16 * hh;
  uint4 raw[8];
  auto request = [&](int i) {  // the rows of block i of this part (past the part's end: some block's, not used)
    const uint16_t* qrow = qbase + (int64_t)min((blk0 + min(i, n_here - 1)) * kRows + l32, p.Lq - 1) * p.q_rows.sL;
#pragma unroll
    for (int s = 0; s < kG; ++s) {
      raw[2 * s] = *reinterpret_cast<const uint4*>(qrow + 32 * s);
      raw[2 * s + 1] = *reinterpret_cast<const uint4*>(qrow + 32 * s + 8);
    }
  };

  float vsm = 0.0f, ksm = 0.0f;
  if (tid < 2 * kD) vsm = tid < kD ? p.v_scale[(int64_t)bhk * kD + tid] : p.v_mean[(int64_t)bhk * kD + tid - kD];
  if (tid < n_tiles) ksm = p.k_scale[(int64_t)bhk * p.nkb + tid];
  const uint8_t* k_src = scalar(reinterpret_cast<const uint8_t*>(p.k_tiles) + (int64_t)bhk * p.nkb * kTileBytes);
  const uint8_t* v_src = scalar(p.v_tiles + (int64_t)bhk * p.nkb * kTileBytes);
  for (int j = 0; j < n_tiles; ++j) {  // a wave moves 1 KiB of each tile
    const unsigned off = (unsigned)(j * kTileBytes + wave * 1024 + lane * 16);
    lds_copy16(k_src, off, smem + j * kTileBytes + wave * 1024);
    lds_copy16(v_src, off, smem + (kMaxTiles + j) * kTileBytes + wave * 1024);
  }
  request(wave);
  if (tid < 2 * kD) s_vs[tid] = vsm;
  if (tid < kMaxTiles) s_ks[tid] = ksm;
  if (tid == 0) *s_next = kWaves;
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  const float2 mm = reinterpret_cast<const float2*>(s_vs + kD)[lane];
  const bool has_mean = __any(mm.x != 0.0f || mm.y != 0.0f);

  for (int i = wave, next; i < n_here; i = next) {
    // Blocks go to whichever wave is free: of the two on a SIMD the older one gets ahead, and with a fixed share each the
    // younger ones were alone on the chip for the last fifth of the time.
    next = 0;
    if (lane == 0) next = atomicAdd(s_next, 1);
    next = __builtin_amdgcn_readfirstlane(next);
    const int q0 = (blk0 + i) * kRows, row = q0 + l32;
    if (q0 + kRows > p.Lq) {  // (uniform) rows that do not exist count as zeros
#pragma unroll
      for (int s = 0; s < 2 * kG; ++s) raw[s] = row < p.Lq ? raw[s] : make_uint4(0, 0, 0, 0);
    }
    v4i qf[4];
    float qs = 0.0f;
#pragma unroll
    for (int s = 0; s < 4; ++s) qf[s] = v4i{0, 0, 0, 0};
    quant_q_rows<DT, kG>(raw, p.q_premul, qf, qs);
    v8i ones;  // the row sums' operand, see the general kernel
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      int one4 = ((lane >> 2) & 1) == ((lane >> 4) & 1) ? 0x38383838 : 0;
      pin(one4);
      ones[r] = one4;
    }
    v16i magic;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      int m = kMagicBits;
      pin(m);
      magic[r] = m;
    }

    v16f oacc[4];
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) oacc[dt][r] = 0.0f;
    v4f lacc = {0.0f, 0.0f, 0.0f, 0.0f};
    float m_run = -INFINITY, x_base = -INFINITY, x_limit = -INFINITY;
    auto scale_o = [&](float alpha) {
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[dt][r] *= alpha;
      lacc[0] *= alpha;
    };
    // the coming tile's scale and exponent constant; the factors the point moves of even and of odd tiles put on everything
    // before them, and whether there is one
    float sc = 0.0f, xc = 0.0f, alpha_even = 1.0f, alpha_odd = 1.0f;
    int moved_even = 0, moved_odd = 0;
    auto look_ahead = [&](int jn, int mx, float ks, float& alpha, int& moved) {
      sc = qs * ks;
      float mneg = -kMagicVal * sc;
      const float m_half = __builtin_fmaf(__int_as_float(mx), sc, mneg);
      moved = 0;
      if (__ballot(!(m_half <= x_limit)) != 0 && jn < n_tiles) {
        alpha = move_point(mx, sc, mneg, qs, m_run, x_base, x_limit);
        moved = 1;
      }
      xc = x_base + mneg;
    };
    auto p_of = [&](int acc_bits) { return fast_exp2(__builtin_fmaf(__int_as_float(acc_bits), sc, xc)); };
    auto k_frag = [&](LdsBytes tile, int i8) { return lds_read<v4i>(tile + ((i8 & 1) * 4 + (i8 >> 1)) * 1024); };
    auto v_frag = [&](LdsBytes tile, int dt) {
      const v4i lo = lds_read<v4i>(tile + dt * 2048);
      const v4i hi = lds_read<v4i>(tile + dt * 2048 + 1024);
      return v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };
    auto has_qk = [](int i8) { return i8 >= 0 && i8 < 8 && (i8 >> 1) < kG; };

    // One tile per step: its probabilities on the vector unit, under the matrix instructions of the next tile's scores
    // (of some tile's, not used, in the last step) and of the previous tile's values (times no probabilities, in the first).
    // alpha, moved: tile j - 1's on the way in, tile j + 1's on the way out.
    auto step = [&](int j, v16i (&s_cur)[2], v16i (&s_nxt)[2], const v8i& pf_prev, v8i& pf, float& alpha, int& moved) {
      const int nxt = min(j + 1, n_tiles - 1);
      LdsBytes kst = my_k + nxt * kTileBytes, vst = my_v + max(j - 1, 0) * kTileBytes;
      pin(kst), pin(vst);
      v4i kf[4];
      v8i vf[4];
      kf[0] = k_frag(kst, 0), kf[1] = k_frag(kst, 1), kf[2] = k_frag(kst, 2);
      const float ks_nxt = s_ks[nxt];
      if (moved != 0) scale_o(alpha);  // wave-uniform
      lacc = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(ones, pf_prev, lacc, 0, 0, 0, 0, 0, 0);
      __builtin_amdgcn_s_setprio(1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        if (c + 3 < 8) {
          if (has_qk(c + 3)) kf[(c + 3) & 3] = k_frag(kst, c + 3);
        } else if (c + 3 - 8 < kG) {
          vf[c + 3 - 8] = v_frag(vst, c + 3 - 8);
        }
        if (has_qk(c)) s_nxt[c & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(kf[c & 3], qf[c >> 1], (c >> 1) == 0 ? magic : s_nxt[c & 1], 0, 0, 0);
        const float e0 = p_of(s_cur[0][2 * c]), e1 = p_of(s_cur[0][2 * c + 1]);
        if (c & 1) {
          int w = __builtin_amdgcn_cvt_pk_fp8_f32(e0, e1, pf[c >> 1], true);
          pin(w);
          pf[c >> 1] = w;
        } else {
          pf[c >> 1] = __builtin_amdgcn_cvt_pk_fp8_f32(e0, e1, __float_as_int(e0), false);  // both halves get written
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if (j + 1 == tail) blank_scores<kMagicBits>(s_nxt, hh, n_last);
      __builtin_amdgcn_s_setprio(0);
      int mx = 0;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) {
        if (dt == 0 && kG == 4) vf[3] = v_frag(vst, 3);
        if (dt < kG) oacc[dt] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(vf[dt], pf_prev, oacc[dt], 0, 0, 0, 0, 0, 0);
        const float e0 = p_of(s_cur[1][4 * dt]), e1 = p_of(s_cur[1][4 * dt + 1]);
        const float e2 = p_of(s_cur[1][4 * dt + 2]), e3 = p_of(s_cur[1][4 * dt + 3]);
        int w = __builtin_amdgcn_cvt_pk_fp8_f32(e0, e1, __float_as_int(e0), false);
        w = __builtin_amdgcn_cvt_pk_fp8_f32(e2, e3, w, true);
        pin(w);
        pf[4 + dt] = w;
        const v16i& blk = s_nxt[dt >> 1];
        const int r0 = (dt & 1) * 8;
        mx = dt == 0 ? max(blk[0], blk[1]) : max(max(mx, blk[r0]), blk[r0 + 1]);
        mx = max(max(mx, blk[r0 + 2]), blk[r0 + 3]);
        mx = max(max(mx, blk[r0 + 4]), blk[r0 + 5]);
        mx = max(max(mx, blk[r0 + 6]), blk[r0 + 7]);
        pin(mx);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (j == tail) blank_probs(pf, hh, n_last);
      look_ahead(j + 1, mx, ks_nxt, alpha, moved);
    };
    v16i s_a[2], s_b[2];
    v8i pf_x = {0, 0, 0, 0, 0, 0, 0, 0}, pf_y = {0, 0, 0, 0, 0, 0, 0, 0};
    qk_tile<kG>(smem, lane, qf, magic, s_a);
    if (tail == 0) blank_scores<kMagicBits>(s_a, hh, n_last);
    {
      int mx = s_a[0][0];
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = max(mx, s_a[u][r]);
      look_ahead(0, mx, s_ks[0], alpha_even, moved_even);
      moved_even = __any(alpha_even != alpha_even);  // nothing has been accumulated yet: only a NaN has anything to say
    }
    int j = 0;
#pragma unroll 1
    for (; j + 2 <= n_tiles; j += 2) {
      step(j, s_a, s_b, pf_x, pf_y, alpha_odd, moved_odd);
      step(j + 1, s_b, s_a, pf_y, pf_x, alpha_even, moved_even);
    }
    if (j < n_tiles) step(j, s_a, s_b, pf_x, pf_y, alpha_odd, moved_odd);
    request(next);  // (the scores' registers are free by now)
    {  // the last tile's values
      const bool odd = (n_tiles & 1) != 0;
      if (odd ? moved_even != 0 : moved_odd != 0) scale_o(odd ? alpha_even : alpha_odd);
      const v8i pf_last = odd ? pf_y : pf_x;
      LdsBytes vst = my_v + (n_tiles - 1) * kTileBytes;
      pin(vst);  // (not an address per piece over the whole loop)
      lacc = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(ones, pf_last, lacc, 0, 0, 0, 0, 0, 0);
#pragma unroll
      for (int dt = 0; dt < kG; ++dt)
        oacc[dt] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(v_frag(vst, dt), pf_last, oacc[dt], 0, 0, 0, 0, 0, 0);
    }

    // O = O^T / rowsum * v_scale (+ the V mean).  A lane has channels 32 dt + 8 g + 4 hh .. + 3 of its row; lanes l and l + 32
    // trade every second four, so that each stores eight in a row.  (Staged through LDS for whole 256-byte rows they
    // would need room that the tiles hold; the L2 puts a row's pieces together.)
    const float inv_l = 1.0f / lacc[0];
    const float keep_mean = inv_l != 0.0f ? 1.0f : 0.0f;
    uint16_t* orow = obase + (int64_t)row * p.o.sL;
    const LdsBytes scales = own_place(smem + kScalesAt + 16 * hh);
    auto store = [&](auto with_mean) {
#pragma unroll
      for (int dt = 0; dt < kG; ++dt)
#pragma unroll
        for (int g = 0; g < 4; g += 2) {
          uint2 w[2];
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const int r = 4 * (g + e), d = 32 * dt + 8 * (g + e);
            const v4f s4 = lds_read<v4f>(scales + 4 * d);
            float o4[4] = {oacc[dt][r] * inv_l * s4[0], oacc[dt][r + 1] * inv_l * s4[1], oacc[dt][r + 2] * inv_l * s4[2], oacc[dt][r + 3] * inv_l * s4[3]};
            if constexpr (decltype(with_mean)::value) {
              const v4f m4 = lds_read<v4f>(scales + 4 * (kD + d));
#pragma unroll
              for (int c = 0; c < 4; ++c) o4[c] += m4[c] * keep_mean;
            }
            // (pinned: the last operation and the conversion may otherwise become one fp16 instruction with a single rounding)
#pragma unroll
            for (int c = 0; c < 4; ++c) pin(o4[c]);
            w[e] = half4<DT>(o4[0], o4[1], o4[2], o4[3]);
          }
          const auto x = __builtin_amdgcn_permlane32_swap(w[0].x, w[1].x, false, false);
          const auto y = __builtin_amdgcn_permlane32_swap(w[0].y, w[1].y, false, false);
          *reinterpret_cast<uint4*>(orow + 32 * dt + 8 * g) = make_uint4(x[0], y[0], x[1], y[1]);
        }
    };
    if (row < p.Lq) {
      if (has_mean) store(std::integral_constant<bool, true>{});
      else store(std::integral_constant<bool, false>{});
    }
  }
}

// Workgroups per (batch, head).  A round of the chip takes as long as its largest part, and about eight blocks' time more: the
// tiles are brought in before its first block, and its waves end one after the other.
int resident_parts(int pairs, int n_blk) {
  int best = 1;
  int64_t best_cost = INT64_MAX;
  for (int rounds = 1; rounds <= 8; ++rounds) {
    const int parts = std::min(n_blk, std::max(1, rounds * kComputeUnits / pairs));
    const int64_t cost = (((int64_t)pairs * parts + kComputeUnits - 1) / kComputeUnits) * ((n_blk + parts - 1) / parts + kWaves);
    if (cost < best_cost) best = parts, best_cost = cost;
  }
  return best;
}

template <int DT, int kG>
hipError_t launch(const AttnParams& p, hipStream_t s) {
  // more than 64 KiB of dynamic LDS has to be requested per kernel, once per device
  constexpr int kMaxDevices = 64;
  static std::atomic<bool> requested[kMaxDevices];
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  if (!requested[dev].load(std::memory_order_acquire)) {
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(&sage_resident_kernel<DT, kG>), hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    if (e != hipSuccess) return e;
    requested[dev].store(true, std::memory_order_release);
  }
  const int n_blk = (p.Lq + kRows - 1) / kRows, pairs = p.B * p.Hq;
  const int parts = resident_parts(pairs, n_blk), n_wg = pairs * parts;
  sage_resident_kernel<DT, kG><<<dim3((n_wg + 7) / 8 * 8), dim3(kWaves * 64), kLds, s>>>(p, n_blk, parts, n_wg);
  return hipGetLastError();
}

}  // namespace

// From where filling LDS and the waves' uneven ends are small next to the blocks.  us per call, general kernel / this: 16384 blocks
// and more - 40 heads of 32760 rows on 512 keys 339 / 317, 2 x 40 on 320 keys 541 / 501, 24 of 75600 on 512 465 / 425, 16 of 38734
// on 192 141 / 116, 2 x 64 of 5000 on 77 146 / 106; fewer, up to 256 keys (Q is otherwise quantized apart there): 40 of 8190 on 77
// 63.6 / 60.2, 2 x 64 of 2700 on 192 78.8 / 68.5; but 40 of 4096 (5120 blocks) on 77 37.7 / 40.2, and beyond 256 keys 40 of 8190
// on 512 88.6 / 90.1, 100 of 4096 on 320 93.9 / 98.0.  (Not for batches with lengths of their own: 3 x 40 heads of 2776 rows on up to
// 463 keys 83 / 113.)
bool resident_call_suits(const AttnParams& p) {
  if (p.block_mask != nullptr || p.causal || p.q_lens != nullptr || p.k_lens != nullptr || !p.exact_exp2 || p.tile_skip || p.wg_waves != 0) return false;
  const int64_t blocks = (int64_t)p.B * p.Hq * ((p.Lq + kRows - 1) / kRows);
  return p.Lk <= kMaxTiles * kBlkK && p.Lq >= 1024 && blocks >= (p.Lk <= kMeanChunk ? 4 : 8) * kWaves * kComputeUnits;
}

hipError_t launch_resident(const AttnParams& p, hipStream_t s) {
  const bool bf16 = p.o.dtype == KSANA_SAGE_BF16;
  if (p.d_out <= 64) return bf16 ? launch<KSANA_SAGE_BF16, 2>(p, s) : launch<KSANA_SAGE_FP16, 2>(p, s);
  return bf16 ? launch<KSANA_SAGE_BF16, 4>(p, s) : launch<KSANA_SAGE_FP16, 4>(p, s);
}

}  // namespace ksana_sage
