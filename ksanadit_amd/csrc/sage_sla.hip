// The linear-attention branch of the sparse-linear ("SLA") backend for gfx950 (MI355X).
//
// Per (batch, head), with phi = softmax over the 128 channels of a row, rounded to the tensors' half type:
//   kv   = sum_l phi(k_l)^T v_l            [128 x 128]
//   ksum = sum_l phi(k_l)                  [128]
//   o_l  = (phi(q_l) kv) / (1e-5 + phi(q_l) . ksum)
// and, where the caller's projection is a plain linear layer, o_l W^T + bias folded in as phi(q_l) (kv W^T) / (...) +
// bias, plus an optional tensor added on the way out (the sparse branch's result).  This is calc_linear and what
// surrounds it in ksana/operations/attention/backends/sage_sla.py:135-139, 273-287 - there five library kernels over
// [B, H, L, D] intermediates, here one pass over k and v, a small finalisation, and one pass over q.
//
//   sla_kv_partial_kernel   reads k and v once; bf16 / fp16 MFMA; one partial kv and ksum per run of rows
//   sla_kv_finalize_kernel  adds the runs in order (repeatable bits), rounds to the half type as the reference's
//                           tensors are, multiplies by W^T, stores the matrix in MFMA operand order
//   sla_apply_kernel        reads q once, writes the result in [B, L, H, D]
#include "sage_sla_device.h"

#include <atomic>

#include "../../include/ksana_sage_hip.h"

namespace ksana_sage {
namespace {

template <int DT>
__global__ __launch_bounds__(kSlaThreads, 2) void sla_kv_partial_kernel(const InTensor k, const InTensor v, int H, int L, int rows_per_run,
                                                                        float* __restrict__ part) {
  sla_kv_run<DT, false>(blockIdx.x, gridDim.x, blockIdx.y, blockIdx.z, k.ptr, k.sB, k.sL, k.sH, v.ptr, v.sB, v.sL, v.sH, H, L, rows_per_run,
                        part, nullptr, nullptr, 0);
}

// the same with the quantizers' statistics of k and v
template <int DT>
__global__ __launch_bounds__(kSlaThreads, 2) void sla_kv_stats_kernel(const InTensor k, const InTensor v, int H, int L, int rows_per_run,
                                                                      float* __restrict__ part, float* __restrict__ k_part,
                                                                      float* __restrict__ v_part, int nch) {
  sla_kv_run<DT, true>(blockIdx.x, gridDim.x, blockIdx.y, blockIdx.z, k.ptr, k.sB, k.sL, k.sH, v.ptr, v.sB, v.sL, v.sH, H, L, rows_per_run,
                       part, k_part, v_part, nch);
}

// grid = (8, B * H)
template <int DT>
__global__ __launch_bounds__(kSlaThreads) void sla_kv_finalize_kernel(const float* __restrict__ part, int runs,
                                                                      const float* __restrict__ proj_w, uint16_t* __restrict__ m_frag,
                                                                      float* __restrict__ ksum) {
  sla_kv_finalize<DT>(blockIdx.x, blockIdx.y, part, runs, proj_w, m_frag, ksum);
}

// ---------------------------------------------------------------------------------------------------------------
// out[b, l, h, :] = (phi(q_l) M) / (1e-5 + phi(q_l) . ksum) + bias (+ add[b, l, h, :]).
// grid = (ceil(L / (128 * blocks)), H, B), 256 threads; a workgroup stages M (32 KiB) in LDS once and walks `blocks`
// blocks of 128 rows, 32 per wave.  Lane (row = lane % 32, g = lane / 32) loads the channels 16 s + 8 g .. + 7 of its
// row, s = 0 .. 7 - half of the row, exactly its B operands of the 32x32x16 instruction (contraction over channels);
// the other half sits in lane + 32.  The product is taken transposed, out^T = M^T phi(q)^T, so that a lane ends up
// with channels of ONE row; the rows leave through LDS as whole 256-byte rows, 16 bytes per lane.
// ---------------------------------------------------------------------------------------------------------------
constexpr int kApplyPitch = 2 * kD + 16;
constexpr int kApplyLds = kD * kD * 2 + 2 * kD * 4 + 4 * 32 * kApplyPitch;  // 68 608 bytes

template <int DT>
__global__ __launch_bounds__(kSlaThreads, 2) void sla_apply_kernel(const uint16_t* __restrict__ q, int64_t qsB, int64_t qsL,
                                                                   int64_t qsH, const uint16_t* __restrict__ m_frag,
                                                                   const float* __restrict__ ksum,
                                                                   const float* __restrict__ bias,
                                                                   const uint16_t* __restrict__ add, int64_t asB, int64_t asL,
                                                                   int64_t asH, uint16_t* __restrict__ out, int64_t osB,
                                                                   int64_t osL, int64_t osH, int H, int L, int blocks) {
  const int h = blockIdx.y, b = blockIdx.z, bh = b * H + h;
  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int l32 = lane & 31, g = lane >> 5;
  // dynamic LDS (kApplyLds bytes): M in operand order, ksum, bias, then one staging area per wave
  extern __shared__ __attribute__((aligned(16))) uint8_t s_dyn[];
  uint4* s_m = reinterpret_cast<uint4*>(s_dyn);
  float* s_ks = reinterpret_cast<float*>(s_dyn + kD * kD * 2);
  float* s_bias = s_ks + kD;
  constexpr int kPitch = kApplyPitch;  // bytes per staged row
  uint8_t* s_stage = s_dyn + kD * kD * 2 + 2 * kD * 4;
  {
    const uint4* src = reinterpret_cast<const uint4*>(m_frag + (int64_t)bh * kD * kD);
#pragma unroll
    for (int i = 0; i < 8; ++i) s_m[i * kSlaThreads + t] = src[i * kSlaThreads + t];
    if (t < kD) {
      s_ks[t] = ksum[bh * kD + t];
      s_bias[t] = bias != nullptr ? bias[t] : 0.0f;
    }
  }
  __syncthreads();
  uint8_t* stage = s_stage + w * (32 * kPitch);
  for (int blk = 0; blk < blocks; ++blk) {
    const int r0 = (blockIdx.x * blocks + blk) * 128 + 32 * w;
    if (r0 >= L) break;  // wave-uniform
    const int row = r0 + l32;
    const uint16_t* qr = q + b * qsB + (int64_t)row * qsL + h * qsH + 8 * g;
    uint4 raw[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) raw[s] = row < L ? *reinterpret_cast<const uint4*>(qr + 16 * s) : make_uint4(0, 0, 0, 0);
    // the pieces of `add` this lane will meet in the output loop below, requested now: they arrive under the
    // arithmetic instead of being waited for one by one between a load and its store
    uint16_t* ob = out + b * osB + h * osH;
    const uint16_t* ab = add != nullptr ? add + b * asB + h * asH : nullptr;
    uint4 other[8];
    if (ab != nullptr) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int idx = i * 64 + lane, r = idx >> 4, cc = idx & 15;
        other[i] = r0 + r < L ? *reinterpret_cast<const uint4*>(ab + (int64_t)(r0 + r) * asL + 8 * cc) : make_uint4(0, 0, 0, 0);
      }
    }
    float x[8][8];
    const float inv = sla_row_exps<DT>(raw, x);
    uint4 fq[8];
    const float scale = sla_row_scale<DT>(x, inv, s_ks, g, fq);
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
      const v16f acc = sla_row_product<DT>(s_m, fq, nt, lane);
      // register r: output channel 32 nt + 8 (r / 4) + 4 g + r % 4 of row l32
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const int n = 32 * nt + 8 * q4 + 4 * g;
        const float4 bs = *reinterpret_cast<const float4*>(s_bias + n);
        const uint32_t lo = pack2<DT>(__builtin_fmaf(acc[4 * q4 + 0], scale, bs.x), __builtin_fmaf(acc[4 * q4 + 1], scale, bs.y));
        const uint32_t hi = pack2<DT>(__builtin_fmaf(acc[4 * q4 + 2], scale, bs.z), __builtin_fmaf(acc[4 * q4 + 3], scale, bs.w));
        *reinterpret_cast<uint2*>(stage + l32 * kPitch + 2 * n) = make_uint2(lo, hi);
      }
    }
    // LDS serves one wave's accesses in order: the reads below see the writes above
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int idx = i * 64 + lane, r = idx >> 4, cc = idx & 15;  // row r of the wave, 16-byte piece cc of it
      uint4 piece = *reinterpret_cast<const uint4*>(stage + r * kPitch + 16 * cc);
      if (r0 + r < L) {
        if (ab != nullptr) {
          float a8[8], o8[8];
          widen8<DT>(piece, a8);
          widen8<DT>(other[i], o8);
          piece = make_uint4(pack2<DT>(a8[0] + o8[0], a8[1] + o8[1]), pack2<DT>(a8[2] + o8[2], a8[3] + o8[3]),
                             pack2<DT>(a8[4] + o8[4], a8[5] + o8[5]), pack2<DT>(a8[6] + o8[6], a8[7] + o8[7]));
        }
        *reinterpret_cast<uint4*>(ob + (int64_t)(r0 + r) * osL + 8 * cc) = piece;
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------------------------
// The block map from the pooled blocks (get_block_map, sage_sla.py:83-90): score = pooled_q pooled_k^T as a tensor of
// the half type (fp32 accumulation, one rounding), then for every query block the `keep` key blocks with the largest
// scores get a one, the others a zero; of equal scores the lower index wins (what a stable descending sort gives;
// torch.topk leaves it open).  grid = (ceil(nq / 32), B * H), 1024 threads; dynamic LDS 32 * nk_pad * 2 bytes.
//
// Bound by the length of the selection, a chain of counts: hence sixteen waves with two query blocks each, not four with
// eight, and registers for 512 key blocks where there are no more (40 heads of 256 x 512 blocks: 59 -> 37 us).
//
// Scores: 32 query blocks x 32 key blocks per 32x32x16 matrix instruction, contraction over the 128 channels - both
// operands are 16-byte pieces of pooled rows as they lie in memory; wave w takes the key tiles w, w + 16, ...  Each
// score goes to LDS as a 16-bit key whose unsigned order is the order of the values.  Selection, one wave per 2 query
// blocks: the keep-th largest key by bisection over its 16 bits (count of keys >= candidate by ballots), then ones for
// the keys above it and for as many of its equals, lowest index first, as are still missing.
// ---------------------------------------------------------------------------------------------------------------
constexpr int kMapMaxKeyBlocks = 1024;
constexpr int kMapThreads = 1024, kMapWaves = kMapThreads / 64;

// kPerLane: 64 * kPerLane key blocks at most
template <int DT, int kPerLane>
__global__ __launch_bounds__(kMapThreads) void sla_block_map_kernel(const uint16_t* __restrict__ pooled_q,
                                                                    const uint16_t* __restrict__ pooled_k, int nq, int nk,
                                                                    int nk_pad, int keep, int8_t* __restrict__ block_map) {
  extern __shared__ __attribute__((aligned(16))) uint8_t s_dyn[];
  uint16_t* s_key = reinterpret_cast<uint16_t*>(s_dyn);  // [32][nk_pad]
  const int bh = blockIdx.y, q0 = blockIdx.x * 32;
  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int l32 = lane & 31, g = lane >> 5;
  const uint16_t* pq = pooled_q + ((int64_t)bh * nq + q0 + l32) * kD + 8 * g;
  const uint16_t* pk = pooled_k + (int64_t)bh * nk * kD + 8 * g;
  uint4 a[8];
#pragma unroll
  for (int s = 0; s < 8; ++s) a[s] = q0 + l32 < nq ? *reinterpret_cast<const uint4*>(pq + 16 * s) : make_uint4(0, 0, 0, 0);
  for (int nt = w; nt * 32 < nk_pad; nt += kMapWaves) {
    const int kb = nt * 32 + l32;
    uint4 b[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) b[s] = kb < nk ? *reinterpret_cast<const uint4*>(pk + (int64_t)kb * kD + 16 * s) : make_uint4(0, 0, 0, 0);
    v16f acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
#pragma unroll
    for (int s = 0; s < 8; ++s) acc = mfma32<DT>(a[s], b[s], acc);
    // register r: query block 8 (r / 4) + 4 g + r % 4 of the group, key block kb
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int m = 8 * (r >> 2) + 4 * g + (r & 3);
      uint32_t bits;
      if constexpr (DT == KSANA_SAGE_BF16)
        bits = __builtin_bit_cast(uint16_t, (__bf16)acc[r]);
      else
        bits = __builtin_bit_cast(uint16_t, (_Float16)acc[r]);
      const uint32_t key = (bits & 0x8000u) ? (~bits & 0xffffu) : (bits | 0x8000u);  // unsigned order = value order
      s_key[m * nk_pad + kb] = (uint16_t)(kb < nk ? key : 0u);                    // padding sorts below everything
    }
  }
  __syncthreads();
  // a row's keys in registers: lane holds the keys lane + 64 i (0, the padding value, beyond nk)
  constexpr int kRowsPerWave = 32 / kMapWaves;
  for (int mi = 0; mi < kRowsPerWave; ++mi) {
    const int m = kRowsPerWave * w + mi;
    if (q0 + m >= nq) break;  // wave-uniform
    const uint16_t* row = s_key + m * nk_pad;
    int8_t* out = block_map + ((int64_t)bh * nq + q0 + m) * nk;
    uint32_t key[kPerLane];
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) key[i] = lane + 64 * i < nk ? row[lane + 64 * i] : 0u;
    uint32_t thr = 0;
    if (keep > 0 && keep < nk) {
      for (int bit = 15; bit >= 0; --bit) {
        const uint32_t cand = thr | (1u << bit);
        int count = 0;
#pragma unroll
        for (int i = 0; i < kPerLane; ++i) count += __popcll(__ballot(key[i] >= cand));  // padding keys are 0 < cand
        if (count >= keep) thr = cand;  // uniform
      }
    }
    int above = 0;
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) above += __popcll(__ballot(key[i] > thr));
    int missing = keep >= nk ? nk : (keep <= 0 ? 0 : keep - above);  // of the keys equal to thr, lowest index first
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) {
      const int idx = lane + 64 * i;
      const bool in = idx < nk;
      const bool eq = in && key[i] == thr;
      const unsigned long long bal = __ballot(eq);
      const int rank = __builtin_amdgcn_mbcnt_hi((unsigned)(bal >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)bal, 0));
      const bool one = in && keep > 0 && (keep >= nk || key[i] > thr || (eq && rank < missing));
      if (in) out[idx] = one ? 1 : 0;
      missing -= __popcll(bal);
    }
  }
}

}  // namespace

// rows per run of sla_kv_partial_kernel, runs a multiple of 256 rows: as many runs per head as keep the whole grid
// within the 512 workgroups the chip holds at once (two per compute unit, 64 KiB of LDS each) - a few workgroups
// more than that and the launch takes two rounds for one round's work (520 workgroups: 212 us; 480: see profiles)
void plan_sla_runs(int B, int H, int L, int* runs, int* rows_per_run) {
  const int steps = (L + kSlaStepRows - 1) / kSlaStepRows;
  int n = 512 / max(1, B * H);
  n = max(1, min(n, steps));
  const int steps_per_run = (steps + n - 1) / n;
  *rows_per_run = steps_per_run * kSlaStepRows;
  *runs = (steps + steps_per_run - 1) / steps_per_run;
}

hipError_t launch_sla_kv_stats(const InTensor& k, const InTensor& v, int B, int H, int L, float* part, float* k_part, float* v_part, int nch,
                               hipStream_t s) {
  int runs = 1, rows_per_run = L;
  plan_sla_runs(B, H, L, &runs, &rows_per_run);
  const dim3 grid(runs, H, B), block(kSlaThreads);
  if (k.dtype == KSANA_SAGE_BF16)
    sla_kv_stats_kernel<KSANA_SAGE_BF16><<<grid, block, 0, s>>>(k, v, H, L, rows_per_run, part, k_part, v_part, nch);
  else
    sla_kv_stats_kernel<KSANA_SAGE_FP16><<<grid, block, 0, s>>>(k, v, H, L, rows_per_run, part, k_part, v_part, nch);
  return hipGetLastError();
}

// the second pass; add: nullptr, or what the result is added to (may be out itself)
hipError_t launch_sla_apply(const InTensor& q, int B, int H, int L, const float* proj_b, const InTensor* add, const OutTensor& out,
                            const uint16_t* m_frag, const float* ksum, hipStream_t s) {
  const dim3 block(kSlaThreads);
  constexpr int kBlocks = 4;  // 128-row blocks per workgroup of the second pass (M is staged once per workgroup)
  const dim3 grid_apply(((L + 127) / 128 + kBlocks - 1) / kBlocks, H, B);
  {  // more than 64 KiB of dynamic LDS has to be requested per kernel, once per device
    static std::atomic<bool> requested[64];
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= 64) return hipErrorInvalidDevice;
    if (!requested[dev].load(std::memory_order_acquire)) {
      e = hipFuncSetAttribute(reinterpret_cast<const void*>(&sla_apply_kernel<KSANA_SAGE_BF16>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, kApplyLds);
      if (e == hipSuccess)
        e = hipFuncSetAttribute(reinterpret_cast<const void*>(&sla_apply_kernel<KSANA_SAGE_FP16>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, kApplyLds);
      if (e != hipSuccess) return e;
      requested[dev].store(true, std::memory_order_release);
    }
  }
  const uint16_t* add_ptr = add != nullptr ? add->ptr : nullptr;
  const int64_t asB = add ? add->sB : 0, asL = add ? add->sL : 0, asH = add ? add->sH : 0;
  if (q.dtype == KSANA_SAGE_BF16)
    sla_apply_kernel<KSANA_SAGE_BF16><<<grid_apply, block, kApplyLds, s>>>(q.ptr, q.sB, q.sL, q.sH, m_frag, ksum, proj_b, add_ptr, asB, asL,
                                                                          asH, out.ptr, out.sB, out.sL, out.sH, H, L, kBlocks);
  else
    sla_apply_kernel<KSANA_SAGE_FP16><<<grid_apply, block, kApplyLds, s>>>(q.ptr, q.sB, q.sL, q.sH, m_frag, ksum, proj_b, add_ptr, asB, asL,
                                                                          asH, out.ptr, out.sB, out.sL, out.sH, H, L, kBlocks);
  return hipGetLastError();
}

hipError_t launch_sla_linear(const InTensor& q, const InTensor& k, const InTensor& v, int B, int H, int L,
                             const float* proj_w, const float* proj_b, const InTensor* add, const OutTensor& out,
                             float* part, uint16_t* m_frag, float* ksum, hipStream_t s) {
  int runs = 1, rows_per_run = L;
  plan_sla_runs(B, H, L, &runs, &rows_per_run);
  const dim3 block(kSlaThreads);
  if (q.dtype == KSANA_SAGE_BF16) {
    sla_kv_partial_kernel<KSANA_SAGE_BF16><<<dim3(runs, H, B), block, 0, s>>>(k, v, H, L, rows_per_run, part);
    sla_kv_finalize_kernel<KSANA_SAGE_BF16><<<dim3(kD / kFinRows, B * H), block, 0, s>>>(part, runs, proj_w, m_frag, ksum);
  } else {
    sla_kv_partial_kernel<KSANA_SAGE_FP16><<<dim3(runs, H, B), block, 0, s>>>(k, v, H, L, rows_per_run, part);
    sla_kv_finalize_kernel<KSANA_SAGE_FP16><<<dim3(kD / kFinRows, B * H), block, 0, s>>>(part, runs, proj_w, m_frag, ksum);
  }
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? launch_sla_apply(q, B, H, L, proj_b, add, out, m_frag, ksum, s) : e;
}

}  // namespace ksana_sage

namespace ksana_sage {
hipError_t launch_sla_block_map(const uint16_t* pooled_q, const uint16_t* pooled_k, int dtype, int BH, int nq, int nk, int keep,
                                int8_t* block_map, hipStream_t s) {
  if (nk > kMapMaxKeyBlocks) return hipErrorInvalidValue;
  const int nk_pad = (nk + 31) / 32 * 32;
  const dim3 grid((nq + 31) / 32, BH), block(kMapThreads);
  const size_t lds = (size_t)32 * nk_pad * 2;
  const bool bf16 = dtype == KSANA_SAGE_BF16;
  constexpr int kAll = kMapMaxKeyBlocks / 64;
  if (nk <= 512) {
    if (bf16)
      sla_block_map_kernel<KSANA_SAGE_BF16, 8><<<grid, block, lds, s>>>(pooled_q, pooled_k, nq, nk, nk_pad, keep, block_map);
    else
      sla_block_map_kernel<KSANA_SAGE_FP16, 8><<<grid, block, lds, s>>>(pooled_q, pooled_k, nq, nk, nk_pad, keep, block_map);
  } else if (bf16) {
    sla_block_map_kernel<KSANA_SAGE_BF16, kAll><<<grid, block, lds, s>>>(pooled_q, pooled_k, nq, nk, nk_pad, keep, block_map);
  } else {
    sla_block_map_kernel<KSANA_SAGE_FP16, kAll><<<grid, block, lds, s>>>(pooled_q, pooled_k, nq, nk, nk_pad, keep, block_map);
  }
  return hipGetLastError();
}
}  // namespace ksana_sage
