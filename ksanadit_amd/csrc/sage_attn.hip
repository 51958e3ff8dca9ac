// Fused quantized attention for gfx950 (MI355X): INT8 QK^T and FP8 PV on MFMA, fp32 online
// softmax in registers.
//
// Work split.  One workgroup = 8 waves = 256 query rows of one (batch, head); each wave owns
// 32 query rows for the whole key loop.  Keys are consumed in tiles of 64 rows (= one int8
// K scale block; Q scales are per row, i.e. per lane), K and V^T tiles are copied asynchronously (global_load ... lds) into an 8-deep LDS ring shared by the 8 waves.
// Two waves share a SIMD, so one wave's softmax (VALU) overlaps the other's MFMAs.
//
// Fragment algebra (32x32 MFMA, lane l: l32 = l % 32, hh = l / 32):
//   S^T = K . Q^T   v_mfma_i32_32x32x32_i8   A = K rows, B = Q rows; both read 16 bytes at channel
//                   offset 32*s + 16*hh, so the contraction order is the same on both sides.
//                   Accumulator register r of sub-tile t holds key 32*t + 8*(r/4) + 4*hh + r%4
//                   for query l32: a lane owns ONE query column -> row max / row sum are
//                   register reductions plus a single lane<->lane+32 exchange.
//   O^T = V^T . P^T v_mfma_f32_32x32x64_f8f6f4   B = P packed to e4m3 straight from the S^T
//                   registers (byte 16*t + r); A = V^T tile whose bytes the quantizer already
//                   stored in that same key order, so P never goes through LDS.
//
// The int32 accumulators start at the bit pattern of 1.5 * 2^23 ("magic"): the result read
// as fp32 IS 12582912 + dot exactly (|dot| <= 127*127*128 < 2^22), which removes the
// int->float conversion from the softmax: p = exp2(fma(acc_as_float, sc, c)).
#include "sage_attn_device.h"
#include "sage_sla_device.h"

#include <atomic>
#include <type_traits>

#include "../../include/ksana_sage_hip.h"

namespace ksana_sage {
namespace {

// Two shapes of workgroup: 8 waves = 256 query rows with an 8-stage tile ring (one workgroup holds a compute unit:
// every K/V tile copied serves 256 rows), and 4 waves = 128 query rows with a 4-stage ring, two of which share a
// compute unit - they run out of step, so one's prologue and epilogue hide under the other's key loop (what short key
// sequences need), and a workgroup is exactly one row of a block mask.
template <int kW, int kG = 4>
struct WgShape {
  static_assert(kW == 8 || kW == 4, "workgroups of 8 or 4 waves");
  static constexpr int kThreads = kW * 64;
  static constexpr int kRows = kW * 32;                // query rows per workgroup
  // K tiles and V^T tiles have a ring of kStages slots each.  A K tile is read one step BEFORE the step of its
  // probabilities and its V^T tile one step AFTER, so in one ring of whole tiles two K halves would always be dead; in a
  // ring of its own K can be requested further ahead.
  static constexpr int kStages = kW == 8 ? 8 : 4;
  static constexpr int kRingBytes = kStages * 2 * kTileBytes;
  // 1 KiB copy instructions per wave and tile, K and V^T: with 64 channels (kG == 2) half of either tile is all that is read,
  // and the other half is not copied
  static constexpr int kCopies = 2 * (8 / kW) * kG / 4;
  // How many tiles ahead step j requests the V^T and the K tile.  4 waves: K into the slot of tile j, which every wave
  // has read; a copy then has three steps (about three microseconds) to arrive, which matters where tiles miss the L2
  // (block masks).  8 waves: what the groups of four steps below allow.
  static constexpr int kAhead = kW == 8 ? 3 : 2, kAheadK = kW == 8 ? 5 : 4;
  // copies that may still be in flight at the barrier that ends a step: those of this step and of the one before
  static constexpr int kInFlight = 2 * kCopies;
  // The 8-wave shape's rings have room for waves that are steps apart: in the loop unrolled over them the waves meet after
  // every fourth step only, so that a wave which rescales its rows holds up the others less often.  The copies of a
  // group's four steps (g .. g+3: V^T tiles g+3 .. g+6, K tiles g+5 .. g+8, into slots last read before the group) go out
  // in its first two steps and have landed when it ends.  A barrier after every second step instead of every step:
  // 2616 -> 2571 us at 40 heads of 16384 tokens (2477 -> 2446 with outliers); after every fourth: 0-0.4 % more, and
  // 515 -> 501 us at B=2, 16 heads of 64 channels, 9001 tokens.
  static constexpr int kGroup = kW == 8 ? 4 : 1;
};
constexpr int kSparseMaxKeyTiles4 = 2048;    // 4-wave workgroups keep their tile list as 16-bit entries so that two fit a compute unit
constexpr int kMaxKeyTiles = 4096;           // K scales of one head are kept in LDS: Lk <= 262144
constexpr int kShortKeyTiles = 16;           // with at most this many key tiles (Lk <= 1024) nobody's keys are cut into runs
constexpr int kShortMaxKeyTiles = 2048;      // the most key tiles a dense 4-wave workgroup can hold scales for

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
// lds_copy16 through a buffer descriptor: 16 bytes per lane from (base + src_off + lane_off) to `lds_base + kSlot`.  One scalar
// offset serves every buffer whose tiles have the same number, and a slot known at compile time rides in the
// instruction that writes M0 - two scalar instructions per copy where the 64-bit form above takes six.
template <int kSlot>
__device__ __forceinline__ void lds_copy16_at(const v4i& buffer, unsigned lane_off, unsigned src_off, unsigned lds_base) {
  asm volatile("s_add_u32 m0, %0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %3, %4 offen lds"
               :
               : "s"(lds_base), "n"(kSlot), "v"(lane_off), "s"(buffer), "s"(src_off)
               : "memory", "m0", "scc");
}
#pragma clang diagnostic pop

// Dense 8-wave calls can hold two kinds of workgroup in one grid: blocks below p.split_first_block walk all key tiles of
// their (head, query block); each of the blocks from there on takes one of `p.n_split` equal runs of key tiles and leaves
// unnormalised accumulators, running maxima and row sums in the workspace for sage_attn_merge_kernel.  The runs stand
// for the query blocks beyond the last full round of the chip, which would otherwise hold it for a whole round alone; in
// the same grid they start as the last whole blocks finish.
// kG: 32-channel groups the matrix instructions cover - 4, or 2 when the head size is 64 (rows run zero-extended to
// 128 channels and the operands keep their layout; see kMagicI2 for what is left out and why nothing is lost; the
// result equals the full-width code's up to the rounding of one constant in the exponent).
// kLinear: the sparse-linear backend's linear branch is added to the result in the epilogue.
// kNumbered: the blocks of a batch are numbered by its counts (batch_rows_wg).  A variant of its own: with this behind a branch in the
// dense ones their scalar registers run short and arguments are loaded anew in every workgroup's set-up (16 heads of 2600 tokens
// 58.7 / 59.3 us, 24 of 2000 53.1 / 54.0).
template <int DT, bool kPwlExp, bool kSparse, int kW, bool kTileSkip, int kG, bool kCausal, bool kLinear, bool kNumbered>
__global__ __launch_bounds__(kW * 64, kW == 8 ? 1 : 2) void sage_attn_fwd_kernel(const AttnParams p, int n_qwg,
                                                                                   int n_wg, int wg_per_xcd) {
  want(p.q_rows.ptr, p.k_tiles, p.o.sH, p.block_mask, n_qwg);
  constexpr bool kCanSplit = !kSparse && kW == 8 && !kNumbered;
  static_assert(!kNumbered || (!kSparse && !kCausal && !kPwlExp && !kTileSkip), "batches with counts: the dense default variant");
  static_assert(kSparse || !kCausal || (kW == 4 && !kPwlExp && !kTileSkip), "causal without a list: the default variant in 4 waves");
  // kCausal == false: the caller vouches that p.causal is 0, and everything that serves the diagonal (the per-wave
  // last tile, 32 lane masks held in scalar registers, the selects that blank a wave's probabilities past its rows)
  // is compiled out of the key loop
  const bool causal = kCausal && (!kSparse || p.causal);
  using Shape = WgShape<kW, kG>;
  constexpr int kThreadsAttn = Shape::kThreads, kRowsWg = Shape::kRows, kStages = Shape::kStages, kAhead = Shape::kAhead;
  constexpr int kListMax = kW == 8 ? kSparseMaxKeyTiles : kSparseMaxKeyTiles4;
  static_assert(!(kTileSkip && kPwlExp), "the piecewise-linear code formula has its own zero point: no tiles are skipped there");
  static_assert(kG == 4 || kG == 2, "128 channels, or 64 zero-extended");
  static_assert(!kLinear || (kSparse && !kCausal && kW == 4 && kG == 4), "the linear branch goes with a block mask, 128 rows a workgroup");
  constexpr bool kUnrolled = !kPwlExp && !kTileSkip && !(kSparse && kW == 8);  // the variants calls take by default
  constexpr int kMagicBits = kG == 4 ? kMagicI : kMagicI2;
  constexpr float kMagicVal = kG == 4 ? kMagicF : kMagicF2;
  int bh, b, h, qwg;  // (batch, head) pair, batch entry and head, query block
  // query rows [0, lq) of this batch take part: all of them, or the caller's per-batch count; the rows from lq up
  // to Lq exist in the output and are written as zeros
  // keys [0, lk) of this batch take part: all of them, or the caller's per-batch count
  int lq = p.Lq, lk = p.Lk;
  const bool is_run = kCanSplit && (int)blockIdx.x >= p.split_first_block;  // uniform
  const int run_id = is_run ? (int)blockIdx.x - p.split_first_block : 0;    // the partial result's place in the workspace
  if constexpr (kNumbered) {  // (BatchRun, BatchPlace)
    const int xcd = blockIdx.x & 7, at = blockIdx.x >> 3;
    int starts[kBatchStarts];
    BatchRun run;
    if (p.numbered == 1) {
      typedef const __attribute__((address_space(4))) int32_t* Constant;
      const Constant at_starts = reinterpret_cast<Constant>(reinterpret_cast<uintptr_t>(p.split_ml));
#pragma unroll
      for (int i = 0; i < kBatchStarts; ++i) starts[i] = at_starts[i];  // (scalar loads, together)
      run = batch_run_of(starts, p.B, at);
      take_counts(p.q_lens, p.k_lens, run.b, lq, lk);
    } else {
      int rows, keys;
      const int mine = batch_number(BatchNumbers{nullptr, p.B, p.Hq, p.Lq, p.Lk, kRowsWg, p.q_lens, p.k_lens}, threadIdx.x & 63, rows, keys);
#pragma unroll
      for (int i = 0; i < kBatchStarts; ++i) starts[i] = __builtin_amdgcn_readlane(mine, i);
      run = batch_run_of(starts, p.B, at);
      lq = __builtin_amdgcn_readlane(rows, run.b), lk = __builtin_amdgcn_readlane(keys, run.b);
    }
    b = run.b;
    const BatchPlace place = batch_place(run, xcd, at, p.Hq, n_qwg, batch_blocks(lq, lk, kRowsWg));
    if (place.b < 0) return;
    h = place.h, qwg = place.qwg;
    bh = b * p.Hq + h;
  } else if (kCausal && p.causal_grid.group != 0) {
    if (!causal_place(p.causal_grid, blockIdx.x, n_qwg, &bh, &qwg)) return;
  } else {
    int wg;
    if (is_run) {
      wg = p.split_first_wg + run_id / p.n_split;
    } else {
      // Consecutive workgroup ids land on consecutive XCDs (8 per chip, one L2 each).  Give every
      // XCD a contiguous run of (head, query block) pairs so the workgroups that stream the same
      // K/V tiles share one L2.
      const int xcd = blockIdx.x & 7, at = blockIdx.x >> 3;
      if (!kSparse && !kCausal && p.small_last != 0) {
        // Short last blocks (see launch_attn_fwd) behind the whole ones: an XCD's run of whole blocks, then its share of the
        // heads' last ones.
        const int whole = wg_per_xcd - p.small_last, n_pairs = p.B * p.Hq, n_whole = n_pairs * (n_qwg - 1);
        if (at < whole) {
          const int w = xcd * whole + at;
          if (w >= n_whole) return;
          const int pair = w / (n_qwg - 1);
          wg = w + pair;
        } else {
          const int pair = xcd * p.small_last + (at - whole);
          if (pair >= n_pairs) return;
          wg = pair * n_qwg + n_qwg - 1;
        }
      } else if (p.batch_run == 0) {
        wg = xcd * wg_per_xcd + at;
        if (wg >= n_wg) return;
      } else {
        // (batches that are not numbered by their counts, see batch_rows_wg)
        // batch entries of unequal length: an eighth of every entry's workgroups to every XCD.  One run across the entries
        // would leave the XCDs that drew the short ones idle.  The entries run in the order of their index, longest first or
        // not: the order that ends with the longest one costs up to 5-8 % in grids of two rounds, nothing in long ones.  us,
        // one run across the entries / this, for lengths falling, rising, the longest last but one: B=3, 24 heads, 100 / 72 /
        // 45 % of 3001 x 4099 265 / 165, 273 / 173, 273 / 178; B=2, 40 heads of 16384 5560 / 3280, 5530 / 3272, 5600 / 3270.
        const int b = at / p.batch_run, n_batch = p.Hq * n_qwg;
        const int in_batch = xcd * p.batch_run + (at - b * p.batch_run);
        wg = b * n_batch + in_batch;
        if (in_batch >= n_batch || wg >= n_wg) return;
      }
    }
    bh = wg / n_qwg;
    qwg = wg - bh * n_qwg;
    if (causal) qwg = n_qwg - 1 - qwg;  // the long ones first, as above
  }
  if constexpr (!kNumbered) {
    b = bh / p.Hq, h = bh - b * p.Hq;
    take_counts(p.q_lens, p.k_lens, b, lq, lk);
  }
  const int bhk = b * p.Hkv + h / (p.Hq / p.Hkv);

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform by construction: keep it scalar
  const int l32 = lane & 31, hh = lane >> 5;
  // A last block of at most 64 rows has work for one or two waves.  Alone on its unit such a workgroup takes half a microsecond a
  // step, next to another one as long as the whole blocks do; so its four waves share the keys out instead (see below).
  constexpr bool kCanShare = !kSparse && !kCausal && kW == 4 && !kPwlExp && !kTileSkip;
  // (by the rows the tensor has: a row's bits do not depend on its batch entry's count)
  const int rows_here = p.Lq - qwg * kRowsWg;
  const bool shared = kCanShare && __builtin_amdgcn_readfirstlane(p.wg_waves == 0 && rows_here <= 64 && lq > qwg * kRowsWg &&
                                                                  lk > kShortKeyTiles * kBlkK) != 0;
  const int sharers = rows_here > 32 ? 2 : 4;  // waves per 32 rows
  const int q0 = qwg * kRowsWg + 32 * (shared ? wave / sharers : wave);
  const bool active = q0 < lq;  // wave-uniform; inactive waves only help move tiles
  auto write_zero_rows = [&]() {  // softmax over no key: the output rows are defined as zeros
    const int q = q0 + l32;
    if (q < p.Lq && 64 * hh < p.d_out) {
      uint4* orow = reinterpret_cast<uint4*>(p.o.ptr + b * p.o.sB + (int64_t)q * p.o.sL + h * p.o.sH + 64 * hh);
#pragma unroll
      for (int i = 0; i < 8; ++i) orow[i] = make_uint4(0, 0, 0, 0);
    }
  };
  int tile0 = 0;  // first key tile of this workgroup's run
  if (is_run) {
    const int split = run_id % p.n_split;
    const int tiles = (lk + kBlkK - 1) / kBlkK;
    const int per = (tiles + p.n_split - 1) / p.n_split;
    tile0 = split * per;
    const int tile1 = min(tiles, tile0 + per);
    if (tile0 >= tile1 || qwg * kRowsWg >= lq) {  // nothing in this run (few tiles, a batch entry without keys, or no query row): an empty partial
      if (active) {
        const int row = wave * 32 + l32;
        float* po = p.split_o + ((int64_t)run_id * kAttnQPerWg + row) * kD + 64 * hh;
#pragma unroll
        for (int i = 0; i < 16; ++i) reinterpret_cast<float4*>(po)[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (hh == 0) reinterpret_cast<float2*>(p.split_ml)[(int64_t)run_id * kAttnQPerWg + row] = make_float2(-INFINITY, 0.f);
      }
      return;
    }
    lk = min(lk, tile1 * kBlkK) - tile0 * kBlkK;  // from here on the run is the whole key sequence
  } else {
    if (lk == 0 || qwg * kRowsWg >= lq) {  // no key, or none of the workgroup's rows takes part
      write_zero_rows();
      return;
    }
  }

  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];

  // ---- Q fragments (B operand), 4 channel steps --------------------------------------
  v4i qf[4];
  float qs = 0.0f;
  uint4 q_raw[8];
  // (not with a block mask: there such calls' key loops ran 1 % slower for the code being there; and out of the way of the
  // calls that do not take it: 12 workgroups of 10 tiles 23.9 us with it in line, 23.0 without)
  constexpr bool kOwnQ = !kSparse || kCausal;
  const bool own_q = __builtin_expect(kOwnQ && active && !shared && p.q_rows.ptr != nullptr, 0);  // uniform per wave
  // Rows that are quantized already are requested first of all and touched by the set-up's one wait only: their loads run under
  // the list's mask bytes, the operands' set-up and the tile copies.  us per call, behind the copies / first: dense, 16 heads of
  // 2600 tokens 59.6 / 58.8, 24 of 2000 53.9 / 53.1, 2 x 24 of 774 36.4 / 35.9, 40 of 420 22.9 / 22.7; causal, 16 of 1500 33.2 / 33.0.
  // (kPinned: what was loaded is taken over in the branch that has no rows of its own.  Elsewhere the compiler copies the registers
  // before that branch, and a workgroup with rows of its own waits for its tile copies before it requests them: 24 heads of 4400 on
  // 700 keys 47.8 / 47.3.  In the causal variants and in 8 waves it costs the calls with stored rows 1 % instead: 16 of 2600 59.3.)
  constexpr bool kPinned = kW == 4 && !kCausal;
  v4i q_codes[4];
  float q_sc = 0.0f;
#pragma unroll
  for (int s = 0; s < 4; ++s) q_codes[s] = v4i{0, 0, 0, 0};
  if (active && !own_q && !(shared && p.q_rows.ptr != nullptr)) {
    const int8_t* qrow = p.q_i8 + ((int64_t)bh * p.lq_pad + q0 + l32) * kD + 16 * hh;
#pragma unroll
    for (int s = 0; s < kG; ++s) q_codes[s] = *reinterpret_cast<const v4i*>(qrow + 32 * s);
    q_sc = p.q_scale[(int64_t)bh * p.lq_pad + q0 + l32];  // one scale per query row = per lane
  }
  auto take_q = [&]() {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      if (kPinned) pin(q_codes[s]);
      qf[s] = q_codes[s];
    }
    if (kPinned) pin(q_sc);
    qs = q_sc;
  };

  v16f oacc[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) oacc[dt][r] = 0.0f;
  // reference point of query l32 in the log2 domain (its "running maximum"), and what the steps read it as: the
  // exponent's constant part and the score above which the point has to move
  // (base -inf: the probabilities of a row without a point are zeros)
  float m_run = -INFINITY, x_base = -INFINITY, x_limit = -INFINITY;
  // Row sums come from the matrix pipe too, of the SAME e4m3-rounded P the numerator uses.  The 16x16x128 instruction
  // takes half the matrix cycles of the 32x32x64 one and a quarter of its accumulators; its B operand is P's register
  // block read as 16 columns with four groups of 16 lanes stacked along the contraction: groups 0 and 2 hold the two
  // halves of query (lane % 16)'s keys, groups 1 and 3 those of query 16 + (lane % 16).  A therefore carries ones
  // (e4m3 1.0 = 0x38) where output row 4 g' .. 4 g' + 3 and group g agree in parity and zeros elsewhere: the lanes of
  // group g' then find the sum of their own query in all four registers.  Only register 0 is read and rescaled.
  // A zero of A meets the probabilities of the query 16 further, and zero times NaN is NaN: no probability may be one
  // (move_point sees to it).
  v4f lacc = {0.0f, 0.0f, 0.0f, 0.0f};
  // eight registers on purpose: left as one value the compiler keeps a single copy and rebuilds
  // the 8-register operand with seven moves in every step
  v8i ones;
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    int one4 = ((lane >> 2) & 1) == ((lane >> 4) & 1) ? 0x38383838 : 0;
    pin(one4);
    ones[r] = one4;
  }

  // kept opaque so the 16 registers stay resident instead of being rebuilt from constants
  // (8 moves) at every tile
  v16i magic;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    int m = kMagicBits;
    pin(m);
    magic[r] = m;
  }

  const uint8_t* k_src = reinterpret_cast<const uint8_t*>(p.k_tiles) + ((int64_t)bhk * p.nkb + tile0) * kTileBytes;  // uniform
  const uint8_t* v_src = p.v_tiles + ((int64_t)bhk * p.nkb + tile0) * kTileBytes;
  const float* ks_ptr = p.k_scale + (int64_t)bhk * p.nkb + tile0;
  const int nkb = (lk + kBlkK - 1) / kBlkK;  // tiles this batch uses; p.nkb stays the per-head stride
  // K scales live in LDS behind the ring: a per-tile global load would share the in-order
  // vmcnt queue with the tile copies and stall on all of them
  // behind the ring: the head's V scales and V means (2 x 128 floats, read by the epilogue), then its K scales
  float* s_vs = reinterpret_cast<float*>(smem + Shape::kRingBytes);
  float* s_ks = s_vs + 2 * kD;

  // ---- block mask: the workgroup's list of key tiles ---------------------------------------
  // A mask row covers 128 query rows, a workgroup two of them (waves 0-3, waves 4-7).  Wave 0
  // compacts, in key order, the tiles either row asks for into LDS: entry = tile | row-0 flag
  // << 16 | row-1 flag << 17.  The loop below then walks list positions instead of tile
  // numbers; a wave whose row does not ask for a tile zeroes its probabilities for it and
  // leaves its running maximum alone, so the result is exactly the masked softmax.
  // Causal attention (key <= query row) on top of a mask runs through the same list, and without one over the tile
  // numbers themselves: the workgroup takes the tiles up to the one holding its last row, a wave leaves alone the tiles past its own last row, and the one
  // tile that straddles its rows' diagonal is masked element by element.
  // (one mask row per 4-wave workgroup: an entry is the tile number and fits 16 bits; with two mask rows per
  // workgroup it carries their two flags above the number)
  using ListEntry = typename std::conditional<kW == 4, uint16_t, int>::type;
  ListEntry* s_list = reinterpret_cast<ListEntry*>(s_ks + kListMax);
  int* s_count = reinterpret_cast<int*>(s_list + kListMax);
  // loop length: list entries with a mask, key tiles without (causal: up to the one holding the workgroup's last row)
  const int wg_tiles = causal ? min(nkb, ((qwg * kRowsWg + kRowsWg - 1) >> 6) + 1) : nkb;
  int n_tiles = wg_tiles;
  // a wave's 32 rows start at a multiple of 32, so exactly one 64-key tile holds their diagonal
  const int my_last = causal ? (q0 >> 6) : 0x7ffffffe;
  if constexpr (kSparse) {
    if (wave == 0) {
      const int nqm = (p.Lq + kMaskBlkQ - 1) / kMaskBlkQ;
      const bool masked = p.block_mask != nullptr;
      constexpr int kMaskRows = kRowsWg / kMaskBlkQ;  // mask rows a workgroup covers: 2 or 1
      const int8_t* m0 = masked ? p.block_mask + b * p.mask_sB + h * p.mask_sH + (int64_t)(kMaskRows * qwg) * p.nkb : nullptr;
      const bool two = kMaskRows == 2 && 2 * qwg + 1 < nqm;
      int base = 0;
      // eight chunks of 64 tiles at a time: their mask bytes are requested together, so a list of 512 tiles costs
      // one memory latency instead of eight
      for (int jb = 0; jb < wg_tiles; jb += 512) {
        int8_t b0[8], b1[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) {
          const int j = jb + 64 * c + lane;
          b0[c] = b1[c] = 1;
          if (masked && j < wg_tiles) {
            b0[c] = m0[j];
            if (two) b1[c] = m0[p.nkb + j];
          }
        }
#pragma unroll
        for (int c = 0; c < 8; ++c) {
          const int j = jb + 64 * c + lane;
          if (jb + 64 * c >= wg_tiles) break;  // uniform
          int f0 = 0, f1 = 0;
          if (j < wg_tiles) {
            f0 = b0[c] != 0;
            f1 = two && b1[c] != 0;
          }
          const bool keep = (f0 | f1) != 0;
          const unsigned long long bal = __ballot(keep);
          const int pre = __builtin_amdgcn_mbcnt_hi((unsigned)(bal >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)bal, 0));
          if (keep) s_list[base + pre] = static_cast<ListEntry>(kW == 4 ? j : (j | (f0 << 16) | (f1 << 17)));
          base += __popcll(bal);
        }
      }
      if (lane == 0) *s_count = base;
    }
    __syncthreads();
    n_tiles = __builtin_amdgcn_readfirstlane(*s_count);
    if (n_tiles == 0) {  // neither mask row allows any key
      write_zero_rows();
      return;
    }
  }
  // the head's K scales (in loop order: tile order, or the list's) and V scales / means go to LDS, once the first
  // tile copies are on their way, so that the loads' latencies overlap
  // (copied as the tiles are, with nothing to wait for but the set-up's one wait)
  auto fill_scales = [&]() {
    if (wave < 4) lds_copy4((wave < 2 ? p.v_scale : p.v_mean) + (int64_t)bhk * kD, (unsigned)((wave & 1) * 64 + lane) * 4, s_vs + wave * 64);
    for (int i0 = wave * 64; i0 < n_tiles; i0 += kThreadsAttn) {
      const int i = i0 + lane;
      if (i < n_tiles) {
        unsigned at = (unsigned)i;
        if constexpr (kSparse) at = (unsigned)(s_list[i] & 0xffff);
        lds_copy4(ks_ptr, at * 4, s_ks + i0);
      }
    }
  };
  if constexpr (kCanShare) {
    if (shared) {
      // A wave takes a run of ceil(tiles / sharers) key tiles, its operands straight from the L2 into registers (each as soon
      // as the step before is through with it), with reference points of its own; the four results are put together as the merge kernel does it, through LDS.  Bound by its chain of steps, a
      // quarter as long.  us per call, whole / shared: 40 heads of 1560 tokens, where eight of the 520 workgroups start when the
      // others end, 67.9 / 56.8.  Errors against 64 bits are those of whole rows or below: 0.0383 / 0.0388 at N(0, 1),
      // 0.0289 / 0.0295 with outliers.
      if (p.q_rows.ptr != nullptr) {
        uint4 raw[8];
        const uint16_t* qrow = p.q_rows.ptr + b * p.q_rows.sB + (int64_t)min(q0 + l32, p.Lq - 1) * p.q_rows.sL + h * p.q_rows.sH + 16 * hh;
#pragma unroll
        for (int i = 0; i < 2 * kG; ++i) {
          raw[i] = *reinterpret_cast<const uint4*>(qrow + 32 * (i >> 1) + 8 * (i & 1));
          if (q0 + l32 >= lq) raw[i] = make_uint4(0, 0, 0, 0);
        }
        quant_q_rows<DT, kG>(raw, p.q_premul, qf, qs);
      } else {
        take_q();
      }
      fill_scales();
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      const int per = (nkb + sharers - 1) / sharers, run = wave & (sharers - 1), j0 = min(run * per, nkb), j1 = min(j0 + per, nkb);
      const uint8_t* kt = k_src + lane * 16;
      const uint8_t* vt = v_src + lane * 16;
      v4i kf[2 * kG];  // (sub-tile t, channel step s) at t * kG + s
      auto fetch_k = [&](int j) {
#pragma unroll
        for (int i = 0; i < 2 * kG; ++i)
          kf[i] = *reinterpret_cast<const v4i*>(kt + (int64_t)j * kTileBytes + ((i / kG) * 4 + i % kG) * 1024);
      };
      v8i vf[kG];
      auto fetch_v = [&](int j) {
#pragma unroll
        for (int dt = 0; dt < kG; ++dt) {
          const v4i lo = *reinterpret_cast<const v4i*>(vt + (int64_t)j * kTileBytes + (2 * dt + 0) * 1024);
          const v4i hi = *reinterpret_cast<const v4i*>(vt + (int64_t)j * kTileBytes + (2 * dt + 1) * 1024);
          vf[dt] = v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        }
      };
      if (j0 < j1) {
        fetch_k(j0);
        fetch_v(j0);
      }
      __builtin_amdgcn_s_setprio(2);  // (a chain with nothing beside it: ahead of the neighbour's waves)
#pragma unroll 1
      for (int j = j0; j < j1; ++j) {
        v16i s[2] = {magic, magic};
#pragma unroll
        for (int c = 0; c < kG; ++c)
#pragma unroll
          for (int u = 0; u < 2; ++u) s[u] = __builtin_amdgcn_mfma_i32_32x32x32_i8(kf[u * kG + c], qf[c], s[u], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        fetch_k(min(j + 1, nkb - 1));
        __builtin_amdgcn_sched_barrier(0);
        const int n_last = j == nkb - 1 ? lk & (kBlkK - 1) : 0;  // (uniform) keys of a ragged tile
        if (n_last != 0) blank_scores<kMagicBits>(s, hh, n_last);
        int top = max(s[0][0], s[1][0]);
#pragma unroll
        for (int r = 1; r < 16; ++r) top = max(max(top, s[0][r]), s[1][r]);
        float sc = qs * s_ks[j], mneg = -kMagicVal * sc;
        const float alpha = move_point(top, sc, mneg, qs, m_run, x_base, x_limit);
        if (j == j0 ? __any(alpha != alpha) : __any(alpha != 1.0f)) {
#pragma unroll
          for (int dt = 0; dt < kG; ++dt)
#pragma unroll
            for (int r = 0; r < 16; ++r) oacc[dt][r] *= alpha;
          lacc[0] *= alpha;
        }
        v8i pf = tile_probs(s, sc, x_base + mneg);
        if (n_last != 0) blank_probs(pf, hh, n_last);
#pragma unroll
        for (int dt = 0; dt < kG; ++dt) oacc[dt] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(vf[dt], pf, oacc[dt], 0, 0, 0, 0, 0, 0);
        lacc = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(ones, pf, lacc, 0, 0, 0, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        fetch_v(min(j + 1, nkb - 1));
      }
      // every wave's accumulators in the ring, points and sums where the K scales were; then the waves of a row group finish a
      // quarter or half of its channels each
      float* s_o = reinterpret_cast<float*>(smem);
      float2* s_ml = reinterpret_cast<float2*>(s_ks);
      __syncthreads();
#pragma unroll
      for (int dt = 0; dt < kG; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) s_o[((wave * 4 + dt) * 16 + r) * 64 + lane] = oacc[dt][r];
      if (hh == 0) s_ml[wave * 32 + l32] = make_float2(m_run, lacc[0]);
      __syncthreads();
      const int first = wave - run;  // the row group's first wave
      float weight[kW];
      float m = -INFINITY, l = 0.0f;
#pragma unroll
      for (int i = 0; i < kW; ++i)
        if (i < sharers) m = fmaxf(m, s_ml[(first + i) * 32 + l32].x);
#pragma unroll
      for (int i = 0; i < kW; ++i) {
        weight[i] = 0.0f;
        if (i < sharers && i * per < nkb) {  // (uniform) a run with tiles
          const float2 ml = s_ml[(first + i) * 32 + l32];
          weight[i] = fast_exp2(ml.x - m);
          l += ml.y * weight[i];
        }
      }
      const int row = q0 + l32;
      const float inv_l = 1.0f / l, keep_mean = inv_l != 0.0f ? 1.0f : 0.0f;
#pragma unroll 1
      for (int cg = run; cg < kG; cg += sharers) {
        float o[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) o[r] = 0.0f;
#pragma unroll
        for (int i = 0; i < kW; ++i) {
          if (i >= sharers || i * per >= nkb) continue;
#pragma unroll
          for (int r = 0; r < 16; ++r) o[r] += s_o[(((first + i) * 4 + cg) * 16 + r) * 64 + lane] * weight[i];
        }
        uint16_t* orow = p.o.ptr + b * p.o.sB + (int64_t)row * p.o.sL + h * p.o.sH + 32 * cg + 8 * hh;
#pragma unroll
        for (int g = 0; g < 4; g += 2) {
          uint2 w[2];
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const int r = 4 * (g + e), d = 32 * cg + 8 * (g + e) + 4 * hh;
            const float4 s4 = *reinterpret_cast<const float4*>(s_vs + d), m4 = *reinterpret_cast<const float4*>(s_vs + kD + d);
            w[e] = half4<DT>(o[r] * inv_l * s4.x + m4.x * keep_mean, o[r + 1] * inv_l * s4.y + m4.y * keep_mean,
                             o[r + 2] * inv_l * s4.z + m4.z * keep_mean, o[r + 3] * inv_l * s4.w + m4.w * keep_mean);
            if (row >= lq) w[e] = make_uint2(0, 0);
          }
          // lanes l and l + 32 trade every second four channels, so that each stores eight in a row
          const auto x = __builtin_amdgcn_permlane32_swap(w[0].x, w[1].x, false, false);
          const auto y = __builtin_amdgcn_permlane32_swap(w[0].y, w[1].y, false, false);
          if (row < p.Lq) *reinterpret_cast<uint4*>(orow + 8 * g) = make_uint4(x[0], y[0], x[1], y[1]);
        }
      }
      __builtin_amdgcn_endpgm();
    }
  }
  // Causal calls: the list is in key order, so the entries this wave takes part in (tile <= the one on its diagonal)
  // are the first n_mine, and the diagonal tile, if listed, is the last of them.  Both are found once here; the key
  // loop then compares loop positions instead of looking list entries up.
  int n_mine = n_tiles, jdiag = -1;  // wave-uniform
  if constexpr (kCausal && !kSparse) {
    n_mine = min(n_tiles, my_last + 1);
    if (my_last < n_tiles) jdiag = my_last;
  }
  if constexpr (kSparse) {
    if (causal) {
      if (p.block_mask == nullptr) {  // the list is 0, 1, 2, ...
        n_mine = min(n_tiles, my_last + 1);
      } else {
        int cnt = 0;
        for (int j0 = 0; j0 < n_tiles; j0 += 64) {
          const int jx = j0 + lane;
          const bool le = jx < n_tiles && (s_list[jx] & 0xffff) <= my_last;
          cnt += __popcll(__ballot(le));
        }
        n_mine = cnt;
      }
      if (n_mine > 0 && (__builtin_amdgcn_readfirstlane(s_list[n_mine - 1]) & 0xffff) == my_last) jdiag = n_mine - 1;
    }
  }
  // key tile behind loop position jj, and whether this wave's mask row asks for it
  auto tile_of = [&](int jj) -> int {
    if constexpr (kSparse) return __builtin_amdgcn_readfirstlane(s_list[jj]) & 0xffff;
    return jj;
  };
  auto mine_at = [&](int jj) -> bool {
    if constexpr (kSparse) {
      if constexpr (kW == 4 && !kCausal) return true;  // one mask row per workgroup: every listed tile is wanted
      if constexpr (kW == 4) return jj < n_mine;
      const int e = __builtin_amdgcn_readfirstlane(s_list[jj]);
      return ((e >> (16 + (wave >> 2))) & 1) != 0 && jj < n_mine;
    }
    if constexpr (kCausal) return jj < n_mine;
    return true;
  };
  // causal only: loop position jj holds the tile on this wave's diagonal
  auto diag_at = [&](int jj) -> bool {
    if constexpr (kCausal) return jj == jdiag;
    return false;
  };
  const int n_diag = (q0 & 63) + l32 + 1;  // keys of its diagonal's tile that a lane's query sees

  // ---- asynchronous tile copies: HBM/L2 -> LDS without passing through registers ----------
  // Each wave moves its 1 KiB slice of the K tile and of the V^T tile (lane i -> byte 16*i of
  // the slice).  Copies retire in issue order, so "at most 2*n outstanding" == "all but the
  // newest n tiles have landed".
  // keys >= lk live only in the last key tile, which (if the list holds it) is the last entry; -1: there are none.  That tile
  // is a step of the loop like the others, blanked as the diagonal's is (blank_scores, blank_probs).  (As a step of its own after the loop, with a branch
  // per blanked score, one key of 64 in it cost 6 us a workgroup, 63 of them 2: 40 heads of 1536 queries, 512 / 513 / 575 keys
  // 18.0 / 24.0 / 20.5 us, 18.1 / 18.8 / 19.1 like this.)
  const int n_last = lk & (kBlkK - 1);
  const int tail = n_last != 0 && tile_of(n_tiles - 1) == nkb - 1 ? n_tiles - 1 : -1;
  // LDS slot of a tile's K half / V^T half
  auto k_slot = [&](int tile) -> uint8_t* { return smem + (tile & (kStages - 1)) * kTileBytes; };
  auto v_slot = [&](int tile) -> uint8_t* { return smem + (kStages + (tile & (kStages - 1))) * kTileBytes; };
  // clamped: past the end the last tile is copied again into a slot nobody reads any more,
  // which keeps the loop free of branches and the outstanding-copy count constant
  // This wave's 1 KiB slices of a tile: slice c * kW + wave; with 64 channels the slices that hold any - of K fragments 0, 1
  // of either half of the keys, of V^T the lower half - are one of each for four waves, and one of either for eight (waves
  // 0-3 copy K, waves 4-7 V^T).
  constexpr bool kEither = kG == 2 && kW == 8;
  const bool copies_k = !kEither || wave < 4, copies_v = !kEither || wave >= 4;
  const int slice_k = kG == 4 ? wave : (wave & 1) + 2 * (wave & 2), slice_v = kG == 4 ? wave : wave & 3;
  auto copy_tile_half = [&](bool is_v, int jl, uint8_t* dst) {  // jl: key tile number, wave-uniform
    if (is_v ? !copies_v : !copies_k) return;
    const int slice = is_v ? slice_v : slice_k;
#pragma unroll
    for (int c = 0; c < (kG == 4 ? 8 / kW : 1); ++c)
      lds_copy16((is_v ? v_src : k_src) + (int64_t)jl * kTileBytes, (unsigned)((c * kW + slice) * 64 + lane) * 16, dst + (c * kW + slice) * 1024);
  };
  auto copy_half = [&](bool is_v, int tile, uint8_t* dst) { copy_tile_half(is_v, tile_of(min(tile, n_tiles - 1)), dst); };
  // With a tile list, the key tiles behind the loop positions whose copies the next steps issue are kept in scalar
  // registers: looked up in the step, a list entry costs an LDS read whose wait also drains the operand reads
  // requested just before it.  ahead[i] = tile at position j + kAhead + i for the step j about to run; a step
  // fetches the one entry that enters the window (position j + 1 + kAheadK) and takes it over at its end.
  constexpr int kWindow = Shape::kAheadK - kAhead + 1;
  int ahead[kWindow];
  if constexpr (kSparse) {
#pragma unroll
    for (int i = 0; i < kWindow; ++i) ahead[i] = tile_of(min(kAhead + i, n_tiles - 1));
  }
  // The key loop's own copies: descriptors over this workgroup's tiles, the lane's offset in a tile, the offset of the
  // tiles the next copies take (past the last tile it stays there, as above)
  auto tiles_from = [&](const void* base) {
    const uint64_t a = reinterpret_cast<uint64_t>(base);
    return v4i{(int)(uint32_t)a, (int)(uint32_t)(a >> 32) & 0xffff, (p.nkb - tile0) * kTileBytes, 0x00020000};
  };
  const v4i k_buf = tiles_from(k_src), v_buf = tiles_from(v_src);
  const unsigned lds_0 = (unsigned)(uintptr_t)(const __attribute__((address_space(3))) void*)smem;
  const unsigned lane_off_k = (unsigned)(slice_k * 64 + lane) * 16, lane_off_v = (unsigned)(slice_v * 64 + lane) * 16;
  const unsigned lds_base_k = lds_0 + (unsigned)slice_k * 1024, lds_base_v = lds_0 + (unsigned)slice_v * 1024;
  const int off_last = (n_tiles - 1) * kTileBytes;
  int off_v = min(kAhead, n_tiles - 1) * kTileBytes, off_k = min(Shape::kAheadK, n_tiles - 1) * kTileBytes;
  auto copy_to = [&](auto slot, const v4i& buffer, unsigned lane_off, int off, unsigned lds_base) {
    constexpr int kSlot = decltype(slot)::value;
    lds_copy16_at<kSlot>(buffer, lane_off, off, lds_base);
    if constexpr (kW == 4 && kG == 4) lds_copy16_at<kSlot + 4096>(buffer, lane_off + 4096, off, lds_base);
  };
  // (kEither) this wave's tiles
  const v4i my_buf = copies_k ? k_buf : v_buf;
  const unsigned my_lane_off = copies_k ? lane_off_k : lane_off_v, my_lds_base = copies_k ? lds_base_k : lds_base_v;
  int off_mine = copies_k ? off_k : off_v;
  // the V^T and K tile that tile number kTile (modulo kStages) would request in a loop of single steps
  auto copies_of = [&](auto tile) {
    constexpr int kTile = decltype(tile)::value;
    using VSlot = std::integral_constant<int, (kStages + ((kTile + kAhead) & (kStages - 1))) * kTileBytes>;
    using KSlot = std::integral_constant<int, ((kTile + Shape::kAheadK) & (kStages - 1)) * kTileBytes>;
    if constexpr (kSparse) {
      copy_to(VSlot{}, v_buf, lane_off_v, ahead[0] * kTileBytes, lds_base_v);
      copy_to(KSlot{}, k_buf, lane_off_k, ahead[kWindow - 1] * kTileBytes, lds_base_k);
    } else if constexpr (kEither) {
      const unsigned slot = copies_k ? KSlot::value : VSlot::value;
      lds_copy16_at<0>(my_buf, my_lane_off, off_mine, my_lds_base + slot);
      off_mine = min(off_mine + kTileBytes, off_last);
    } else {
      copy_to(VSlot{}, v_buf, lane_off_v, off_v, lds_base_v);  // first: it is awaited first
      copy_to(KSlot{}, k_buf, lane_off_k, off_k, lds_base_k);
      off_v = min(off_v + kTileBytes, off_last);
      off_k = min(off_k + kTileBytes, off_last);
    }
  };
  // the copies of loop step j at ring position kAt (= j modulo kStages)
  auto issue_copy_at = [&](auto at) {
    constexpr int kAt = decltype(at)::value, kIn = kAt & (Shape::kGroup - 1);  // position in the group of steps
    if constexpr (Shape::kGroup == 1) {
      copies_of(at);
    } else if constexpr (kIn < 2) {
      copies_of(std::integral_constant<int, kAt + kIn>{});
      copies_of(std::integral_constant<int, kAt + kIn + 1>{});
    }
  };
  // the copies of loop step j (step -1: nothing; the prologue below brings the first tiles in)
  auto issue_copy = [&](int j) {
    if constexpr (kSparse) {
      copy_tile_half(true, ahead[0], v_slot(j + kAhead));
      copy_tile_half(false, ahead[kWindow - 1], k_slot(j + Shape::kAheadK));
    } else {
      copy_half(true, j + kAhead, v_slot(j + kAhead));  // first: it is awaited first
      copy_half(false, j + Shape::kAheadK, k_slot(j + Shape::kAheadK));
    }
  };
  // wait until every copy except the newest Shape::kInFlight has landed, then meet the other waves.
  // Plain s_barrier: a fence here would drain ALL copies and undo the prefetch.
  auto tile_barrier = [&]() {
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(Shape::kInFlight) : "memory");
  };
  // the same after the last step of a group (Shape::kGroup): everything has landed.  Steps [0, n_grouped) run in groups.
  auto group_barrier = [&]() { asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory"); };
  // K tile kStages goes into the slot of K tile 0, which every wave must have read by then - in the set-up, and a single
  // step requests tiles kAheadK ahead, the first group of steps all up to kStages, before the loop's first barrier.
  constexpr bool kSlotZeroSoon = Shape::kAheadK == kStages || (kUnrolled && Shape::kGroup > 1);
  // Without a list, the steps before any of the workgroup's waves meets its diagonal tile know nothing of it: they are the
  // dense loop's (with the diagonal's code in every unrolled step to be jumped over,
  // 8 191 tokens of 32 heads took 334 us instead of 323).  No unrolled step meets the ragged last tile either.
  constexpr bool kDiagApart = kCausal && !kSparse && kUnrolled;
  const int n_whole = tail >= 0 ? max(0, n_tiles - 2) : n_tiles;  // steps that neither form that tile's scores nor its probabilities
  const int n_plain = kDiagApart ? min(n_whole, max(0, ((qwg * kRowsWg) >> 6) - 1)) : n_whole;
  const int n_grouped = kUnrolled && Shape::kGroup > 1 ? n_plain / kStages * kStages : 0;

  // The compiler does not see the asynchronous copies in the memory-operation counter it models.  Every ordinary global
  // load of the set-up (Q fragments, scales) must therefore be known to have returned before the key loop starts:
  // left to itself the compiler would wait for "all but its n newest loads" at the first use of a loaded value
  // inside the loop, and drain the copies issued since.  The first copies go out first and everything is awaited
  // together.
  // The V^T slot of "tile -1" is read (times P = 0) by the first loop iteration: make it finite.
#pragma unroll
  for (int c = 0; c < 8 / kW; ++c)
    *reinterpret_cast<uint4*>(v_slot(-1) + (c * kThreadsAttn + tid) * 16) = make_uint4(0, 0, 0, 0);
  // Awaited here is what must be there before the first barrier of the loop: in single steps (4 waves) K tiles 0 and 1; the
  // rest goes out after the wait as the copies of "steps -2 and -1" and is awaited by the loop's own count (8 key
  // tiles, 32760 queries, 40 heads: -1.2 %).
  constexpr bool kLateCopies = Shape::kGroup == 1;
#pragma unroll
  for (int t = 0; t < (kLateCopies ? 0 : kAhead); ++t) copy_half(true, t, v_slot(t));
#pragma unroll
  for (int t = 0; t < (kLateCopies ? 2 : Shape::kAheadK); ++t) copy_half(false, t, k_slot(t));
  fill_scales();
  if (__builtin_expect(own_q, 0)) {
    // Requested behind the copies and without a condition (unlike stored rows, these are worked on in the set-up): loads return in
    // the order they were issued, and a wait for one issued before a copy, which the compiler does not count, is a wait for the copy too.  With the loads first and zeros
    // for what does not exist in their stead, the second pair of loads went out when the first had arrived.
    const int row = q0 + l32;
    const bool half = kG == 4 && p.q_rows.D != kD;  // (uniform) 64 channels in the full-width code
    const uint16_t* qrow = p.q_rows.ptr + b * p.q_rows.sB + (int64_t)min(row, p.Lq - 1) * p.q_rows.sL + h * p.q_rows.sH + 16 * hh;
#pragma unroll
    for (int s = 0; s < kG; ++s) {
      const int at = 32 * (half ? s & 1 : s);
      q_raw[2 * s] = *reinterpret_cast<const uint4*>(qrow + at);
      q_raw[2 * s + 1] = *reinterpret_cast<const uint4*>(qrow + at + 8);
    }
    if (half || q0 + 32 > p.Lq) {
#pragma unroll
      for (int s = 0; s < kG; ++s)
        if (row >= p.Lq || (half && s >= 2)) q_raw[2 * s] = q_raw[2 * s + 1] = make_uint4(0, 0, 0, 0);
    }
    quant_q_rows<DT, kG>(q_raw, p.q_premul, qf, qs);
  } else {
    take_q();
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the set-up's loads and, older than some of them, the copies
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  if constexpr (kLateCopies) {
    static_assert(Shape::kAheadK == kAhead + 2, "V^T tiles 0, 1 with K tiles 2, 3");
#pragma unroll
    for (int t = 0; t < kAhead; ++t) {
      copy_half(true, t, v_slot(t));
      copy_half(false, t + 2, k_slot(t + 2));
    }
  }

  if (!active) {
    // same copy / barrier sequence as the active waves
    if constexpr (kSlotZeroSoon) __builtin_amdgcn_s_barrier();
    for (int j = 0; j < n_tiles; ++j) {
      // (looks the tiles up where they are needed: a wave without rows has nothing an LDS wait could hold up)
      copy_half(true, j + kAhead, v_slot(j + kAhead));
      copy_half(false, j + Shape::kAheadK, k_slot(j + Shape::kAheadK));
      if (j >= n_grouped) tile_barrier();
      else if ((j & (Shape::kGroup - 1)) == Shape::kGroup - 1) group_barrier();
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (!is_run) write_zero_rows();  // rows in [lq, Lq), if any (the merge kernel writes them for cut blocks)
    return;
  }

  auto scale_o = [&](float alpha) {
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) oacc[dt][r] *= alpha;
    lacc[0] *= alpha;
  };
  // max over the 16 keys one S^T register block holds for query l32, as two independent chains
  auto max8 = [&](const v16i& blk, int r0) {
    int m = max(max(blk[r0], blk[r0 + 1]), blk[r0 + 2]);
    m = max(max(m, blk[r0 + 3]), blk[r0 + 4]);
    m = max(max(m, blk[r0 + 5]), blk[r0 + 6]);
    return max(m, blk[r0 + 7]);
  };
  // this lane's maximum over a whole tile (32 of query l32's 64 keys)
  auto lane_max = [&](const v16i (&blk)[2]) {
    return max(max(max8(blk[0], 0), max8(blk[0], 8)), max(max8(blk[1], 0), max8(blk[1], 8)));
  };
  // p = exp2(sc*dot - m_run + shift); the magic is folded into the constant c, which is off by
  // at most ~1.5 integer steps of the dot product
  auto p_of = [&](int acc_bits, float sc, float c) { return fast_exp2(__builtin_fmaf(__int_as_float(acc_bits), sc, c)); };
  // Four probabilities -> one dword of e4m3 codes (bytes in register order).
  //   exact:  p = exp2(x) on the transcendental unit, then the hardware e4m3 conversion;
  //   kPwlExp: the e4m3 CODE is computed directly, code = rne(8*x + 55.5) (saturating at 0): an
  //           e4m3 code is a 3-bit-mantissa logarithm, so this is exp2 with a piecewise-linear
  //           mantissa - two VALU slots per key instead of 3.5, no transcendental.  x <= 8.7 keeps
  //           the code <= 125, clear of the NaN code 127.
  auto pack4 = [&](int s0, int s1, int s2, int s3, float sc, float c) -> int {
    if constexpr (kPwlExp) {
      // here sc and c arrive pre-multiplied by 8, c with the +55.5 folded in
      unsigned w = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_fmaf(__int_as_float(s0), sc, c), 0, 0u);
      w = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_fmaf(__int_as_float(s1), sc, c), 1, w);
      w = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_fmaf(__int_as_float(s2), sc, c), 2, w);
      w = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_fmaf(__int_as_float(s3), sc, c), 3, w);
      return (int)w;
    } else {
      const float e0 = p_of(s0, sc, c), e1 = p_of(s1, sc, c), e2 = p_of(s2, sc, c), e3 = p_of(s3, sc, c);
      int w = __builtin_amdgcn_cvt_pk_fp8_f32(e0, e1, __float_as_int(e0), false);  // both halves get written
      return __builtin_amdgcn_cvt_pk_fp8_f32(e2, e3, w, true);
    }
  };
  // O^T += V^T . P^T for one 32-channel slice
  auto pv_slice = [&](const uint8_t* vst, int dt, const v8i& pf) {
    const v4i lo = *reinterpret_cast<const v4i*>(vst + ((dt * 2 + 0) * 64 + lane) * 16);
    const v4i hi = *reinterpret_cast<const v4i*>(vst + ((dt * 2 + 1) * 64 + lane) * 16);
    const v8i vf = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    oacc[dt] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(vf, pf, oacc[dt], 0, 0, 0, 0, 0, 0);
  };
  // S^T chunk i of a step: its channel step and half of the keys; the chunks without a product carry only their share of the
  // probabilities.  Two products in turn share Q's operand; in 8 waves with 64 channels a half is finished before the other.  us
  // per call, shared / one half after the other: 32760 tokens of 40 heads of 64 channels 8145 / 8046, 9001 of 2 x 16 549.5 /
  // 544.3; in 4 waves 3000 of 8 40.7 / 41.0, with 128 channels 27280 of 24 4664 / 4676.
  constexpr bool kByHalves = kG == 2 && kW == 8;
  auto qk_step = [](int i) { return kByHalves ? i % kG : i >> 1; };
  auto qk_half = [](int i) { return kByHalves ? i / kG : i & 1; };
  auto has_qk = [](int i) { return i >= 0 && i < 2 * kG; };

  v16i s_a[2], s_b[2];
  qk_tile<kG>(k_slot(0), lane, qf, magic, s_a);
  // (with the wait: a bare barrier lets the tile's last reads be on their way still when a wave without rows, which has nothing
  // else to do, requests the tile that goes into their slot)
  if constexpr (kSlotZeroSoon) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  if (diag_at(0)) blank_scores<kMagicBits>(s_a, hh, n_diag);
  if (tail == 0) blank_scores<kMagicBits>(s_a, hh, n_last);

  // What a step needs to know about its tile before the first probability: the scale, the exponent's constant and
  // whether a reference point moves.  Worked out at the end of the step before, so that its chain of dependent
  // operations runs under that step's last matrix instruction and the wait at the barrier.  Points move in few steps
  // (11 % of a wave's on outlier-ridden scores, 3 % on flat ones): a lane compares its own half's maximum with the
  // limit, and only when some lane of the wave exceeds it are the halves joined and points, factors and constants
  // formed anew (one wave-uniform branch instead of eight vector operations and a transcendental in every step).
  // With the 16x16 row sums, same bits: 10.60 -> 10.35 ms at B=1 H=40 L=32760 with outliers, 11.44 -> 11.05 without
  // (2045 cycles per step, from 2073, and 1843 with the loop unrolled and grouped; the chip runs at its power limit there,
  // and fewer operations raise its clock too).
  float sc = 0.0f, xc = 0.0f;           // scale of the coming tile, its exponent constant
  // factor a tile's point move puts on everything before it, and (wave-uniform) whether there is one: of even tiles and
  // of odd ones (step j applies tile j-1's and then finds tile j+1's)
  float alpha_even = 1.0f, alpha_odd = 1.0f;
  int moved_even = 0, moved_odd = 0;
  bool nothing = false;                 // (wave-uniform) every probability of the coming tile converts to zero
  auto look_ahead = [&](int jn, int mx, float ks, float& alpha, int& moved) {
    sc = qs * ks;
    float mneg = -kMagicVal * sc;
    const float m_half = __builtin_fmaf(__int_as_float(mx), sc, mneg);
    moved = 0;
    if (__ballot(!(m_half <= x_limit)) != 0) {  // (NaN counts as above)
      asm volatile("");  // (two branches on purpose: merged into one condition, the second is computed in every step)
      // (a tile this wave's mask row does not ask for, or that is not this loop's, leaves the points alone)
      if (jn < n_tiles && mine_at(jn)) {
        alpha = move_point<kPwlExp>(mx, sc, mneg, qs, m_run, x_base, x_limit);
        moved = 1;
      }
    }
    // exponent of key r: x = sc*dot - m_run + shift, with the magic folded into the constant
    // (which is therefore off by at most ~1.5 integer steps of the dot product)
    xc = x_base + mneg;
    // Every probability of a row in this tile is below 2^(m_tile - m_run + shift).  Under 2^-10 (half the smallest
    // e4m3 subnormal; a tie goes to the even code, zero) each one converts to the zero code - taken with a margin of
    // one octave for the exponent's few units of rounding.  With every row of the wave that far down, the wave writes
    // the zeros directly and leaves out the 64 exponentials and 32 conversions per lane (every chunk below tests this
    // one scalar); the matrix work that concerns the neighbouring tiles stays.  Same bits either way - the
    // pvthreshold idea of the reference's sparse kernel (sage_sla.py:237-253) with a threshold at which nothing changes.
    if constexpr (kTileSkip) nothing = __all(m_half < m_run - (kPShift + 11.0f));
  };
  look_ahead(0, lane_max(s_a), s_ks[0], alpha_even, moved_even);
  moved_even = __any(alpha_even != alpha_even);  // nothing has been accumulated yet: only a NaN has anything to say

  // Software pipeline, one key tile per step.  While this tile's probabilities are computed on
  // the VALU, the matrix pipe runs the S^T MFMAs of the NEXT tile and the PV MFMAs of the
  // PREVIOUS tile: every MFMA below is followed by the VALU work that hides it, LDS operands are
  // requested three MFMAs ahead, and sched_barrier pins that order.  The max reduction of the
  // next tile rides in the PV chunks.
  // Because PV lags one tile, so does the rescaling of O:
  //   at step j   O holds tiles <= j-2 relative to point m(j-2); alpha = 2^(m(j-2) - m(j-1)), tile j-1's
  //   step j      O *= alpha (rare branch), then O += P(j-1) V(j-1), both relative to m(j-1)
  // probabilities of the previous and of the current tile swap registers every step, like s_a / s_b
  v8i pf_x = {0, 0, 0, 0, 0, 0, 0, 0}, pf_y = {0, 0, 0, 0, 0, 0, 0, 0};
  // `at`: the step's position in the tile ring (j modulo kStages) where the loop is unrolled over the ring, so that every
  // LDS address is a constant; -1 in the loop over what remains.
  // byte offset into LDS of the next tile's K scale (a vector register on purpose: as a scalar it is moved to one at every use)
  int ks_off = (int)(reinterpret_cast<const uint8_t*>(s_ks) - smem) + 4;
  pin(ks_off);
  auto tile_step = [&](auto at, int j, v16i (&s_cur)[2], v16i (&s_nxt)[2], const v8i& pf_prev, v8i& pf, float& alpha, int& moved) {
    constexpr int kAt = decltype(at)::value;
    const uint8_t* kst = k_slot(kAt >= 0 ? kAt + 1 : j + 1);
    const uint8_t* vst = v_slot(kAt >= 0 ? kAt - 1 : j - 1);
    auto k_frag = [&](int i) { return *reinterpret_cast<const v4i*>(kst + ((qk_half(i) * 4 + qk_step(i)) * 64 + lane) * 16); };
    auto v_frag = [&](int dt) {
      const v4i lo = *reinterpret_cast<const v4i*>(vst + ((dt * 2 + 0) * 64 + lane) * 16);
      const v4i hi = *reinterpret_cast<const v4i*>(vst + ((dt * 2 + 1) * 64 + lane) * 16);
      return v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };
    v4i kf[4];
    v8i vf[4];
    // operands of the first three S^T MFMAs and the next tile's K scale
    kf[0] = k_frag(0);
    kf[1] = k_frag(1);
    kf[2] = k_frag(2);  // (kG >= 2: chunks 0 .. 3 always exist)
    // (one past the last tile's reads whatever follows the scales in LDS: a value nothing uses)
    const float ks_nxt = *reinterpret_cast<const float*>(smem + ks_off + (kAt >= 0 ? 4 * kAt : 0));
    if constexpr (kAt < 0) ks_off += 4;
    int entering = 0;  // the list entry the next step's window gains; it arrives with the operands above
    if constexpr (kSparse) entering = s_list[min(j + 1 + Shape::kAheadK, n_tiles - 1)];
    if (moved != 0) scale_o(alpha);  // wave-uniform
    // row sums of tile j-1: they cover the latency of the operands just requested
    lacc = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(ones, pf_prev, lacc, 0, 0, 0, 0, 0, 0);
    const float scp = kPwlExp ? 8.0f * sc : sc;
    const float cp = kPwlExp ? __builtin_fmaf(8.0f, xc, 55.5f) : xc;
    const bool skip = nothing;
    // The S^T chunks are short (a 32-cycle MFMA each): a wave inside them goes ahead of the SIMD's other
    // wave, which is usually in its PV chunks and has 64-cycle MFMAs to hide behind (measured: -1.3 %).
    __builtin_amdgcn_s_setprio(1);
    __builtin_amdgcn_sched_barrier(0);
    // 8 x [S^T MFMA of tile j+1 (32 matrix cycles) | 2 probabilities of tile j]
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int s = qk_step(i) & 3, t = qk_half(i) & 1;
      if (i + 3 < 8) {
        if (has_qk(i + 3)) kf[(i + 3) & 3] = k_frag(i + 3);
      } else if (i + 3 - 8 < kG) {
        vf[i + 3 - 8] = v_frag(i + 3 - 8);
      }
      // the copies, clear of the step's first operand reads and of the barrier (-1 % against issuing them at the head)
      if (i == 4) {
        if constexpr (kAt >= 0) issue_copy_at(at);
        else issue_copy(j);
      }
      if (has_qk(i)) s_nxt[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(kf[i & 3], qf[s], s == 0 ? magic : s_nxt[t], 0, 0, 0);
      if constexpr (kPwlExp) {
        unsigned w = (i & 1) ? (unsigned)pf[i >> 1] : 0u;
        w = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_fmaf(__int_as_float(s_cur[0][2 * i]), scp, cp), (2 * i) & 3, w);
        w = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_fmaf(__int_as_float(s_cur[0][2 * i + 1]), scp, cp), (2 * i + 1) & 3, w);
        int wi = (int)w;
        if (i & 1) pin(wi);
        pf[i >> 1] = wi;
      } else if (!skip) {
        const float e0 = p_of(s_cur[0][2 * i], scp, cp), e1 = p_of(s_cur[0][2 * i + 1], scp, cp);
        if (i & 1) {
          int w = __builtin_amdgcn_cvt_pk_fp8_f32(e0, e1, pf[i >> 1], true);
          pin(w);
          pf[i >> 1] = w;
        } else {
          pf[i >> 1] = __builtin_amdgcn_cvt_pk_fp8_f32(e0, e1, __float_as_int(e0), false);  // both halves get written
        }
      } else {
        pf[i >> 1] = 0;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (kCausal && !(kDiagApart && kAt >= 0)) {  // rare, wave-uniform: the next tile is the one on this wave's diagonal
      if (j + 1 < n_tiles && diag_at(j + 1)) blank_scores<kMagicBits>(s_nxt, hh, n_diag);
    }
    if constexpr (kAt < 0) {
      if (j + 1 == tail) blank_scores<kMagicBits>(s_nxt, hh, n_last);
    }
    __builtin_amdgcn_s_setprio(0);
    // 4 x [PV MFMA of tile j-1 (64 matrix cycles) | 4 probabilities of tile j | a quarter of
    // the max reduction of tile j+1, whose S^T MFMAs were issued at least one chunk ago]
    int mx = 0;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) {
      if (dt == 0 && kG == 4) vf[3] = v_frag(3);
      if (dt < kG) oacc[dt] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(vf[dt], pf_prev, oacc[dt], 0, 0, 0, 0, 0, 0);
      int w = 0;
      if (!skip) w = pack4(s_cur[1][4 * dt], s_cur[1][4 * dt + 1], s_cur[1][4 * dt + 2], s_cur[1][4 * dt + 3], scp, cp);
      pin(w);
      pf[4 + dt] = w;
      // one chain over the 32 scores, two per instruction
      const v16i& blk = s_nxt[dt >> 1];
      const int r0 = (dt & 1) * 8;
      mx = dt == 0 ? max(blk[0], blk[1]) : max(max(mx, blk[r0]), blk[r0 + 1]);
      mx = max(max(mx, blk[r0 + 2]), blk[r0 + 3]);
      mx = max(max(mx, blk[r0 + 4]), blk[r0 + 5]);
      mx = max(max(mx, blk[r0 + 6]), blk[r0 + 7]);
      pin(mx);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (kSparse) {
#pragma unroll
      for (int i = 0; i + 1 < kWindow; ++i) ahead[i] = ahead[i + 1];
      ahead[kWindow - 1] = __builtin_amdgcn_readfirstlane(entering) & 0xffff;
    }
    if constexpr (kSparse || (kCausal && !(kDiagApart && kAt >= 0))) {
      if (!mine_at(j)) {  // wave-uniform and rare: a tile this wave's row does not take part in contributes nothing
#pragma unroll
        for (int i = 0; i < 8; ++i) pf[i] = 0;
      }
      if (diag_at(j)) blank_probs(pf, hh, n_diag);
    }
    if constexpr (kAt < 0) {
      if (j == tail) blank_probs(pf, hh, n_last);
    }
    look_ahead(j + 1, mx, ks_nxt, alpha, moved);
    // after this barrier: K tile j+2 and V^T tile j are visible to every wave, and nobody reads their predecessors any
    // more (after a group's: K tiles up to j+5, V^T tiles up to j+3, the ones the next group reads)
    if constexpr (kAt < 0 || Shape::kGroup == 1) tile_barrier();
    else if constexpr ((kAt & (Shape::kGroup - 1)) == Shape::kGroup - 1) group_barrier();
  };

  {
    int j = 0;
    using Anywhere = std::integral_constant<int, -1>;
    if constexpr (kUnrolled) {
      auto two = [&](auto at) {
        constexpr int kAt = decltype(at)::value;
        tile_step(std::integral_constant<int, kAt>{}, j + kAt, s_a, s_b, pf_x, pf_y, alpha_odd, moved_odd);
        tile_step(std::integral_constant<int, kAt + 1>{}, j + kAt + 1, s_b, s_a, pf_y, pf_x, alpha_even, moved_even);
      };
      for (; j + kStages <= n_plain; j += kStages) {
        two(std::integral_constant<int, 0>{});
        two(std::integral_constant<int, 2>{});
        if constexpr (kStages == 8) {
          two(std::integral_constant<int, 4>{});
          two(std::integral_constant<int, 6>{});
        }
        ks_off += 4 * kStages;
      }
    }
    for (; j + 2 <= n_tiles; j += 2) {
      tile_step(Anywhere{}, j, s_a, s_b, pf_x, pf_y, alpha_odd, moved_odd);
      tile_step(Anywhere{}, j + 1, s_b, s_a, pf_y, pf_x, alpha_even, moved_even);
    }
    if (j < n_tiles) tile_step(Anywhere{}, j, s_a, s_b, pf_x, pf_y, alpha_odd, moved_odd);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no copy may outlive the workgroup's LDS
  {  // drain: PV of the last tile
    if ((n_tiles & 1) != 0) {
      if (moved_even != 0) scale_o(alpha_even);
    } else {
      if (moved_odd != 0) scale_o(alpha_odd);
    }
    const uint8_t* vst = v_slot(n_tiles - 1);
    const v8i pf_last = (n_tiles & 1) ? pf_y : pf_x;  // written by the last step
#pragma unroll
    for (int dt = 0; dt < kG; ++dt) pv_slice(vst, dt, pf_last);
    lacc = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(ones, pf_last, lacc, 0, 0, 0, 0, 0, 0);
  }

  if (is_run) {
    // partial result of this run of keys: O^T and the row sum relative to the run's own maximum
    const int row = wave * 32 + l32;
    float* po = p.split_o + ((int64_t)run_id * kAttnQPerWg + row) * kD;
#pragma unroll
    for (int dt = 0; dt < kG; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<float4*>(po + 32 * dt + 8 * g + 4 * hh) =
            make_float4(oacc[dt][4 * g + 0], oacc[dt][4 * g + 1], oacc[dt][4 * g + 2], oacc[dt][4 * g + 3]);
    if (hh == 0) reinterpret_cast<float2*>(p.split_ml)[(int64_t)run_id * kAttnQPerWg + row] = make_float2(m_run, lacc[0]);
    return;
  }
  // ---- epilogue: O = O^T / rowsum * v_scale (+ the V mean), written [B, Lq, H, D] ---------------
  // A lane holds its query row in pieces of four channels; stored as they are, every store instruction would
  // touch 32 rows with 16 bytes each.  The rows go through LDS instead (the tile ring is free once every wave is
  // past its last tile) and leave as whole 256-byte rows, 16 bytes per lane.
  // zero for a mask row that allows none of its keys (an empty sum, not 0/0)
  const float inv_l = !(kSparse || kCausal) || lacc[0] > 0.0f ? 1.0f / lacc[0] : 0.0f;
  // the channel means the V quantizer took off come back here (rows of P sum to one); they are zeros without V
  // smoothing, and a row that saw no key stays zero
  const float keep_mean = inv_l != 0.0f ? 1.0f : 0.0f;
  constexpr int kPitch = 2 * kD + 16;  // bytes per staged row: 16 bytes of padding spread the rows over the banks
  // The lane's 16 quadruples of V scales are requested together and ahead of the barrier (the score registers are
  // free by now); read one quadruple at a time where they are used, every one of the 16 groups below would start
  // with an LDS round trip of its own.  Without V smoothing the means are all zero - seen here by the wave as a
  // whole - and their products and sums are left out (a zero output may then keep a minus sign it used to lose).
  uint8_t* stage = smem + wave * (32 * kPitch);
  const float4* vs4 = reinterpret_cast<const float4*>(s_vs);
  const float4* vm4 = reinterpret_cast<const float4*>(s_vs + kD);
  float4 s4a[16];
#pragma unroll
  for (int i = 0; i < 4 * kG; ++i) s4a[i] = vs4[(32 * (i >> 2) + 8 * (i & 3) + 4 * hh) >> 2];
  if constexpr (kLinear) {
    // The linear branch of the lane's row, of the row as the caller has it, and the sum of the two results, each rounded to
    // the half type first - what a pass of its own (sla_apply_kernel) gives, bit for bit.  A lane of that product holds the
    // same channels of the same row as a lane of O^T, so the sum is taken in registers.  LDS from the ring's start: the
    // head's matrix, ksum and bias, the staged rows (the V scales have been read; no V means on this path).  The matrix
    // is on its way while the row's exponentials are taken.
    // As a pass of its own the branch reads q and the result and writes the result again, 1 GB at 32760 rows of 40 heads,
    // bound by memory; here its arithmetic runs beside the neighbour workgroup's key loop.  us per call, a tenth of the keys
    // kept, pass of its own / here: 40 heads of 32760 rows 2000 / 1859, of 6867 272 / 230, 12 of 2000 72 / 52.
    const uint16_t* lrow = p.q_rows.ptr + b * p.q_rows.sB + (int64_t)min(q0 + l32, p.Lq - 1) * p.q_rows.sL + h * p.q_rows.sH + 8 * hh;
    uint4 lraw[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) lraw[s] = *reinterpret_cast<const uint4*>(lrow + 16 * s);
    const float2 ks2 = reinterpret_cast<const float2*>(p.lin.ksum + (int64_t)bh * kD)[lane];
    float2 bias2 = make_float2(0.0f, 0.0f);
    if (p.lin.bias != nullptr) bias2 = reinterpret_cast<const float2*>(p.lin.bias)[lane];
    uint2 oh[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int dt = i >> 2, g = i & 3;
      float o4[4] = {oacc[dt][4 * g + 0] * inv_l * s4a[i].x, oacc[dt][4 * g + 1] * inv_l * s4a[i].y,
                     oacc[dt][4 * g + 2] * inv_l * s4a[i].z, oacc[dt][4 * g + 3] * inv_l * s4a[i].w};
      // (pinned: the product and the conversion may otherwise become one fp16 instruction, with one rounding instead of two)
#pragma unroll
      for (int e = 0; e < 4; ++e) pin(o4[e]);
      oh[i] = half4<DT>(o4[0], o4[1], o4[2], o4[3]);
    }
    __syncthreads();  // waves that ended early (no query rows) do not count
    constexpr int kMatBytes = kD * kD * 2;
    const uint8_t* mat = reinterpret_cast<const uint8_t*>(p.lin.frag + (int64_t)bh * kD * kD);
    const int n_waves = min(kW, (lq - qwg * kRowsWg + 31) >> 5);  // the waves still here share the copies
    if (n_waves == kW) {
#pragma unroll
      for (int i = 0; i < kMatBytes / 1024 / kW; ++i) lds_copy16(mat, (unsigned)((i * kW + wave) * 64 + lane) * 16, smem + (i * kW + wave) * 1024);
    } else {
#pragma unroll 1
      for (int i = wave; i < kMatBytes / 1024; i += n_waves) lds_copy16(mat, (unsigned)(i * 64 + lane) * 16, smem + i * 1024);
    }
    float* s_ksum = reinterpret_cast<float*>(smem + kMatBytes);
    float* s_bias = s_ksum + kD;
    if (wave == 0) {
      reinterpret_cast<float2*>(s_ksum)[lane] = ks2;
      reinterpret_cast<float2*>(s_bias)[lane] = bias2;
    }
    float x[8][8];
    const float rinv = sla_row_exps<DT>(lraw, x);
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    uint4 fq[8];
    const float scale = sla_row_scale<DT>(x, rinv, s_ksum, hh, fq);
    stage = smem + kMatBytes + 2 * kD * 4 + wave * (32 * kPitch);
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) {
      const v16f lin = sla_row_product<DT>(reinterpret_cast<const uint4*>(smem), fq, dt, lane);
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int d = 32 * dt + 8 * g + 4 * hh;
        const float4 bs = *reinterpret_cast<const float4*>(s_bias + d);
        const uint2 lh = half4<DT>(__builtin_fmaf(lin[4 * g + 0], scale, bs.x), __builtin_fmaf(lin[4 * g + 1], scale, bs.y),
                                   __builtin_fmaf(lin[4 * g + 2], scale, bs.z), __builtin_fmaf(lin[4 * g + 3], scale, bs.w));
        float a4[8], o4[8];
        widen8<DT>(make_uint4(lh.x, lh.y, 0, 0), a4);
        widen8<DT>(make_uint4(oh[4 * dt + g].x, oh[4 * dt + g].y, 0, 0), o4);
        *reinterpret_cast<uint2*>(stage + l32 * kPitch + 2 * d) = half4<DT>(a4[0] + o4[0], a4[1] + o4[1], a4[2] + o4[2], a4[3] + o4[3]);
      }
    }
  } else {
    const float2 mm = reinterpret_cast<const float2*>(s_vs + kD)[lane];
    const bool has_mean = __any(mm.x != 0.0f || mm.y != 0.0f);  // wave-uniform
    __syncthreads();  // waves that ended early (no query rows) do not count
    if (!has_mean) {
#pragma unroll
      for (int i = 0; i < 4 * kG; ++i) {
        const int dt = i >> 2, g = i & 3;
        const int d = 32 * dt + 8 * g + 4 * hh;
        const float4 s4 = s4a[i];
        *reinterpret_cast<uint2*>(stage + l32 * kPitch + 2 * d) =
            half4<DT>(oacc[dt][4 * g + 0] * inv_l * s4.x, oacc[dt][4 * g + 1] * inv_l * s4.y,
                      oacc[dt][4 * g + 2] * inv_l * s4.z, oacc[dt][4 * g + 3] * inv_l * s4.w);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4 * kG; ++i) {
        const int dt = i >> 2, g = i & 3;
        const int d = 32 * dt + 8 * g + 4 * hh;
        const float4 s4 = s4a[i];
        const float4 m4 = vm4[d >> 2];
        *reinterpret_cast<uint2*>(stage + l32 * kPitch + 2 * d) =
            half4<DT>(oacc[dt][4 * g + 0] * inv_l * s4.x + m4.x * keep_mean, oacc[dt][4 * g + 1] * inv_l * s4.y + m4.y * keep_mean,
                      oacc[dt][4 * g + 2] * inv_l * s4.z + m4.z * keep_mean, oacc[dt][4 * g + 3] * inv_l * s4.w + m4.w * keep_mean);
      }
    }
    // rows at or beyond lq (zeros put in their place and not a factor of zero: what q holds there, or v, need not be finite)
    if (q0 + 32 > lq && q0 + l32 >= lq) {
#pragma unroll
      for (int i = 0; i < 2 * kG; ++i) *reinterpret_cast<uint4*>(stage + l32 * kPitch + 32 * i + 16 * hh) = make_uint4(0, 0, 0, 0);
    }
  }
  // LDS serves one wave's accesses in order: the reads below see the writes above
  uint16_t* obase = p.o.ptr + b * p.o.sB + h * p.o.sH;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int idx = i * 64 + lane, r = idx >> 4, c = idx & 15;  // row r of the wave, 16-byte piece c of it
    const uint4 piece = *reinterpret_cast<const uint4*>(stage + r * kPitch + 16 * c);
    if (q0 + r < p.Lq && 8 * c < p.d_out && 8 * c < 32 * kG) *reinterpret_cast<uint4*>(obase + (int64_t)(q0 + r) * p.o.sL + 8 * c) = piece;
  }
}

// Combines the partial results of the key runs: for every query row the run maxima are brought to a common one,
// then O = sum_i O_i 2^(m_i - m), l = sum_i l_i 2^(m_i - m), and the usual last step follows.
// grid = (items, 32), 256 threads: a thread owns one row and four channels of a 8-row slab.
template <int DT>
__global__ __launch_bounds__(256) void sage_attn_merge_kernel(const AttnParams p, int n_qwg) {
  const int item = blockIdx.x, wg = p.split_first_wg + item;
  const int bh = wg / n_qwg, qwg = wg - bh * n_qwg;
  const int b = bh / p.Hq, h = bh - b * p.Hq;
  const int bhk = b * p.Hkv + h / (p.Hq / p.Hkv);
  const int row = blockIdx.y * 8 + (threadIdx.x >> 5), d = (threadIdx.x & 31) * 4;
  const int q = qwg * kAttnQPerWg + row;
  if (q >= p.Lq || d >= p.d_out) return;
  uint16_t* orow = p.o.ptr + b * p.o.sB + (int64_t)q * p.o.sL + h * p.o.sH;
  if (p.q_lens != nullptr && q >= rows_counted(p.q_lens[b], p.Lq)) {  // a row that does not take part: zeros
    *reinterpret_cast<uint2*>(orow + d) = make_uint2(0, 0);
    return;
  }
  const float2* ml = reinterpret_cast<const float2*>(p.split_ml) + (int64_t)item * p.n_split * kAttnQPerWg + row;
  const float* po = p.split_o + ((int64_t)item * p.n_split * kAttnQPerWg + row) * kD + d;
  // Eight runs at a time, their loads in flight together: one run after the other, a row waits for as many memory
  // latencies as it has runs (8 query blocks of 32 runs: 29.5 us, 10.5 like this).
  constexpr int kAtOnce = 8;
  float m = -INFINITY;
  for (int s0 = 0; s0 < p.n_split; s0 += kAtOnce) {
    float mm[kAtOnce];
#pragma unroll
    for (int i = 0; i < kAtOnce; ++i) mm[i] = ml[(int64_t)min(s0 + i, p.n_split - 1) * kAttnQPerWg].x;
#pragma unroll
    for (int i = 0; i < kAtOnce; ++i) m = fmaxf(m, mm[i]);
  }
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  float l = 0.0f;
  for (int s0 = 0; s0 < p.n_split; s0 += kAtOnce) {
    float2 e[kAtOnce];
    float4 o[kAtOnce];
#pragma unroll
    for (int i = 0; i < kAtOnce; ++i) {
      const int64_t at = min(s0 + i, p.n_split - 1);
      e[i] = ml[at * kAttnQPerWg];
      o[i] = *reinterpret_cast<const float4*>(po + at * (kAttnQPerWg * kD));
    }
#pragma unroll
    for (int i = 0; i < kAtOnce; ++i) {
      if (s0 + i >= p.n_split || e[i].y == 0.0f) continue;  // (no such run, or an empty one, whose maximum is -inf)
      const float w = fast_exp2(e[i].x - m);
      acc.x += o[i].x * w, acc.y += o[i].y * w, acc.z += o[i].z * w, acc.w += o[i].w * w;
      l += e[i].y * w;
    }
  }
  const float inv_l = l > 0.0f ? 1.0f / l : 0.0f;
  const float keep_mean = l > 0.0f ? 1.0f : 0.0f;
  const float4 s4 = *reinterpret_cast<const float4*>(p.v_scale + (int64_t)bhk * kD + d);
  const float4 m4 = *reinterpret_cast<const float4*>(p.v_mean + (int64_t)bhk * kD + d);
  store4<DT>(orow + d, acc.x * inv_l * s4.x + m4.x * keep_mean, acc.y * inv_l * s4.y + m4.y * keep_mean,
             acc.z * inv_l * s4.z + m4.z * keep_mean, acc.w * inv_l * s4.w + m4.w * keep_mean);
}

// dynamic LDS of one instantiation: tile ring + K scales (+ the tile list and its length with a mask or causal)
template <bool kSparse, int kW>
constexpr size_t max_lds() {
  return kSparse ? WgShape<kW>::kRingBytes + 1024 + (kW == 8 ? kSparseMaxKeyTiles * 8 : kSparseMaxKeyTiles4 * 6) + 1024
                 : WgShape<kW>::kRingBytes + 2048 + (kW == 8 ? kMaxKeyTiles : kShortMaxKeyTiles) * 4;
}

template <int DT, bool kPwlExp, bool kSparse, int kW, bool kCausal, bool kTileSkip = false, int kG = 4, bool kLinear = false, bool kNumbered = false>
hipError_t launch_variant(const AttnParams& p, dim3 grid, size_t lds, int n_qwg, int n_wg, int wg_per_xcd,
                          hipStream_t s) {
  // more than 64 KiB of dynamic LDS has to be requested per kernel, once per device
  constexpr int kMaxDevices = 64;
  static std::atomic<bool> requested[kMaxDevices];
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  if (!requested[dev].load(std::memory_order_acquire)) {
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(&sage_attn_fwd_kernel<DT, kPwlExp, kSparse, kW, kTileSkip, kG, kCausal, kLinear, kNumbered>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)max_lds<kSparse, kW>());
    if (e != hipSuccess) return e;
    requested[dev].store(true, std::memory_order_release);
  }
  sage_attn_fwd_kernel<DT, kPwlExp, kSparse, kW, kTileSkip, kG, kCausal, kLinear, kNumbered><<<grid, dim3(kW * 64), lds, s>>>(p, n_qwg, n_wg, wg_per_xcd);
  return hipGetLastError();
}

// Causal calls without a block mask, in the default variant: key tiles are walked without a list, and the steps before the
// diagonal are the dense loop's.  us per call, tile list / this: 8 191 tokens of 32 heads (8 of keys) 350 / 323, 12 x 7 411
// 151 / 142, 40 x 32 760 6 285 / 5 820, 20 000 tokens of one head 239 / 207, 40 x 1 024 36.9 / 35.3.  (8 waves: 2 % faster from
// eight rounds of 90 blocks per head, 5 - 30 % slower in short grids; not built.)
hipError_t launch_causal(const AttnParams& p, dim3 grid, size_t lds, int n_qwg, int n_wg, int wg_per_xcd, hipStream_t s) {
  const bool bf16 = p.o.dtype == KSANA_SAGE_BF16;
  if (p.d_out <= 64)
    return bf16 ? launch_variant<KSANA_SAGE_BF16, false, false, 4, true, false, 2>(p, grid, lds, n_qwg, n_wg, wg_per_xcd, s)
                : launch_variant<KSANA_SAGE_FP16, false, false, 4, true, false, 2>(p, grid, lds, n_qwg, n_wg, wg_per_xcd, s);
  return bf16 ? launch_variant<KSANA_SAGE_BF16, false, false, 4, true>(p, grid, lds, n_qwg, n_wg, wg_per_xcd, s)
              : launch_variant<KSANA_SAGE_FP16, false, false, 4, true>(p, grid, lds, n_qwg, n_wg, wg_per_xcd, s);
}

// the (dtype, exp2 form, tile skip) instantiations behind one (mask, workgroup shape) choice
template <bool kSparse, int kW, bool kCausal = false>
hipError_t launch_shape(const AttnParams& p, dim3 grid, size_t lds, int n_qwg, int n_wg, int wg_per_xcd, hipStream_t s) {
  const bool bf16 = p.o.dtype == KSANA_SAGE_BF16;
  // head size 64: the matrix instructions on the zero halves are left out (plain exact-exponential calls; the other
  // variants run the full-width code on the same operands, which gives the same bits)
  if constexpr (!kSparse && !kCausal)
    if (p.numbered != 0) {
      if (p.d_out <= 64)
        return bf16 ? launch_variant<KSANA_SAGE_BF16, false, false, kW, false, false, 2, false, true>(p, grid, lds, n_qwg, n_wg, wg_per_xcd, s)
                    : launch_variant<KSANA_SAGE_FP16, false, false, kW, false, false, 2, false, true>(p, grid, lds, n_qwg, n_wg, wg_per_xcd, s);
      return bf16 ? launch_variant<KSANA_SAGE_BF16, false, false, kW, false, false, 4, false, true>(p, grid, lds, n_qwg, n_wg, wg_per_xcd, s)
                  : launch_variant<KSANA_SAGE_FP16, false, false, kW, false, false, 4, false, true>(p, grid, lds, n_qwg, n_wg, wg_per_xcd, s);
    }
  if (p.exact_exp2 && !p.tile_skip && p.d_out <= 64)
    return bf16 ? launch_variant<KSANA_SAGE_BF16, false, kSparse, kW, kCausal, false, 2>(p, grid, lds, n_qwg, n_wg, wg_per_xcd, s)
                : launch_variant<KSANA_SAGE_FP16, false, kSparse, kW, kCausal, false, 2>(p, grid, lds, n_qwg, n_wg, wg_per_xcd, s);
  if (p.exact_exp2 && p.tile_skip)
    return bf16 ? launch_variant<KSANA_SAGE_BF16, false, kSparse, kW, kCausal, true>(p, grid, lds, n_qwg, n_wg, wg_per_xcd, s)
                : launch_variant<KSANA_SAGE_FP16, false, kSparse, kW, kCausal, true>(p, grid, lds, n_qwg, n_wg, wg_per_xcd, s);
  if (p.exact_exp2)
    return bf16 ? launch_variant<KSANA_SAGE_BF16, false, kSparse, kW, kCausal>(p, grid, lds, n_qwg, n_wg, wg_per_xcd, s)
                : launch_variant<KSANA_SAGE_FP16, false, kSparse, kW, kCausal>(p, grid, lds, n_qwg, n_wg, wg_per_xcd, s);
  return bf16 ? launch_variant<KSANA_SAGE_BF16, true, kSparse, kW, kCausal>(p, grid, lds, n_qwg, n_wg, wg_per_xcd, s)
              : launch_variant<KSANA_SAGE_FP16, true, kSparse, kW, kCausal>(p, grid, lds, n_qwg, n_wg, wg_per_xcd, s);
}

// compute units of the current device (the size of one round of workgroups: one workgroup per unit)
int compute_units() {
  constexpr int kMaxDevices = 64;
  static std::atomic<int> cached[kMaxDevices];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return 256;
  int n = cached[dev].load(std::memory_order_acquire);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cached[dev].store(n, std::memory_order_release);
  }
  return n;
}

}  // namespace

// How a dense call is laid out: workgroups of 4 or 8 waves, and (8 waves) the first workgroup that is cut into runs of
// key tiles, and into how many (0: none).
struct DensePlan {
  int waves, first_cut, runs;
};

// n_wg: the grid in 256-row workgroups, nkb: key tiles.  The choice is between
//   8 waves        one workgroup per compute unit: the lowest time per tile, but the workgroups beyond the last full round
//                  of the chip take most of a round however few they are (alone, they run a third faster),
//   8 waves, cut   those workgroups as runs of keys that fill the chip: a short round, then the merge kernel,
//   4 waves        two workgroups per compute unit, which hide each other's set-up and epilogue; in an incomplete round
//                  one alone on its unit takes half the time.
// Estimates in units of one tile of an 8-wave workgroup (about a microsecond), fitted to measurements of grids of 0.03 ..
// 4.5 rounds and 8 .. 200 tiles: a full round of T tiles takes 1.005 T + 5.5 (8 waves) or 1.05 T + 4.5 (4 waves).  An
// incomplete one takes at least 0.75 of that in 8 waves; in 4 waves 0.5 up to half full and its own filling and 0.1 more
// from there (0.55 and 0.17 more where it is the only round).  Runs of keys take their own tiles, and writing and merging
// up to 256 partial results of 128 KiB costs 5 .. 15.
// Examples, us, 4 waves / 8 waves cut: 2.25 rounds of 96 tiles 258 / 242, 1.1 of 68 tiles 114 / 97, 3.1 of 80 tiles
// 312 / 282; but a quarter of a round of 20 tiles 17 / 28, of 32 tiles 24 / 32.
static DensePlan plan_dense(int n_wg, int nkb) {
  const int cus = compute_units();
  const int rounds = n_wg / cus, rest = n_wg % cus;
  int runs = 0;
  if (rest != 0 && 2 * rest <= cus && nkb > kShortKeyTiles) {
    runs = min(min(cus / rest, kMaxSplitPartials / rest), nkb / kMinTilesPerSplit);
    if (runs < 2) runs = 0;
  }
  if (n_wg <= cus / 16 && runs != 0) return DensePlan{8, 0, runs};  // a handful of workgroups: as many runs as there are
  const float part = (float)rest / (float)cus, alone = rounds == 0 ? 1.0f : 0.0f;
  const float round8 = 1.005f * (float)nkb + 5.5f, round4 = 1.05f * (float)nkb + 4.5f;
  const float whole8 = ((float)rounds + (rest == 0 ? 0.0f : fmaxf(0.75f, part))) * round8 + 4.0f * alone;
  const float cut8 = runs == 0 ? INFINITY
                               : (float)rounds * round8 + 0.9f * ((float)((nkb + runs - 1) / runs) + 5.5f) + 5.0f +
                                     10.0f * (float)(rest * runs) / (float)cus;
  const float part4 = rest == 0         ? 0.0f
                      : 2 * rest <= cus ? 0.5f + 0.045f * alone
                                        : fminf(1.0f, part + 0.1f + 0.07f * alone);
  const float whole4 = nkb > kShortMaxKeyTiles ? INFINITY : ((float)rounds + part4) * round4 + 3.6f * alone;
  if (whole4 < fminf(whole8, cut8)) return DensePlan{4, n_wg, 0};
  if (cut8 < whole8) return DensePlan{8, n_wg - rest, runs};
  return DensePlan{8, n_wg, 0};
}

void plan_key_split(int n_wg, int nkb, int* first_wg, int* runs) {
  const DensePlan plan = plan_dense(n_wg, nkb);
  *first_wg = plan.first_cut, *runs = plan.runs;
}

// Quantized in the attention kernel, Q is read once (2 bytes per channel where the quantizer's pass moves 4 with its reading
// back), for its transform in every workgroup's set-up.  us replayed from a graph, through memory / in the kernel, by blocks of 256
// rows and on 300, 600, 1024, 2048, 4096 keys:
//    32 blocks   17.8 / 18.6   21.1 / 21.9   25.4 / 26.0   36.6 / 37.5     46.8 / 47.1
//    96          20.2 / 19.9   24.5 / 24.1   29.0 / 28.8   43.4 / 42.4     70.1 / 69.5
//   160          24.5 / 23.8   31.5 / 30.2   37.9 / 36.8   56.9 / 56.3     96.3 / 95.5
//   256          30.5 / 27.5   38.8 / 35.5   49.3 / 46.2   80.1 / 77.1    145.6 / 143.2
//   320          38.2 / 34.9   50.0 / 45.9   62.9 / 60.6  102.4 / 99.1    181.6 / 179.1
// That pays
//   from one full round of the chip: below it every workgroup's set-up is exposed, and the quantizer's Q blocks ride in
//     the launches of K and V.  (The line is older than the present set-up, whose break-even is near 96 blocks; between the
//     two 1-7 % are left.)
//   beyond 256 keys: up to there all quantizers are one launch (256 blocks, 2 tiles 23.0 / 24.1 and 8 tiles 33.1 / 30.0 with an
//     earlier set-up; calls of one round on so few keys are one launch altogether, see small_call_suits);
//   up to 256 tiles: there the gain is half a per cent (40 heads of 16384 rows on 2048 keys 447.5 / 426.7, 8192 1439 / 1413, 16384
//     2726 / 2715), and on chips at their power limit the instructions cost the key loop as much (24000 keys 3962 / 3969).
bool q_in_attention_pays(int n_wg, int nkb) { return n_wg >= compute_units() && nkb * kBlkK > kMeanChunk && nkb <= 256; }

// Workgroup shape for a call: 4-wave workgroups (two per compute unit) when a block mask or causal masking is
// involved (a workgroup is then one 128-row mask row, so no wave multiplies a tile only the neighbouring mask row
// asked for), plan_dense's choice otherwise.  p.wg_waves (4 or 8) overrides the choice.
static int pick_wg_waves(const AttnParams& p) {
  if (p.wg_waves == 4 || p.wg_waves == 8) return p.wg_waves;
  const bool sparse = p.block_mask != nullptr || p.causal;
  if (sparse) return p.nkb <= kSparseMaxKeyTiles4 ? 4 : 8;
  return plan_dense(p.B * p.Hq * ((p.Lq + kAttnQPerWg - 1) / kAttnQPerWg), p.nkb).waves;
}

// Grid of a launch whose workgroups are numbered in runs per XCD (see the kernel's first lines), and the run's length.
// Per-entry counts live in device memory, so entries of a batch that has any are taken to be unequal.
static dim3 xcd_grid(AttnParams* p, int n_qwg, int n_wg, int* wg_per_xcd) {
  p->batch_run = p->B > 1 && (p->k_lens != nullptr || p->q_lens != nullptr) ? (p->Hq * n_qwg + 7) / 8 : 0;
  *wg_per_xcd = p->batch_run != 0 ? p->batch_run * p->B : (n_wg + 7) / 8;
  return dim3(*wg_per_xcd * 8);
}

// Dense calls in the default variant, uncut, of more than one round - one round has no order - and up to four and a half.  us, by the
// tensor's numbering / by the counts (entries full, falling to or rising from 45 %, half full, of random counts):
//                                        full          falling         rising          half          random
//   2 x 12 heads of 6946 on 138 (2.6)    42.5 / 43.3   38.7 / 37.2     38.5 / 38.1     34.1 / 32.2   37.2 / 35.0
//   2 x 24 of 3500 (2.6)                 216 / 216     151.4 / 152.9   167.2 / 152.2   98.8 / 100    140.7 / 140.4
//   3 x 24 of 3001 on 4099 (3.4)         287.5 / 288   187.4 / 183.7   195.7 / 183.4   104 / 102.4   132.6 / 135.8
//   5 x 32 of 1500 (3.8)                 181 / 181     142 / 129.5     139 / 129.5     103 / 93      147 / 155
//   6 x 24 of 2000 (4.5)                 246 / 247     175 / 170       177 / 171       120 / 119     137 / 132
//   8 x 24 of 1000 on 600 (3.0)          82.0 / 82.2   69.5 / 66.0     70.0 / 66.9     53.2 / 51.3   62.6 / 58.0
// What full entries can lose, up to 0.8 us a call, is the load of the numbers ahead of the counts.  In longer grids the last round's
// order is a smaller part, and gains and losses cancel: eight shapes of 5 to 15 rounds in eight such sets of counts 0.991 on average, 0.92
// to 1.05 each (6 x 64 of 2000, 12 rounds, half full 331 / 347: blocks that start together keep in step).
int batch_rows_wg(const AttnParams& p) {
  if (p.B < 2 || p.B > kBatchEntries || (p.q_lens == nullptr && p.k_lens == nullptr) || p.block_mask != nullptr || p.causal || !p.exact_exp2 || p.tile_skip ||
      p.nkb > kMaxKeyTiles)
    return 0;
  int waves = pick_wg_waves(p);
  if (waves == 4 && p.nkb > kShortMaxKeyTiles) waves = 8;
  const int rows = 32 * waves, n_wg = p.B * p.Hq * ((p.Lq + rows - 1) / rows);
  const int round = (waves == 4 ? 2 : 1) * compute_units();
  if (n_wg <= round || 2 * n_wg > 9 * round) return 0;
  if (waves == 8) {
    int first = n_wg, runs = 0;
    plan_key_split(n_wg, p.nkb, &first, &runs);
    if (runs != 0) return 0;
  }
  return rows;
}

hipError_t launch_attn_fwd(const AttnParams& params, hipStream_t s) {
  AttnParams p = params;
  p.split_first_block = INT32_MAX;
  if (p.nkb > kMaxKeyTiles) return hipErrorInvalidValue;
  const bool sparse = p.block_mask != nullptr || p.causal;
  if (sparse && p.nkb > kSparseMaxKeyTiles) return hipErrorInvalidValue;
  if (p.q_rows.ptr != nullptr && resident_call_suits(p)) return launch_resident(p, s);
  const bool plain_causal = p.causal && p.block_mask == nullptr && p.exact_exp2 && !p.tile_skip;  // no tile list
  int waves = pick_wg_waves(p);
  if (waves == 4 && p.nkb > (sparse ? kSparseMaxKeyTiles4 : kShortMaxKeyTiles)) waves = 8;
  const int rows = 32 * waves;
  const int n_qwg = (p.Lq + rows - 1) / rows;
  const int n_wg = p.B * p.Hq * n_qwg;
  int wg_per_xcd = 0;
  dim3 grid = xcd_grid(&p, n_qwg, n_wg, &wg_per_xcd);
  if (p.numbered != 0) {
    if (batch_rows_wg(p) != rows) return hipErrorInvalidValue;
    grid = dim3(8 * p.B * (p.batch_run + 1));  // (either kind of an entry's blocks is divided by eight)
  }
  if (p.causal && p.batch_run == 0) p.causal_grid = causal_grid(p.B * p.Hq, n_qwg);  // (the same number of workgroups)
  // tile ring + the head's K scales (a multiple of 1 KiB keeps the request tidy)
  const size_t lds = (waves == 4 ? WgShape<4>::kRingBytes : WgShape<8>::kRingBytes) + 1024 + (((size_t)(p.nkb + 1) * 4 + 1023) & ~size_t(1023));
  if (p.lin.frag != nullptr) {
    if (waves != 4 || p.block_mask == nullptr || p.causal || !p.exact_exp2 || p.tile_skip || p.d_out != kD || p.q_lens != nullptr ||
        p.k_lens != nullptr)
      return hipErrorInvalidValue;
    return p.o.dtype == KSANA_SAGE_BF16
               ? launch_variant<KSANA_SAGE_BF16, false, true, 4, false, false, 4, true>(p, grid, max_lds<true, 4>(), n_qwg, n_wg, wg_per_xcd, s)
               : launch_variant<KSANA_SAGE_FP16, false, true, 4, false, false, 4, true>(p, grid, max_lds<true, 4>(), n_qwg, n_wg, wg_per_xcd, s);
  }
  // Dense calls whose heads end in a short block, of at most half a workgroup's rows, and that take a round less without these: the
  // short ones start last, so that the round they do not fit into is longer by one of them and not by a whole block.  us, in the order
  // of their index / last, 4 waves: 40 heads of 1560 tokens (1.02 rounds) 56.7 / 54.8, 2 x 32 of 1062 (1.1) 58.7 / 55.5, 4 x 40 of 416
  // on 2446 (1.25) 107 / 95.5, 4 x 24 of 2110 (3.2, 64 channels) 130 / 123.4, 4 x 40 of 6185 on 819 (15.3) 357 / 359; 8 waves: 4 x 64 of 624
  // on 4389 (3.0) 359 / 346.5, of 541 on 2302 (3.0) 238 / 241.5; 45 such calls 0.979 on average.  Where the rounds are as many without them
  // it is no gain: 45 calls 1.003, 64 of 3603 (3.75) 296 / 301, 4 x 16 of 1551 (1.75) 87.5 / 89.1; below a round 12 of 2873 63.1 / 64.3.
  auto small_blocks_last = [&]() {
    const int pairs = p.B * p.Hq, round = (waves == 4 ? 2 : 1) * compute_units();
    if (sparse || p.batch_run != 0 || n_qwg < 2 || 2 * (p.Lq - (n_qwg - 1) * rows) > rows) return;
    if ((n_wg - pairs + round - 1) / round == (n_wg + round - 1) / round) return;
    p.small_last = (pairs + 7) / 8;
    wg_per_xcd = (pairs * (n_qwg - 1) + 7) / 8 + p.small_last;
    grid = dim3(wg_per_xcd * 8);
  };
  if (waves == 4) {
    small_blocks_last();
    if (plain_causal) return launch_causal(p, grid, lds, n_qwg, n_wg, wg_per_xcd, s);
    if (sparse)
      return p.causal ? launch_shape<true, 4, true>(p, grid, max_lds<true, 4>(), n_qwg, n_wg, wg_per_xcd, s)
                      : launch_shape<true, 4, false>(p, grid, max_lds<true, 4>(), n_qwg, n_wg, wg_per_xcd, s);
    return launch_shape<false, 4>(p, grid, lds, n_qwg, n_wg, wg_per_xcd, s);
  }
  // (tile lists in 256-row workgroups, by flag only: one instantiation serves causal and plain calls)
  if (sparse) return launch_shape<true, 8, true>(p, grid, max_lds<true, 8>(), n_qwg, n_wg, wg_per_xcd, s);
  // The workgroups beyond the last full round of the chip (one workgroup per compute unit) would hold it for a
  // whole round alone.  When they are few, each is cut into runs of key tiles that together fill a round, and a
  // small kernel merges the runs: 2568 workgroups are then 10 rounds and a bit instead of 11, 280 are 1.1 instead of 2.
  int n_full = n_wg, n_split = 0;
  if (p.split_o != nullptr) plan_key_split(n_wg, p.nkb, &n_full, &n_split);
  if (n_split == 0) {
    small_blocks_last();
    return launch_shape<false, 8>(p, grid, lds, n_qwg, n_wg, wg_per_xcd, s);
  }
  const int rest = n_wg - n_full;
  const dim3 grid_full = n_full > 0 ? xcd_grid(&p, n_qwg, n_full, &wg_per_xcd) : dim3(0);
  p.split_first_block = (int)grid_full.x;
  p.split_first_wg = n_full;
  p.n_split = n_split;
  const hipError_t e = launch_shape<false, 8>(p, dim3(grid_full.x + rest * n_split), lds, n_qwg, n_full, wg_per_xcd, s);
  if (e != hipSuccess) return e;
  if (p.o.dtype == KSANA_SAGE_BF16)
    sage_attn_merge_kernel<KSANA_SAGE_BF16><<<dim3(rest, kAttnQPerWg / 8), dim3(256), 0, s>>>(p, n_qwg);
  else
    sage_attn_merge_kernel<KSANA_SAGE_FP16><<<dim3(rest, kAttnQPerWg / 8), dim3(256), 0, s>>>(p, n_qwg);
  return hipGetLastError();
}

}  // namespace ksana_sage
