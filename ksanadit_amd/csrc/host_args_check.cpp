// Host-side check of the C ABI's argument validation, meant to be built with AddressSanitizer on the host pass
// (ksanadit_amd/build_host_check.py) and run on a machine without a GPU: every call below must be refused by the
// library before it touches a device, so whatever the host code reads on the way - shapes, strides, the descriptor
// of the step before attention, the host-resident grid sizes - is read under the sanitizer.  Exit code 0 = every
// call returned what it should; the sanitizer aborts the process on a bad access.
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <vector>

#include "../../include/ksana_sage_hip.h"
#include "sage_kernels.h"

// Counts of batch entries are any int32, clamped to the tensor before anything is added to them.  As constant expressions: an
// overflow on the way is an error of the build.
static_assert(ksana_sage::tiles_counted(INT32_MAX, 5) == 5 && ksana_sage::tiles_counted(INT32_MAX - 63, 5) == 5);
static_assert(ksana_sage::tiles_counted(321, 5) == 5 && ksana_sage::tiles_counted(257, 5) == 5 && ksana_sage::tiles_counted(256, 5) == 4);
static_assert(ksana_sage::tiles_counted(1, 5) == 1 && ksana_sage::tiles_counted(0, 5) == 0);
static_assert(ksana_sage::tiles_counted(-1, 5) == 0 && ksana_sage::tiles_counted(INT32_MIN, 5) == 0);
static_assert(ksana_sage::rows_counted(INT32_MAX, 300) == 300 && ksana_sage::rows_counted(299, 300) == 299 && ksana_sage::rows_counted(INT32_MIN, 300) == 0);

static int g_failed = 0;
#define EXPECT(call, want)                                                                        \
  do {                                                                                            \
    const int rc_ = (call);                                                                       \
    if (rc_ != (want)) {                                                                          \
      ++g_failed;                                                                                 \
      std::printf("line %d: %s -> %d (want %d): %s\n", __LINE__, #call, rc_, (want), ksana_sage_last_error()); \
    }                                                                                             \
  } while (0)

// Every (pair, query block) of a causal launch belongs to one workgroup, and an XCD never starts a longer block of a pair
// after a shorter one.  `kinds` collects what the grids seen have had: more than one group, an uneven first group, pairs left over,
// none to an XCD itself.
static int causal_numbering_is_wrong(int pairs, int n_qwg, unsigned* kinds) {
  const ksana_sage::CausalGrid c = ksana_sage::causal_grid(pairs, n_qwg);
  if (c.group < 1) return 1;
  *kinds |= (c.own >= 2 * c.group ? 1u : 0) | (c.own % c.group != 0 && c.own > c.group ? 2u : 0) | (c.rest != 0 ? 4u : 0) | (c.own == 0 ? 8u : 0);
  std::vector<char> seen((size_t)pairs * n_qwg, 0);
  std::vector<int> last(8 * (size_t)pairs, n_qwg);  // the block of the pair that the XCD started last
  int n = 0;
  for (int block = 0; block < (pairs * n_qwg + 7) / 8 * 8; ++block) {
    int pair = -1, qwg = -1;
    if (!ksana_sage::causal_place(c, block, n_qwg, &pair, &qwg)) continue;
    if (pair < 0 || pair >= pairs || qwg < 0 || qwg >= n_qwg) return 1;
    char& here = seen[(size_t)pair * n_qwg + qwg];
    int& before = last[(size_t)(block & 7) * pairs + pair];
    if (here++ != 0 || qwg >= before) return 1;
    before = qwg;
    ++n;
  }
  return n != pairs * n_qwg;
}

// Every block of a batch numbered by its counts belongs to one workgroup of a grid of the launcher's size, and an XCD starts the
// entries in the given order, blocks that have only zeros to write after all others.
static int batch_numbering_is_wrong(int B, int heads, int n_qwg, const int* with_rows, const int* order) {
  int starts[ksana_sage::kBatchStarts], at = 0, entries = 0;
  for (int i = 0; i < ksana_sage::kBatchStarts; ++i) {
    starts[i] = i < 2 * B ? at : INT32_MAX;
    if (i < 2 * B) at += ksana_sage::batch_share(heads, i < B ? with_rows[order[i]] : n_qwg - with_rows[order[i - B]]);
    if (i < B) entries |= order[i] << (4 * i);
  }
  starts[0] = entries;
  const int per_xcd = B * ((heads * n_qwg + 7) / 8 + 1);
  if (at > per_xcd) return 1;
  std::vector<char> seen((size_t)B * heads * n_qwg, 0);
  int n = 0;
  for (int xcd = 0; xcd < 8; ++xcd) {
    int before = 0;
    for (int i = 0; i < per_xcd; ++i) {
      const ksana_sage::BatchRun run = ksana_sage::batch_run_of(starts, B, i);
      if (run.b < 0 || run.b >= B) return 1;
      const ksana_sage::BatchPlace p = ksana_sage::batch_place(run, xcd, i, heads, n_qwg, with_rows[run.b]);
      if (p.b < 0) continue;
      if (p.b != run.b || p.h < 0 || p.h >= heads || p.qwg < 0 || p.qwg >= n_qwg) return 1;
      const bool zero = p.qwg >= with_rows[p.b];
      int here = zero ? B : 0;
      while (order[here % B] != p.b) ++here;
      if (zero != run.zeros || here < before || seen[((size_t)p.b * heads + p.h) * n_qwg + p.qwg]++ != 0) return 1;
      before = here;
      ++n;
    }
  }
  return n != B * heads * n_qwg;
}

// Which calls are numbered, and with how many rows a workgroup (without a device: 256 compute units)
static int batch_rows(int B, int heads, int Lq, int Lk, int waves = 0, int causal = 0, bool counts = true) {
  static const int32_t some[1] = {1};
  ksana_sage::AttnParams p{};
  p.B = B, p.Hq = p.Hkv = heads, p.Lq = Lq, p.Lk = Lk, p.nkb = (Lk + 63) / 64, p.causal = causal, p.wg_waves = waves, p.exact_exp2 = 1, p.d_out = 128;
  p.k_lens = counts ? some : nullptr;
  return ksana_sage::batch_rows_wg(p);
}

int main() {
  void* const fake = reinterpret_cast<void*>(0x1000);  // aligned and never dereferenced
  ksana_sage_shape s{1, 2, 2, 64, 64, 128};
  const int64_t st[4] = {64 * 2 * 128, 2 * 128, 128, 1};
  ksana_sage_ws_layout lay;
  EXPECT(ksana_sage_workspace_layout(nullptr, nullptr), KSANA_SAGE_EINVAL);
  EXPECT(ksana_sage_workspace_layout(&s, &lay), 0);
  if (lay.total_bytes == 0 || lay.nkb != 1 || lay.lq_pad != 128) ++g_failed, std::printf("layout of the small shape is off\n");
  ksana_sage_shape big{1, 40, 40, 32760, 32760, 128};
  EXPECT(ksana_sage_workspace_layout(&big, &lay), 0);
  ksana_sage_shape odd_d{1, 2, 2, 64, 64, 96};
  EXPECT(ksana_sage_workspace_layout(&odd_d, &lay), KSANA_SAGE_ENOTSUP);
  ksana_sage_shape gqa{1, 3, 2, 64, 64, 128};
  EXPECT(ksana_sage_workspace_layout(&gqa, &lay), KSANA_SAGE_EINVAL);

  EXPECT(ksana_sage_quant_q(nullptr, KSANA_SAGE_BF16, st, &s, 0.1f, fake, nullptr), KSANA_SAGE_EINVAL);
  EXPECT(ksana_sage_quant_k(fake, 7, st, &s, 1, fake, nullptr), KSANA_SAGE_EINVAL);
  EXPECT(ksana_sage_quant_v(reinterpret_cast<void*>(0x1008), KSANA_SAGE_BF16, st, &s, fake, nullptr), KSANA_SAGE_EINVAL);
  const int64_t bad_d[4] = {64 * 2 * 128, 2 * 128, 128, 2};
  EXPECT(ksana_sage_quant_q(fake, KSANA_SAGE_BF16, bad_d, &s, 0.1f, fake, nullptr), KSANA_SAGE_EINVAL);
  EXPECT(ksana_sage_quant_q(fake, KSANA_SAGE_BF16, nullptr, &s, 0.1f, fake, nullptr), KSANA_SAGE_EINVAL);
  EXPECT(ksana_sage_quant_q(fake, KSANA_SAGE_BF16, st, &s, 0.1f, nullptr, nullptr), KSANA_SAGE_EINVAL);
  EXPECT(ksana_sage_quant_k_static(fake, KSANA_SAGE_BF16, st, &s, 1, nullptr, nullptr), KSANA_SAGE_EINVAL);
  ksana_sage_shape many{1, 65, 65, 64, 65536, 128};
  EXPECT(ksana_sage_quant_k_static(fake, KSANA_SAGE_BF16, st, &many, 1, fake, nullptr), KSANA_SAGE_ENOTSUP);

  // the descriptor of the step before attention, with its host-resident grid sizes
  ksana_sage_prep prep;
  std::memset(&prep, 0, sizeof(prep));
  prep.norm_eps = 1e-6f;
  prep.q_norm_weight = reinterpret_cast<const float*>(0x1004);  // misaligned
  EXPECT(ksana_sage_quant_q_prep(fake, KSANA_SAGE_BF16, st, &s, &prep, 0.1f, fake, nullptr), KSANA_SAGE_EINVAL);
  std::memset(&prep, 0, sizeof(prep));
  prep.rope_freqs = reinterpret_cast<const double*>(0x1000);
  prep.rope_rows = 1024;  // a rotation without grid sizes
  EXPECT(ksana_sage_quant_k_prep(fake, KSANA_SAGE_BF16, st, &s, &prep, 1, fake, nullptr), KSANA_SAGE_EINVAL);
  std::vector<int32_t> grid = {2, 8, 8};  // exactly B * 3 values: reading past them is what the sanitizer would catch
  prep.grid_sizes = grid.data();
  EXPECT(ksana_sage_quant_k_prep(fake, KSANA_SAGE_BF16, st, &s, &prep, 1, fake, nullptr), KSANA_SAGE_EINVAL);  // 128 positions, 64 rows
  grid = {1, 8, 2000};  // an extent beyond the table
  prep.grid_sizes = grid.data();
  EXPECT(ksana_sage_quant_qk_prep(fake, fake, KSANA_SAGE_BF16, st, st, &s, &prep, 0.1f, 1, fake, nullptr), KSANA_SAGE_EINVAL);
  ksana_sage_shape two{2, 2, 2, 64, 64, 128};
  std::vector<int32_t> grid2 = {1, 8, 8, 1, 8, 9};  // the second batch entry is the bad one
  prep.grid_sizes = grid2.data();
  EXPECT(ksana_sage_forward_prep(fake, fake, fake, fake, KSANA_SAGE_BF16, st, st, st, st, &two, &prep, nullptr, 0.1f, 1, 0, 0, fake, nullptr),
         KSANA_SAGE_EINVAL);
  std::memset(&prep, 0, sizeof(prep));
  prep.kind = KSANA_SAGE_PREP_QWEN;
  prep.txt_len = 65;  // beyond the sequence
  prep.q_norm_weight = reinterpret_cast<const float*>(0x1000);
  EXPECT(ksana_sage_quant_q_prep(fake, KSANA_SAGE_BF16, st, &s, &prep, 0.1f, fake, nullptr), KSANA_SAGE_EINVAL);
  prep.kind = 9;
  EXPECT(ksana_sage_quant_q_prep(fake, KSANA_SAGE_BF16, st, &s, &prep, 0.1f, fake, nullptr), KSANA_SAGE_EINVAL);

  // attention entry points
  ksana_sage_shape long_k{1, 2, 2, 64, 131073, 128};
  EXPECT(ksana_sage_attn_fwd(fake, fake, KSANA_SAGE_BF16, st, &long_k, nullptr, 1, 0, nullptr), KSANA_SAGE_ENOTSUP);
  EXPECT(ksana_sage_attn_fwd(fake, fake, KSANA_SAGE_BF16, st, &s, nullptr, 0, 0x20, nullptr), KSANA_SAGE_EINVAL);
  EXPECT(ksana_sage_attn_fwd(fake, fake, KSANA_SAGE_BF16, st, &s, nullptr, 0, KSANA_SAGE_FLAG_TILE_SKIP | KSANA_SAGE_FLAG_PWL_EXP2, nullptr),
         KSANA_SAGE_EINVAL);
  EXPECT(ksana_sage_attn_fwd(fake, fake, KSANA_SAGE_BF16, st, &s, reinterpret_cast<const int32_t*>(0x1002), 0, 0, nullptr), KSANA_SAGE_EINVAL);
  EXPECT(ksana_sage_attn_fwd_masked(fake, fake, KSANA_SAGE_BF16, st, &s, reinterpret_cast<const int8_t*>(fake), nullptr, nullptr, 0, 0, nullptr),
         KSANA_SAGE_EINVAL);
  const int64_t neg[2] = {-1, 0};
  EXPECT(ksana_sage_attn_fwd_masked(fake, fake, KSANA_SAGE_BF16, st, &s, reinterpret_cast<const int8_t*>(fake), neg, nullptr, 0, 0, nullptr),
         KSANA_SAGE_EINVAL);
  EXPECT(ksana_sage_forward(fake, fake, nullptr, fake, KSANA_SAGE_BF16, st, st, st, st, &s, nullptr, 0.1f, 1, 0, 0, fake, nullptr), KSANA_SAGE_EINVAL);
  ksana_sage_call call{s, KSANA_SAGE_BF16, KSANA_SAGE_BF16, 1, 0, 0, 0.1f, {}, {}, {}, {}};
  for (int64_t* to : {call.q_strides, call.k_strides, call.v_strides, call.o_strides}) std::memcpy(to, st, sizeof(st));
  EXPECT(ksana_sage_forward_call(nullptr, fake, fake, fake, fake, fake, nullptr), KSANA_SAGE_EINVAL);
  EXPECT(ksana_sage_forward_call(&call, fake, fake, fake, nullptr, fake, nullptr), KSANA_SAGE_EINVAL);
  EXPECT(ksana_sage_forward_call(&call, fake, fake, fake, fake, nullptr, nullptr), KSANA_SAGE_EINVAL);
  call.flags = 0x4000;
  EXPECT(ksana_sage_forward_call(&call, fake, fake, fake, fake, fake, nullptr), KSANA_SAGE_EINVAL);
  int first = -1, runs = -1;
  EXPECT(ksana_sage_attn_key_split(&s, &first, nullptr), KSANA_SAGE_EINVAL);

  unsigned kinds = 0;
  for (int pairs = 1; pairs <= 130; ++pairs)
    for (int n_qwg : {1, 2, 3, 7, 11, 24, 63, 64, 65, 96, 97, 128, 192, 255, 256, 383, 384, 385, 590, 1024})
      if (causal_numbering_is_wrong(pairs, n_qwg, &kinds)) ++g_failed, std::printf("causal numbering of %d pairs of %d blocks\n", pairs, n_qwg);
  if (kinds != 15) ++g_failed, std::printf("causal numbering: kinds of grids seen 0x%x\n", kinds);

  // the sparse-linear backend's entry points
  uint64_t bytes = 0;
  EXPECT(ksana_sage_sla_workspace_bytes(1, 40, 32760, &bytes), 0);
  EXPECT(ksana_sage_sla_workspace_bytes(0, 40, 32760, &bytes), KSANA_SAGE_EINVAL);
  EXPECT(ksana_sage_sla_linear(fake, fake, nullptr, KSANA_SAGE_BF16, st, st, st, 1, 2, 64, nullptr, nullptr, nullptr, nullptr, fake, st, fake, nullptr),
         KSANA_SAGE_EINVAL);
  EXPECT(ksana_sage_sla_block_map(fake, fake, KSANA_SAGE_BF16, 1, 2, 8, 2000, 3, reinterpret_cast<int8_t*>(fake), nullptr), KSANA_SAGE_ENOTSUP);
  EXPECT(ksana_sage_block_means(fake, KSANA_SAGE_BF16, st, 1, 2, 64, 48, nullptr, fake, nullptr), KSANA_SAGE_ENOTSUP);
  ksana_sage_shape d64{1, 2, 2, 64, 64, 64};
  EXPECT(ksana_sage_quant_qk_pooled(fake, fake, KSANA_SAGE_BF16, st, st, &d64, 0.1f, fake, fake, fake, nullptr), KSANA_SAGE_ENOTSUP);
  EXPECT(ksana_sage_quant_qk_pooled(fake, fake, KSANA_SAGE_BF16, st, st, &s, 0.1f, fake, nullptr, fake, nullptr), KSANA_SAGE_EINVAL);
  EXPECT(ksana_sage_quant_qk_pooled(fake, nullptr, KSANA_SAGE_BF16, st, st, &s, 0.1f, fake, fake, fake, nullptr), KSANA_SAGE_EINVAL);

  // settings and self-checks
  EXPECT(ksana_sage_configure("kx", KSANA_SAGE_KEEP), KSANA_SAGE_EINVAL);
  EXPECT(ksana_sage_configure("kv", 123), 0);
  int k1 = 0, v1 = 0, dem = -1;
  int64_t ticks = 0;
  EXPECT(ksana_sage_one_read_state(&k1, &v1, &ticks, &dem), 0);
  if (!k1 || !v1 || ticks != 123 || dem != 0) ++g_failed, std::printf("settings did not stick\n");
  unsigned seed = 1;
  for (int i = 0; i < 4000; ++i) {
    auto next = [&](int n) { return (int)((seed = seed * 1664525u + 1013904223u) >> 8) % n; };
    const int B = 2 + next(ksana_sage::kBatchEntries - 1), heads = 1 + next(70), n_qwg = 1 + next(40), kind = next(4);
    int with_rows[ksana_sage::kBatchEntries];
    for (int& w : with_rows) w = kind == 0 ? next(n_qwg + 1) : kind == 1 ? n_qwg : kind == 2 ? 0 : next(2) * n_qwg;
    int order[ksana_sage::kBatchEntries];
    for (int e = 0; e < B; ++e) {
      const int to = next(e + 1);
      order[e] = order[to], order[to] = e;
    }
    if (batch_numbering_is_wrong(B, heads, n_qwg, with_rows, order)) ++g_failed, std::printf("batch numbering: %d entries, %d heads, %d blocks\n", B, heads, n_qwg);
  }
  // one round and a block more, four and a half rounds and a block more, entries, options, cut blocks
  EXPECT(batch_rows(2, 16, 2048, 600), 0);
  EXPECT(batch_rows(2, 16, 2049, 600), 128);
  EXPECT(batch_rows(2, 64, 18 * 128, 600), 128);
  EXPECT(batch_rows(2, 64, 18 * 128 + 1, 600), 0);
  EXPECT(batch_rows(8, 24, 1000, 600), 128);
  EXPECT(batch_rows(9, 24, 1000, 600), 0);
  EXPECT(batch_rows(1, 64, 1500, 600), 0);
  EXPECT(batch_rows(8, 24, 1000, 600, 0, 1), 0);
  EXPECT(batch_rows(8, 24, 1000, 600, 0, 0, false), 0);
  EXPECT(batch_rows(8, 24, 1000, 600, 8), 256);
  EXPECT(batch_rows(2, 50, 1250, 2560), 256);
  EXPECT(batch_rows(2, 24, 4352, 4352), 0);
  EXPECT(ksana_sage_selftest(), 0);
  if (ksana_sage_abi_version() != KSANA_SAGE_ABI_VERSION) ++g_failed, std::printf("ABI number differs from the header's\n");
  std::printf("host argument checks: %d failed\n", g_failed);
  return g_failed == 0 ? 0 : 1;
}
