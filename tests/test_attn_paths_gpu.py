"""The attention kernel's own branches at the sizes where they can go wrong, against the tile-by-tile emulation fed with
the operands the GPU quantized.

Tolerance of every comparison: kernel and emulation do the same fp32 operations up to summation order and up to an
exponential that may differ in its last place, so a probability lands on another e4m3 code only within an ulp of a
rounding boundary (6 % of one probability); everything else is the final rounding to the output type, 2^-9 relative."""

import pytest
import torch

from ksanadit_amd import sage_ops
from ksanadit_amd.layout import untile_k, untile_v
from oracle.sage_emul_ref import sage_emul_from_quant

pytestmark = pytest.mark.gpu


def _emul(ws, Lq, Lk, dtype, **kw):
    return sage_emul_from_quant(
        ws.q_i8.cpu()[:, :, :Lq], ws.q_scale.cpu()[:, :, :Lq], untile_k(ws.k_tiles.cpu(), Lk), ws.k_scale.cpu(),
        untile_v(ws.v_tiles.cpu(), Lk).view(torch.float8_e4m3fn), ws.v_scale.cpu(), dtype, **kw)


def _close(out, want):
    out, want = out.float(), want.float()
    scale = max(float(want.abs().max()), 1e-3)
    diff = (out - want).abs()
    assert torch.isfinite(out).all()
    assert float(diff.max()) <= 2e-2 * scale
    assert float((diff > 5e-3 * scale).float().mean()) <= 1e-3


@pytest.mark.parametrize("waves", [4, 8])
@pytest.mark.parametrize("Lk", [64, 128, 192, 448, 470])
@pytest.mark.parametrize("lift", [0.5, 6.0], ids=["below_the_limit", "above_the_limit"])
def test_reference_points_move_at_any_tile(hip_device, waves, Lk, lift):
    """Each key tile in turn outdoes every tile before it, for some query rows only: the reference point of those rows
    moves at the first, a middle, the last full and the ragged tile (or stays, where the step is small)."""
    Lq, H = 160, 1
    print(f"case waves={waves} Lk={Lk} lift={lift}", flush=True)
    g = torch.Generator().manual_seed(Lk)
    q, k, v = (torch.randn((1, n, H, 128), generator=g) for n in (Lq, Lk, Lk))
    direction = torch.randn(128, generator=g)
    direction /= direction.norm()
    # key tile t leans towards the direction by t steps, query row i towards it or away: scores rise (or fall) tile by tile
    step = torch.arange(Lk) // 64
    k = k * 0.2 + (step[None, :, None, None] * lift) * direction
    q = q * 0.2 + (torch.where(torch.arange(Lq) % 3 == 0, -4.0, 4.0)[None, :, None, None]) * direction
    q, k, v = (t.to(torch.bfloat16) for t in (q, k, v))
    qd, kd, vd = (t.to(hip_device) for t in (q, k, v))
    ws = sage_ops.workspace_for(qd, kd)
    sage_ops.quant_q(qd, ws, 128**-0.5), sage_ops.quant_k(kd, ws, True), sage_ops.quant_v(vd, ws)
    out = sage_ops.attn_fwd(ws, torch.empty_like(qd), wg_waves=waves).cpu()
    _close(out, _emul(ws, Lq, Lk, q.dtype))


@pytest.mark.parametrize("waves", [4, 8])
@pytest.mark.parametrize("tiles,tail", [(1, 0), (3, 5), (4, 0), (7, 0), (8, 0), (8, 1), (9, 63), (15, 2), (16, 0), (17, 0), (21, 7)])
@pytest.mark.parametrize("mode", ["dense", "causal", "masked"])
def test_key_loop_around_its_unrolled_groups(hip_device, waves, tiles, tail, mode):
    """Numbers of key tiles around the unrolled loop's length (8, or 4), with and without a ragged last tile, with waves
    that have no query rows (they only take part in the copies and barriers) and a last wave of a few rows."""
    Lq, Lk, H = 300, 64 * tiles + tail, 1
    print(f"case waves={waves} Lk={Lk} {mode}", flush=True)
    g = torch.Generator().manual_seed(Lk)
    q, k, v = (torch.randn((1, n, H, 128), generator=g).to(torch.bfloat16) for n in (Lq, Lk, Lk))
    qd, kd, vd = (t.to(hip_device) for t in (q, k, v))
    ws = sage_ops.workspace_for(qd, kd)
    sage_ops.quant_q(qd, ws, 128**-0.5), sage_ops.quant_k(kd, ws, True), sage_ops.quant_v(vd, ws)
    kw = {}
    if mode == "causal":
        kw["causal"] = True
    if mode == "masked":
        kw["block_mask"] = (torch.rand((1, H, 3, -(-Lk // 64)), generator=g) < 0.7).to(torch.int8)
    out = sage_ops.attn_fwd(ws, torch.empty_like(qd), wg_waves=waves, **kw).cpu()
    split = sage_ops.key_split_plan(ws) if mode == "dense" and waves == 8 else None
    _close(out, _emul(ws, Lq, Lk, q.dtype, key_split=split, **kw))


@pytest.mark.parametrize("Lk", [64 * 33, 64 * 40 + 1])
def test_whole_and_cut_query_blocks_in_one_grid(hip_device, Lk):
    """65 heads of 4 query blocks: one full round of whole blocks and 4 blocks cut into runs of keys.  The last head holds
    the cut ones (ragged rows in the last), the head before it whole ones."""
    Lq, H, at = 1000, 65, 63
    print(f"case Lk={Lk}", flush=True)
    g = torch.Generator().manual_seed(Lk)
    q, k, v = (torch.randn((1, n, H, 128), generator=g).to(torch.bfloat16) for n in (Lq, Lk, Lk))
    qd, kd, vd = (t.to(hip_device) for t in (q, k, v))
    ws = sage_ops.workspace_for(qd, kd)
    plan = sage_ops.key_split_plan(ws)
    if torch.cuda.get_device_properties(hip_device).multi_processor_count == 256:
        assert plan is not None and plan[0] == 256 and plan[1] >= 2, plan
    out = sage_ops.sageattn(qd, kd, vd, workspace=ws)[:, :, at:].cpu()
    heads = slice(at, H)
    split = None if plan is None else (max(plan[0] - 4 * at, 0), plan[1])
    want = sage_emul_from_quant(
        ws.q_i8.cpu()[:, heads, :Lq], ws.q_scale.cpu()[:, heads, :Lq], untile_k(ws.k_tiles.cpu()[:, heads], Lk),
        ws.k_scale.cpu()[:, heads], untile_v(ws.v_tiles.cpu()[:, heads], Lk).view(torch.float8_e4m3fn),
        ws.v_scale.cpu()[:, heads], q.dtype, key_split=split)
    _close(out, want)


@pytest.mark.parametrize("B,H", [(1, 1), (1, 3), (1, 8), (3, 5), (1, 17), (2, 24)])
@pytest.mark.parametrize("L", [100, 128, 640, 1300])
def test_causal_blocks_are_shared_out_over_the_chip(hip_device, B, H, L):
    """Every (batch, head, query block) is computed once, whether its pair belongs to one XCD or to all of them; one block
    ahead of the diagonal, on it, and several.  An XCD's own pairs are one group here."""
    print(f"case B={B} H={H} L={L}", flush=True)
    g = torch.Generator().manual_seed(100 * L + 10 * B + H)
    q, k, v = (torch.randn((B, L, H, 128), generator=g).to(torch.bfloat16) for _ in range(3))
    qd, kd, vd = (t.to(hip_device) for t in (q, k, v))
    ws = sage_ops.workspace_for(qd, kd)
    sage_ops.quant_q(qd, ws, 128**-0.5), sage_ops.quant_k(kd, ws, True), sage_ops.quant_v(vd, ws)
    out = sage_ops.attn_fwd(ws, torch.full_like(qd, float("nan")), causal=True).cpu()
    _close(out, _emul(ws, L, L, q.dtype, causal=True))


def test_causal_pairs_are_walked_in_groups(hip_device):
    """192 query blocks a head: an XCD walks its five pairs in groups of three and two, and three pairs are left over.  The same
    bits as eight heads at a time, one to an XCD."""
    L, H = 24500, 43
    print(f"case H={H} L={L}", flush=True)
    g = torch.Generator(device=hip_device).manual_seed(L)
    q, k, v = (torch.randn((1, L, H, 128), generator=g, device=hip_device).to(torch.bfloat16) for _ in range(3))
    out = sage_ops.sageattn(q, k, v, is_causal=True)
    for h in range(0, H, 8):
        part = sage_ops.sageattn(q[:, :, h : h + 8], k[:, :, h : h + 8], v[:, :, h : h + 8], is_causal=True)
        assert torch.equal(out[:, :, h : h + 8], part), h


@pytest.mark.parametrize("waves", [4, 8])
@pytest.mark.parametrize("Lk", [64 * 8, 64 * 9, 64 * 17 + 3])
def test_repeated_calls_give_the_same_bits(hip_device, waves, Lk):
    """The waves of a workgroup share the tile ring and meet seldom: whatever their pace, no tile is replaced before all have
    read it."""
    print(f"case waves={waves} Lk={Lk}", flush=True)
    g = torch.Generator().manual_seed(Lk)
    q, k, v = (torch.randn((1, n, 16, 128), generator=g).to(torch.float16).to(hip_device) for n in (512, Lk, Lk))
    ws = sage_ops.workspace_for(q, k)
    sage_ops.quant_q(q, ws, 128**-0.5), sage_ops.quant_k(k, ws, True), sage_ops.quant_v(v, ws)
    first = sage_ops.attn_fwd(ws, torch.empty_like(q), wg_waves=waves)
    for _ in range(40):
        assert torch.equal(sage_ops.attn_fwd(ws, torch.empty_like(q), wg_waves=waves), first)


@pytest.mark.parametrize("waves", [4, 8])
@pytest.mark.parametrize("Lk", [30, 64, 200, 64 * 12])
@pytest.mark.parametrize("mode", ["exact", "pwl", "skip", "causal"])
def test_query_rows_that_are_not_finite_stay_on_their_own(hip_device, waves, Lk, mode):
    """Rows of q with an infinity in them (padding rows may hold anything) give NaN and leave every other row's bits alone."""
    print(f"case waves={waves} Lk={Lk} {mode}", flush=True)
    g = torch.Generator().manual_seed(Lk)
    q, k, v = (torch.randn((1, n, 1, 128), generator=g).to(torch.bfloat16) for n in (100, Lk, Lk))
    bad = torch.zeros(100, dtype=torch.bool)
    bad[[0, 5, 37, 40, 99]] = True
    outs = []
    for value in (0.0, float("inf")):
        q[0, bad, 0, 9] = value
        qd, kd, vd = (t.to(hip_device) for t in (q, k, v))
        ws = sage_ops.workspace_for(qd, kd)
        sage_ops.quant_q(qd, ws, 128**-0.5), sage_ops.quant_k(kd, ws, True), sage_ops.quant_v(vd, ws)
        outs.append(sage_ops.attn_fwd(ws, torch.empty_like(qd), wg_waves=waves, pwl_exp2=mode == "pwl", tile_skip=mode == "skip",
                                      causal=mode == "causal").cpu()[0])
    assert torch.isnan(outs[1][bad]).all()
    assert torch.isfinite(outs[1][~bad]).all() and torch.equal(outs[0][~bad], outs[1][~bad])


@pytest.mark.parametrize("waves", [4, 8])
@pytest.mark.parametrize("whole", range(15))
@pytest.mark.parametrize("rest", [1, 37, 63])
def test_the_ragged_tile_at_any_place_of_the_ring(hip_device, waves, whole, rest):
    """The last, ragged key tile is a step of the loop like the others: at every place of the ring and of a group, with few
    and with all but one of its keys, and the largest score of a row among the ones that exist or just short of them."""
    Lq, H, Lk = 130, 1, 64 * whole + rest
    print(f"case waves={waves} Lk={Lk}", flush=True)
    g = torch.Generator().manual_seed(Lk)
    q, k, v = (torch.randn((1, n, H, 128), generator=g).to(torch.bfloat16) for n in (Lq, Lk, Lk))
    k[:, -1] = 3 * q[:, 5]  # row 5 sees little but the very last key
    qd, kd, vd = (t.to(hip_device) for t in (q, k, v))
    ws = sage_ops.workspace_for(qd, kd)
    sage_ops.quant_q(qd, ws, 128**-0.5), sage_ops.quant_k(kd, ws, True), sage_ops.quant_v(vd, ws)
    out = sage_ops.attn_fwd(ws, torch.empty_like(qd), wg_waves=waves).cpu()
    _close(out, _emul(ws, Lq, Lk, q.dtype))
    short = torch.tensor([max(Lk - 1, 1)], dtype=torch.int32, device=hip_device)  # the count a batch entry may have of its own
    out = sage_ops.attn_fwd(ws, torch.empty_like(qd), wg_waves=waves, k_lens=short).cpu()
    _close(out, _emul(ws, Lq, Lk, q.dtype, k_lens=short.cpu()))


@pytest.mark.parametrize("rows", [1, 31, 40, 96])
@pytest.mark.parametrize("Lk", [77, 128, 300, 448])
def test_a_workgroup_with_waves_that_have_no_rows(hip_device, rows, Lk):
    """The last workgroup of a head has one, two or three waves with rows; the others only move tiles and run ahead as far
    as the barriers let them.  With many heads, in a kernel's first launch after another one: the same bits as in 8 waves."""
    B, H, Lq = 2, 64, 4096 + rows
    print(f"case rows={rows} Lk={Lk}", flush=True)
    g = torch.Generator(device=hip_device).manual_seed(Lk)
    q, k, v = (torch.randn((B, n, h, 128), generator=g, device=hip_device).half() for n, h in ((Lq, H), (Lk, 16), (Lk, 16)))
    ws = sage_ops.workspace_for(q, k)
    for _ in range(3):
        sage_ops.quant_q(q, ws, 128**-0.5), sage_ops.quant_k(k, ws, True), sage_ops.quant_v(v, ws)
        four = sage_ops.attn_fwd(ws, torch.empty_like(q), wg_waves=4)
        eight = sage_ops.attn_fwd(ws, torch.empty_like(q), wg_waves=8)
        assert torch.equal(four, eight)


@pytest.mark.parametrize("rows,Lk,D,dtype", [(1, 1025, 128, torch.bfloat16), (24, 1560, 128, torch.float16), (32, 64 * 20, 128, torch.bfloat16),
                                             (17, 1100, 64, torch.float16), (32, 64 * 17, 64, torch.bfloat16), (9, 2049, 128, torch.bfloat16),
                                             (33, 1025, 128, torch.float16), (57, 64 * 18, 128, torch.bfloat16), (64, 1300, 64, torch.bfloat16)])
@pytest.mark.parametrize("whole_call", [False, True])
def test_a_last_block_whose_waves_share_the_keys(hip_device, rows, Lk, D, dtype, whole_call):
    """A last block of up to 32 or 64 rows: its waves take a quarter or half of the key tiles each, like key runs; the blocks
    before it are whole.  Numbers of tiles that divide and do not, ragged last tiles, the first tile of a run the ragged one."""
    H, Lq = 60, 128 * 2 + rows  # 120 blocks of 256 rows: the plan takes 4-wave workgroups
    print(f"case rows={rows} Lk={Lk} D={D} {dtype}", flush=True)
    g = torch.Generator().manual_seed(Lk)
    q, k, v = (torch.randn((1, n, H, D), generator=g).to(dtype) for n in (Lq, Lk, Lk))
    q[0, -1, 1] = float("inf")
    qd, kd, vd = (t.to(hip_device) for t in (q, k, v))
    ws = sage_ops.workspace_for(qd, kd)
    assert sage_ops.key_split_plan(ws) is None
    sage_ops.quant_q(qd, ws, D**-0.5), sage_ops.quant_k(kd, ws, True), sage_ops.quant_v(vd, ws)
    out = (sage_ops.sageattn(qd, kd, vd) if whole_call else sage_ops.attn_fwd(ws, torch.empty_like(qd))).cpu()
    four = sage_ops.attn_fwd(ws, torch.empty_like(qd), wg_waves=4).cpu()
    assert torch.equal(out[:, :-rows], four[:, :-rows])
    assert torch.equal(out.isnan(), four.isnan()) and out[0, -1, 1].isnan().any()
    heads, last = slice(2, 4), slice(Lq - rows, Lq)
    magic = {} if D == 128 else {"magic": 25165824.0}
    want = sage_emul_from_quant(
        ws.q_i8.cpu()[:, heads, last], ws.q_scale.cpu()[:, heads, last], untile_k(ws.k_tiles.cpu()[:, heads], Lk), ws.k_scale.cpu()[:, heads],
        untile_v(ws.v_tiles.cpu()[:, heads], Lk).view(torch.float8_e4m3fn), ws.v_scale.cpu()[:, heads], dtype, key_split=(0, 4 if rows <= 32 else 2), **magic)
    _close(out[:, last, heads], want[..., :D])


@pytest.mark.parametrize("k_len", [1100, 900])
@pytest.mark.parametrize("rows", [57, 20])
def test_a_shared_last_block_in_batches_with_lengths(hip_device, k_len, rows):
    """Entries that end before, inside and with a last block whose waves share the keys (1100 of them; not 900): rows that
    count have the bits they have without counts of rows, the others are zeros."""
    B, H, Lq, Lk = 5, 16, 256 + rows, 1100
    g = torch.Generator(device=hip_device).manual_seed(k_len)
    q, k, v = (torch.randn((B, n, H, 128), generator=g, device=hip_device).half() for n in (Lq, Lk, Lk))
    k_lens = torch.tensor([Lk, k_len, k_len, k_len, Lk], dtype=torch.int32, device=hip_device)
    q_lens = [Lq, 257, 256 + rows // 2, 192, 0]
    q[4, :] = float("nan")
    for call in (lambda **kw: sage_ops.sageattn(q, k, v, k_lens=k_lens, **kw),
                 lambda **kw: sage_ops.attn_fwd(ws, torch.empty_like(q).fill_(float("nan")), k_lens=k_lens, **kw)):
        ws = sage_ops.workspace_for(q, k)
        sage_ops.quant_q(q, ws, 128**-0.5), sage_ops.quant_k(k, ws, True), sage_ops.quant_v(v, ws)
        out, full = call(q_lens=torch.tensor(q_lens, dtype=torch.int32, device=hip_device)), call()
        for b, n in enumerate(q_lens):
            assert torch.equal(out[b, :n], full[b, :n]) and not out[b, n:].isnan().any() and not out[b, n:].any(), b


@pytest.mark.parametrize("B,H,Lq,Lk", [(3, 40, 700, 900), (5, 16, 1000, 300), (64, 2, 700, 130), (65, 2, 700, 130), (2, 40, 2000, 700)])
@pytest.mark.parametrize("wg_waves", [4, 8])
def test_batches_with_counts(hip_device, B, H, Lq, Lk, wg_waves):
    """Counts in any order, equal, none, one, all, out of range against the same operands walked through a mask of ones: grids
    numbered by the counts and (64 and 65 entries, three rounds of 8 waves and more) entry after entry."""
    print(f"case B={B} H={H} Lq={Lq} Lk={Lk} waves={wg_waves}", flush=True)
    g = torch.Generator().manual_seed(B * Lq + Lk)
    q, k, v = (torch.randn((B, n, H, 128), generator=g).to(torch.bfloat16).to(hip_device) for n in (Lq, Lk, Lk))
    ws = sage_ops.workspace_for(q, k)
    sage_ops.sageattn(q, k, v, workspace=ws)
    ones = torch.ones((-(-Lq // 128), -(-Lk // 64)), dtype=torch.int8, device=hip_device)
    choice = [0, 1, 63, 64, Lk // 2, Lk - 1, Lk, Lk + 100, -5]
    lens = [torch.randint(0, n + 1, (B,), generator=g) for n in (Lq, Lk)]
    some = torch.tensor([choice[i % len(choice)] for i in range(B)])
    for q_lens, k_lens in ((lens[0], lens[1]), (lens[0].flip(0), some), (None, lens[1].sort()[0]), (lens[0], None), (torch.full((B,), Lq), torch.full((B,), Lk)),
                           (torch.zeros(B, dtype=torch.int64), lens[1])):
        got, want = torch.full_like(q, 7.0), torch.full_like(q, 9.0)
        sage_ops.attn_fwd(ws, got, q_lens=q_lens, k_lens=k_lens, wg_waves=wg_waves)
        sage_ops.attn_fwd(ws, want, q_lens=q_lens, k_lens=k_lens, wg_waves=4, block_mask=ones)
        assert torch.equal(got, want)
        if q_lens is not None:
            for b in range(B):
                assert (got[b, int(q_lens[b]) :] == 0).all()


@pytest.mark.parametrize("B,H,Lq,Lk,D", [(2, 32, 1062, 1062, 128), (2, 30, 1034, 300, 64), (4, 64, 541, 2302, 128), (4, 64, 624, 1500, 64), (3, 11, 1932, 700, 128)])
def test_short_last_blocks_that_start_last(hip_device, B, H, Lq, Lk, D):
    """Grids that take a round less without the heads' short last blocks, which are numbered behind all others, in 4 and 8 waves,
    against the same call with counts that leave nothing out, whose blocks are numbered by these or in the order of their index."""
    print(f"case B={B} H={H} Lq={Lq} Lk={Lk} D={D}", flush=True)
    g = torch.Generator(device=hip_device).manual_seed(Lq)
    q, k, v = (torch.randn((B, n, H, D), generator=g, device=hip_device).half() for n in (Lq, Lk, Lk))
    want = sage_ops.sageattn(q, k, v, k_lens=torch.full((B,), Lk))
    del_me = torch.full_like(q, float("nan"))  # (memory that the next result may lie in)
    del del_me
    assert torch.equal(sage_ops.sageattn(q, k, v), want)


# Grids of 1.3 to 4.5 rounds.  The numbers come from the quantizers' first stage, their launch for at most 256 keys or the one that
# reads K and V once.
NUMBERED = [
    (3, 24, 8, 3001, 1100, 128, torch.float16),  # 57 rows in the last block, whose waves share the keys of entries with more than 1024
    (4, 24, 24, 1300, 1300, 128, torch.bfloat16),  # 20 rows
    (2, 24, 24, 1500, 300, 64, torch.float16),
    (8, 24, 24, 1000, 600, 128, torch.bfloat16),  # the most entries
    (6, 16, 16, 1500, 300, 128, torch.bfloat16),
    (2, 12, 12, 6946, 138, 128, torch.float16),  # K and V in one launch
    (3, 40, 40, 1500, 700, 64, torch.bfloat16),
    (2, 50, 50, 1250, 2560, 128, torch.bfloat16),  # workgroups of 8 waves
    (2, 50, 10, 1250, 2560, 64, torch.float16),
    (2, 16, 16, 3500, 16500, 128, torch.bfloat16),  # K and V read once
    (3, 7, 7, 3200, 600, 128, torch.bfloat16),  # heads that eight does not divide
]


def _counts(B, Lq, Lk):
    g = torch.Generator().manual_seed(B * Lq + Lk)
    rand = [torch.randint(0, n + 1, (B,), generator=g) for n in (Lq, Lk)]
    fall = [torch.tensor([n - n * 55 * b // (100 * max(B - 1, 1)) for b in range(B)]) for n in (Lq, Lk)]
    odd = torch.tensor([(0, 1, Lq - 1, Lq + 100, -5, 128, 129, Lq)[(b + 2) % 8] for b in range(B)])
    few = torch.tensor([(0, Lk, 1, Lk + 1, -1, 64, 65, Lk)[b % 8] for b in range(B)])
    yield from ((fall[0], fall[1]), (fall[0].flip(0), fall[1].flip(0)), (rand[0], rand[1]), (odd, few), (torch.full((B,), Lq), torch.full((B,), Lk)),
                (torch.full((B,), Lq // 2), torch.full((B,), Lk // 2)), (rand[0], None), (None, few), (torch.zeros(B, dtype=torch.int64), None))


def _by_index(q, k, v, q_lens, k_lens, **kw):
    """The same call with empty entries up to nine, whose blocks are not numbered by the counts; none of NUMBERED is cut with these,
    and those whose last blocks share their keys stay in workgroups of 4 waves."""
    B = q.shape[0]
    q, k, v = (torch.cat([x, x.new_zeros((9 - B, *x.shape[1:]))]) for x in (q, k, v))
    assert sage_ops.key_split_plan(sage_ops.workspace_for(q, k)) is None
    more = lambda n: None if n is None else torch.cat([n, n.new_zeros(9 - B)])  # noqa: E731
    return sage_ops.sageattn(q, k, v, q_lens=more(q_lens), k_lens=more(k_lens), **kw)[:B]


@pytest.mark.parametrize("B,H,Hkv,Lq,Lk,D,dtype", NUMBERED)
def test_batches_numbered_by_their_counts(hip_device, B, H, Hkv, Lq, Lk, D, dtype):
    """Calls whose blocks are numbered by the entries' counts - in one piece, on a kept workspace, in stages on its operands, with V
    smoothed - against the same calls numbered entry after entry."""
    print(f"case B={B} H={H}/{Hkv} Lq={Lq} Lk={Lk} D={D} {dtype}", flush=True)
    g = torch.Generator(device=hip_device).manual_seed(Lq)
    q, k, v = (torch.randn((B, n, h, D), generator=g, device=hip_device).to(dtype) for n, h in ((Lq, H), (Lk, Hkv), (Lk, Hkv)))
    ws = sage_ops.workspace_for(q, k)
    for i, (q_lens, k_lens) in enumerate(_counts(B, Lq, Lk)):
        kw = {"q_lens": q_lens, "k_lens": k_lens}
        want = _by_index(q, k, v, **kw)
        calls = [lambda: sage_ops.sageattn(q, k, v, **kw)]
        if i < 4:
            calls += [lambda: sage_ops.sageattn(q, k, v, workspace=ws, **kw), lambda: sage_ops.attn_fwd(ws, torch.empty_like(q), **kw)]
        if i in (2, 3):
            calls += [lambda: sage_ops.sageattn(q, k, v, smooth_v=True, **kw)]
        for c, call in enumerate(calls):
            if c == 3:
                want = _by_index(q, k, v, smooth_v=True, **kw)
            del_me = torch.full_like(q, float("nan"))  # (memory that the next result may lie in)
            del del_me
            got = call()
            assert torch.equal(got, want), (kw, c)
            for b in range(B if q_lens is not None else 0):
                assert not got[b, max(0, int(q_lens[b])) :].any(), (kw, b)


@pytest.mark.parametrize("B,H,Lq,Lk,rows", [(3, 24, 3001, 1100, 128), (2, 12, 6946, 138, 128), (2, 50, 1250, 2560, 256), (2, 16, 3500, 16500, 256)])
@pytest.mark.parametrize("smooth_v", [False, True])
def test_the_quantizers_number_every_whole_call(hip_device, B, H, Lq, Lk, rows, smooth_v):
    """A kept workspace and smoothed V too: the numbers that the attention kernel has read are those that the counts make."""
    print(f"case B={B} H={H} Lq={Lq} Lk={Lk} smooth_v={smooth_v}", flush=True)
    g = torch.Generator(device=hip_device).manual_seed(Lq)
    q, k, v = (torch.randn((B, n, H, 128), generator=g, device=hip_device).half() for n in (Lq, Lk, Lk))
    ws = sage_ops.workspace_for(q, k)
    blocks = -(-Lq // rows)
    for q_lens, k_lens in _counts(B, Lq, Lk):
        sage_ops.sageattn(q, k, v, workspace=ws, q_lens=q_lens, k_lens=k_lens, smooth_v=smooth_v)
        ql, kl = ([min(max(int(x), 0), n) for x in (lens if lens is not None else [n] * B)] for lens, n in ((q_lens, Lq), (k_lens, Lk)))
        order = sorted(range(B), key=lambda b: -kl[b])
        some = [-(-ql[b] // rows) if kl[b] else 0 for b in order]
        starts = [0]
        for n in some + [blocks - n for n in some]:
            starts.append(starts[-1] + (H * n + 7) // 8)
        want = [sum(b << (4 * i) for i, b in enumerate(order)), *starts[1 : 2 * B]] + [2**31 - 1] * (16 - 2 * B)
        assert ws.blob[ws.layout.split_ml :][:64].view(torch.int32).tolist() == want, (q_lens, k_lens)


@pytest.mark.parametrize("H,Lq,Lk,step", [(16, 3500, 16500, False), (24, 1500, 1500, True)])
def test_batches_numbered_in_the_attention_kernel(hip_device, quant_settings, H, Lq, Lk, step):
    """.. where no launch of the quantizers can take the numbering along: K and V in passes of their own, or a step folded in."""
    print(f"case H={H} Lq={Lq} Lk={Lk} step={step}", flush=True)
    B = 2
    if not step:
        quant_settings(one_read="")
    g = torch.Generator(device=hip_device).manual_seed(3)
    q, k, v = (torch.randn((B, n, H, 128), generator=g, device=hip_device).to(torch.bfloat16) for n in (Lq, Lk, Lk))
    w = torch.rand((4, 128), generator=g, device=hip_device).to(torch.bfloat16) + 0.5
    prep = sage_ops.QwenPrep(100, *w, 1e-6) if step else None
    for q_lens, k_lens in list(_counts(B, Lq, Lk))[:4]:
        kw = {"q_lens": q_lens, "k_lens": k_lens, "prep": prep}
        want = _by_index(q, k, v, **kw)
        assert torch.equal(sage_ops.sageattn(q, k, v, **kw), want), kw


def test_numbered_batches_replayed_with_other_counts(hip_device):
    """A captured call numbers its blocks anew in every replay, by the counts that are there then."""
    B, H, L = 4, 24, 1300
    g = torch.Generator(device=hip_device).manual_seed(5)
    q, k, v = (torch.randn((B, L, H, 128), generator=g, device=hip_device).half() for _ in "qkv")
    q_lens, k_lens = (torch.full((B,), L, dtype=torch.int32, device=hip_device) for _ in "qk")
    call = lambda: sage_ops.sageattn(q, k, v, q_lens=q_lens, k_lens=k_lens)  # noqa: E731
    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    for i, (ql, kl) in enumerate(_counts(B, L, L)):
        for to, n in ((q_lens, ql), (k_lens, kl)):
            to.copy_(torch.full((B,), L, dtype=torch.int32) if n is None else n.to(torch.int32))
        out.fill_(float("nan"))
        graph.replay()
        want = call()
        torch.cuda.synchronize()
        assert torch.equal(out, want), i
