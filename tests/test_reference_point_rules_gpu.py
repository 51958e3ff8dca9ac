"""Where a row's reference points lie: as the emulation has them, by the row's own scores alone, and close enough to its strongest
keys - with more key tiles than the kernel has in flight, and with scores that are neither flat nor peaked."""

import pytest
import torch

from ksanadit_amd import sage_ops
from ksanadit_amd.layout import untile_k, untile_v
from oracle.quant_ref import BLKK
from oracle.sage_emul_ref import sage_emul_from_quant

pytestmark = pytest.mark.gpu

LOG2E = 1.4426950408889634


def _inputs(Lq, Lk, H, octaves, seed):
    """fp16 q, k, v of 128 channels whose scores have a standard deviation of ``octaves`` in the exponent's base 2."""
    g = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn((1, n, H, 128), generator=g) for n in (Lq, Lk, Lk))
    return (q * (octaves / LOG2E)).half(), k.half(), v.half()


def _quantized(q, k, v, device):
    qd, kd, vd = (t.to(device) for t in (q, k, v))
    ws = sage_ops.workspace_for(qd, kd)
    sage_ops.quant_q(qd, ws, q.shape[3] ** -0.5), sage_ops.quant_k(kd, ws, True), sage_ops.quant_v(vd, ws)
    return ws


def _operands(ws, Lq, Lk):
    return (ws.q_i8.cpu()[:, :, :Lq], ws.q_scale.cpu()[:, :, :Lq], untile_k(ws.k_tiles.cpu(), Lk), ws.k_scale.cpu(),
            untile_v(ws.v_tiles.cpu(), Lk).view(torch.float8_e4m3fn), ws.v_scale.cpu())


def _distance(out, want):
    out, want = out.double(), want.double()
    return float((out - want).norm() / want.norm())


@pytest.mark.parametrize("octaves", [1.0, 1.44, 1.8, 2.0, 2.4])
@pytest.mark.parametrize("mode", ["dense", "masked", "causal"])
def test_points_are_where_the_emulation_has_them(hip_device, octaves, mode):
    """Relative, over the whole result (2-norm).  With the same points: fp16's rounding, at most 2^-11 and 2e-4 root mean square, and
    the probabilities that an exponential one ulp off takes across a rounding boundary, 1 in 1e5 of them by one code (6 %),
    another 2e-4: 3e-4 together (0.6e-4 to 1.9e-4 seen).  Points elsewhere, and with them e4m3 roundings, give 1.1e-3 to 1.2e-2."""
    tiles = 41
    Lk = 64 * tiles - 7
    Lq = Lk if mode == "causal" else 512
    print(f"case {mode} octaves={octaves}", flush=True)
    q, k, v = _inputs(Lq, Lk, 1, octaves, int(100 * octaves))
    ws = _quantized(q, k, v, hip_device)
    kw = {"dense": {}, "causal": {"causal": True}, "masked": {"block_mask": torch.ones((-(-Lq // 128), tiles), dtype=torch.int8)}}[mode]
    if mode == "masked":
        kw["block_mask"][::2, 1::5] = 0
    out = sage_ops.attn_fwd(ws, torch.empty((1, Lq, 1, 128), dtype=torch.float16, device=hip_device), **kw,
                            **({"wg_waves": 4} if mode == "dense" else {})).cpu()
    distance = _distance(out, sage_emul_from_quant(*_operands(ws, Lq, Lk), torch.float16, **kw))
    print(f"distance {distance:.6f}", flush=True)
    assert distance <= 5e-4


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("mode", ["dense4", "dense8", "masked", "masked8", "causal", "skip", "pwl"])
def test_a_row_has_the_same_bits_among_other_rows(hip_device, mode, D):
    """Every row but one in 32 replaced, flat scores by spread ones (in causal calls too, rows after it among them): the row's own
    scores decide where its probabilities are rounded."""
    tiles = 41
    Lk = 64 * tiles
    Lq, H = (Lk if mode == "causal" else 512), (130 if mode == "dense8" else 2)  # (260 blocks of 256 rows)
    print(f"case {mode} D={D}", flush=True)
    g = torch.Generator(device=hip_device).manual_seed(D)
    q, k, v = (torch.randn((1, n, H, D), generator=g, device=hip_device) for n in (Lq, Lk, Lk))
    kept = torch.arange(Lq, device=hip_device) % 32 == 5
    kw = {"dense4": {"wg_waves": 4}, "dense8": {"wg_waves": 8}, "causal": {"causal": True}, "skip": {"tile_skip": True, "wg_waves": 4},
          "pwl": {"pwl_exp2": True, "wg_waves": 4}}.get(mode)
    if kw is None:
        kw = {"block_mask": torch.ones((4, tiles), dtype=torch.int8), **({"wg_waves": 8} if mode == "masked8" else {})}
        kw["block_mask"][::2, 1::5] = 0
    outs = []
    for others in (1.0, 3.0):
        ws = _quantized(torch.where(kept[:, None, None], q, others * q).half(), k.half(), v.half(), hip_device)
        outs.append(sage_ops.attn_fwd(ws, torch.empty((1, Lq, H, D), dtype=torch.float16, device=hip_device), **kw))
    if mode == "dense8":
        plan = sage_ops.key_split_plan(ws)
        whole = H if plan is None else plan[0] // 2  # heads whose blocks are not cut into runs of keys
        assert whole >= 128
        outs = [o[:, :, :whole] for o in outs]
    assert torch.equal(outs[0][:, kept], outs[1][:, kept])
    assert not torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("kw", [{}, {"is_causal": True}, {"block_mask": True}], ids=["dense", "causal", "masked"])
@pytest.mark.parametrize("holds", [3.0, float("inf"), float("nan")])
def test_padding_rows_do_not_move_the_points_of_the_others(hip_device, holds, kw):
    """A wave of 10 rows that count and 22 that do not: whatever these hold, also as spread scores, the others' bits stay."""
    B, H, L = 2, 8, 64 * 41
    print(f"case holds={holds} {kw}", flush=True)
    g = torch.Generator(device=hip_device).manual_seed(3)
    q, k, v = (torch.randn((B, L, H, 128), generator=g, device=hip_device).half() for _ in range(3))
    q_lens = [L - 118, 2250]
    kw = dict(kw, q_lens=torch.tensor(q_lens, dtype=torch.int32, device=hip_device))
    if "block_mask" in kw:
        kw["block_mask"] = torch.ones((-(-L // 128), L // 64), dtype=torch.int8, device=hip_device)
    want = sage_ops.sageattn(q, k, v, **kw)
    for b, n in enumerate(q_lens):
        assert n % 32 == 10
        q[b, n:] *= holds
    got = sage_ops.sageattn(q, k, v, **kw)
    for b, n in enumerate(q_lens):
        assert torch.equal(got[b, :n], want[b, :n]) and not got[b, n:].any()


# the error with points that move by more than 2.7 octaves, to the strongest key of the tile that asks for it; with points that move by more
# than 2.86, and first points up to the maximum of four tiles where a wave's scores are flat; the bound lies between
@pytest.mark.parametrize("octaves,tiles,bound", [(1.8, 48, 0.02545),  # 0.025307 / 0.025626
                                                 (2.0, 48, 0.02455),  # 0.024425 / 0.024732
                                                 (2.2, 48, 0.02355),  # 0.023423 / 0.023693
                                                 (2.0, 8, 0.02302),   # 0.022968 / 0.023072
                                                 (2.4, 8, 0.02048)])  # 0.020415 / 0.020535
def test_what_the_rounding_of_probabilities_costs(hip_device, octaves, tiles, bound):
    """Against 64 bits on the same quantized operands, over 2 million values: what is left is the rounding of the
    probabilities."""
    Lq, H, Lk = 1024, 16, BLKK * tiles
    print(f"case octaves={octaves} tiles={tiles}", flush=True)
    ws = _quantized(*_inputs(Lq, Lk, H, octaves, tiles), hip_device)
    out = sage_ops.attn_fwd(ws, torch.empty((1, Lq, H, 128), dtype=torch.float16, device=hip_device), wg_waves=4).cpu()
    q, qs, k, ks, v, vs = (t.double() if t.dtype != torch.float8_e4m3fn else t.float().double() for t in _operands(ws, Lq, Lk))
    num = den = 0.0
    for h in range(H):
        s = (q[0, h] @ k[0, h].t()) * qs[0, h][:, None] * ks[0, h].repeat_interleave(BLKK)[None, :]
        want = torch.softmax(s * (1.0 / LOG2E), dim=1) @ v[0, h] * vs[0, h]
        num, den = num + float((out[0, :, h].double() - want).square().sum()), den + float(want.square().sum())
    error = (num / den) ** 0.5
    print(f"error {error:.6f}", flush=True)
    assert error <= bound
