"""Reference points of rows with many key tiles: set by the first tile and moved by later ones, in every part of the key loop.

Tolerance: that of test_attn_paths_gpu.py, for the reason given there."""

import pytest
import torch

from ksanadit_amd import sage_ops
from ksanadit_amd.layout import untile_k, untile_v
from oracle.sage_emul_ref import sage_emul_from_quant

pytestmark = pytest.mark.gpu


def _inputs(Lq, Lk, D, lifted, seed):
    """Flat scores; key tile ``lifted[i]`` stands 5 to 9 octaves above them for the query rows r with r % len == i."""
    g = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn((1, n, 1, D), generator=g) for n in (Lq, Lk, Lk))
    dirs = torch.linalg.qr(torch.randn(D, D, generator=g))[0]
    for i, tile in enumerate(lifted):
        rows = torch.arange(Lq) % len(lifted) == i
        q[0, rows, 0] += 4.0 * dirs[i]
        k[0, 64 * tile : 64 * tile + 64 : 7, 0] += (12.0 if D == 128 else 8.5) * dirs[i]
    return q, k, v


def _quantized(q, k, v, device):
    qd, kd, vd = (t.to(device) for t in (q, k, v))
    ws = sage_ops.workspace_for(qd, kd)
    sage_ops.quant_q(qd, ws, q.shape[3] ** -0.5), sage_ops.quant_k(kd, ws, True), sage_ops.quant_v(vd, ws)
    return ws


# tiles, keys in a ragged last one, lifted tiles: none; the first ones; at the ends of unrolled rounds, in the single steps, the last
@pytest.mark.parametrize("tiles,tail,lifted", [(33, 0, []), (32, 0, [9, 31]), (33, 0, [4, 32]), (40, 0, [7, 8, 39]), (41, 0, [38, 39, 40]),
                                               (41, 9, [5, 40]), (47, 1, [15, 16, 45, 46]), (48, 0, [1, 2, 3, 20]), (36, 63, [0, 3, 35])])
@pytest.mark.parametrize("mode", ["dense4", "dense8", "dense8_whole", "causal", "masked"])
@pytest.mark.parametrize("D,dtype", [(128, torch.bfloat16), (64, torch.float16)])
def test_points_of_long_rows(hip_device, tiles, tail, lifted, mode, D, dtype):
    Lk = 64 * (tiles - 1) + (tail or 64)
    Lq = 140 if mode != "causal" else Lk
    print(f"case {mode} tiles={tiles} tail={tail} lifted={lifted} D={D}", flush=True)
    H = 256 if mode == "dense8_whole" else 1  # (a round of 8-wave workgroups: nobody's keys are cut; one alone walks its keys in runs)
    q, k, v = (t.to(dtype).expand(1, -1, H, -1) for t in _inputs(Lq, Lk, D, lifted, tiles + tail))
    ws = _quantized(q, k, v, hip_device)
    kw, emul = {}, {"magic": 25165824.0} if D == 64 else {}
    if mode == "masked":
        mask = torch.ones((-(-Lq // 128), tiles), dtype=torch.int8)
        mask[0, 1::9] = 0
        kw = {"block_mask": mask}
        emul["block_mask"] = mask
    elif mode == "causal":
        kw = {"causal": True}
        emul["causal"] = True
    else:
        kw = {"wg_waves": int(mode[5])}
    out = sage_ops.attn_fwd(ws, torch.empty((1, Lq, H, D), dtype=dtype, device=hip_device), **kw)
    assert all(torch.equal(out[:, :, 0], out[:, :, h]) for h in range(1, H))
    out = out[:, :, :1].cpu().float()
    plan = sage_ops.key_split_plan(ws)
    if mode.startswith("dense8"):
        assert (plan is None) == (H > 1)
        if plan is not None:
            emul["key_split"] = plan
    want = sage_emul_from_quant(ws.q_i8[:, :1, :Lq].cpu(), ws.q_scale[:, :1, :Lq].cpu(), untile_k(ws.k_tiles[:, :1].cpu(), Lk), ws.k_scale[:, :1].cpu(),
                                untile_v(ws.v_tiles[:, :1].cpu(), Lk).view(torch.float8_e4m3fn), ws.v_scale[:, :1].cpu(), dtype, **emul)
    want = want[..., :D].float()
    scale, diff = float(want.abs().max()), (out - want).abs()
    assert torch.isfinite(out).all()
    assert float(diff.max()) <= 2e-2 * scale
    assert float((diff > 5e-3 * scale).float().mean()) <= 1e-3


@pytest.mark.parametrize("bad_tile", [0, 2, 6, 20, 37, 39, 40])
@pytest.mark.parametrize("mode", ["dense4", "dense8", "dense8_whole", "skip", "masked8"])
def test_an_infinite_key_in_a_long_row(hip_device, bad_tile, mode):
    """A key with an infinity in it makes every row NaN that sees its tile, whichever step finds out, and ends no loop."""
    Lq, Lk = 200, 64 * 41
    print(f"case {mode} bad_tile={bad_tile}", flush=True)
    H = 256 if mode == "dense8_whole" else 1
    q, k, v = (t.to(torch.bfloat16).expand(1, -1, H, -1) for t in _inputs(Lq, Lk, 128, [11, 30], 3))
    ws = _quantized(q, k, v, hip_device)
    if mode.startswith("dense8"):
        assert (sage_ops.key_split_plan(ws) is None) == (H > 1)
    ws.k_scale[0, :, bad_tile] = float("inf")
    mask = torch.ones((2, 41), dtype=torch.int8)
    mask[1, bad_tile] = 0
    kw = {"dense4": {"wg_waves": 4}, "dense8": {"wg_waves": 8}, "dense8_whole": {"wg_waves": 8}, "skip": {"tile_skip": True}, "masked8": {"block_mask": mask, "wg_waves": 8}}[mode]
    out = sage_ops.attn_fwd(ws, torch.empty((1, Lq, H, 128), dtype=torch.bfloat16, device=hip_device), **kw).cpu()
    if mode == "masked8":
        four = sage_ops.attn_fwd(ws, torch.empty((1, Lq, 1, 128), dtype=torch.bfloat16, device=hip_device), block_mask=mask).cpu()
        assert out[0, :128].isnan().all() and torch.isfinite(out[0, 128:]).all()
        assert torch.equal(out[0, 128:], four[0, 128:]) and four[0, :128].isnan().all()
    else:
        assert out.isnan().all()


@pytest.mark.parametrize("lifted", [[], [9, 30], [2, 3]])
def test_shapes_and_variants_agree_on_long_rows(hip_device, lifted):
    """Both workgroup shapes, each with the tile skip and with an all-ones tile list: the same points, the same bits."""
    Lq, Lk, H = 256, 64 * 41, 260  # the first 256 heads are a full round of 8-wave workgroups: nobody's keys are cut there
    print(f"case lifted={lifted}", flush=True)
    q, k, v = (t.to(torch.bfloat16).expand(1, -1, H, -1).contiguous() for t in _inputs(Lq, Lk, 128, lifted, 5))
    ws = _quantized(q, k, v, hip_device)
    plan = sage_ops.key_split_plan(ws)
    assert plan is None or plan[0] >= 256
    ones = torch.ones((2, 41), dtype=torch.int8)
    outs = [sage_ops.attn_fwd(ws, torch.empty((1, Lq, H, 128), dtype=torch.bfloat16, device=hip_device), **kw)[:, :, :256].cpu()
            for kw in ({"wg_waves": 4}, {"wg_waves": 8}, {"wg_waves": 4, "tile_skip": True}, {"wg_waves": 8, "tile_skip": True},
                       {"block_mask": ones}, {"block_mask": ones, "wg_waves": 8})]
    for other in outs[1:]:
        assert torch.equal(outs[0], other)


# points that go on moving to the last tiles; that move once more after hundreds of tiles without; that hardly move
@pytest.mark.parametrize("lifted", [[1, 2, 3, 505, 511, 529, 538], [1, 2, 3, 100, 540], []])
@pytest.mark.parametrize("mode", ["dense4", "dense8", "masked", "causal"])
def test_very_long_rows_with_and_without_the_tile_skip(hip_device, lifted, mode):
    """More than 512 tiles, in the unrolled loop and in the tile skip's, which takes single steps: the same points, the same bits."""
    tiles, tail = 545, 9
    Lk = 64 * (tiles - 1) + tail
    Lq, H = (Lk, 1) if mode == "causal" else (256, 136 if mode == "dense8" else 2)  # (136 blocks: nobody's keys are cut)
    print(f"case {mode} lifted={lifted}", flush=True)
    q, k, v = (t.to(hip_device).to(torch.bfloat16).expand(1, -1, H, -1).contiguous() for t in _inputs(Lq, Lk, 128, lifted, 6))
    ws = _quantized(q, k, v, hip_device)
    kw = {"masked": {"block_mask": torch.ones((2, tiles), dtype=torch.int8)}, "causal": {"causal": True}}.get(mode, {"wg_waves": int(mode[-1]) if mode[-1].isdigit() else 0})
    if mode == "dense8":
        assert sage_ops.key_split_plan(ws) is None
    unrolled, single = (sage_ops.attn_fwd(ws, torch.empty_like(q), tile_skip=skip, **kw) for skip in (False, True))
    assert torch.isfinite(unrolled).all() and torch.equal(unrolled, single)
