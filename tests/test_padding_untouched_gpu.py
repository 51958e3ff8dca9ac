"""Batches with lengths of their own: what takes no part.  Workspace unseen, blocks of such rows or keys are not quantized; against the
stage-wise entry points, which quantize everything: the statistics are the same, so the results are the same bits."""

import pytest
import torch

from ksanadit_amd import sage_ops

pytestmark = pytest.mark.gpu


def _spoil(q, ws):
    """What the allocator hands out next, a result and a workspace, holds neither a finished result nor an earlier call's codes."""
    mem = torch.full_like(q, float("nan")), torch.full((ws.layout.total_bytes,), 0xFF, dtype=torch.uint8, device=q.device)
    del mem


# (B, Hq, Hkv, Lq, Lk): all quantizers in one launch, two stages with one and two tiles a workgroup, K's and V's chunks meeting
@pytest.mark.parametrize("B,Hq,Hkv,Lq,Lk", [(5, 64, 32, 900, 230), (5, 4, 2, 700, 1500), (5, 24, 24, 300, 3000), (5, 8, 8, 200, 17000)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_same_bits_as_with_everything_quantized(hip_device, B, Hq, Hkv, Lq, Lk, dtype):
    print(f"case B={B} Hq={Hq} Lq={Lq} Lk={Lk} {dtype}", flush=True)
    g = torch.Generator(device=hip_device).manual_seed(Lk)
    q, k, v = (torch.randn((B, n, h, 128), generator=g, device=hip_device).to(dtype) for n, h in ((Lq, Hq), (Lk, Hkv), (Lk, Hkv)))
    k += 1.5
    ws = sage_ops.workspace_for(q, k)
    sage_ops.quant_q(q, ws, 128**-0.5), sage_ops.quant_k(k, ws, True), sage_ops.quant_v(v, ws)
    for k_lens, q_lens in (([Lk, 0, 1, 64, Lk // 2 + 1], None), ([Lk - 64, Lk // 3, 65, Lk, 128], [Lq, 1, 0, 128, Lq // 2])):
        kw = dict(k_lens=torch.tensor(k_lens, dtype=torch.int32, device=hip_device))
        if q_lens is not None:
            kw["q_lens"] = torch.tensor(q_lens, dtype=torch.int32, device=hip_device)
        _spoil(q, ws)
        got = sage_ops.sageattn(q, k, v, **kw)
        assert torch.equal(got, sage_ops.attn_fwd(ws, torch.empty_like(q), **kw)), (k_lens, q_lens)


INT_MAX, INT_MIN = 2**31 - 1, -(2**31)


# (.. and the calls of one launch, and K and V of less than a tile)
@pytest.mark.parametrize("B,Hq,Hkv,Lq,Lk", [(5, 4, 4, 100, 37), (5, 8, 4, 300, 230), (5, 64, 32, 900, 230), (5, 4, 2, 700, 1500), (5, 8, 8, 200, 17000)])
def test_counts_of_any_value_are_clamped(hip_device, B, Hq, Hkv, Lq, Lk):
    """A count is clamped to the tensor before anything is added to it: negative ones are none, those beyond the tensor all."""
    print(f"case B={B} Hq={Hq} Lq={Lq} Lk={Lk}", flush=True)
    g = torch.Generator(device=hip_device).manual_seed(Lk)
    q, k, v = (torch.randn((B, n, h, 128), generator=g, device=hip_device).bfloat16() for n, h in ((Lq, Hq), (Lk, Hkv), (Lk, Hkv)))
    ws = sage_ops.workspace_for(q, k)
    sage_ops.quant_q(q, ws, 128**-0.5), sage_ops.quant_k(k, ws, True), sage_ops.quant_v(v, ws)
    for k_lens, q_lens in (([INT_MAX, INT_MAX - 62, INT_MAX - 63, Lk + 1, Lk - 1], [INT_MAX, Lq + 1, Lq - 1, INT_MAX - 62, 1]),
                           ([-1, INT_MIN, -Lk, 1, INT_MAX], [Lq, Lq, Lq, INT_MIN, -1])):
        within = [[max(0, min(n, most)) for n in lens] for lens, most in ((k_lens, Lk), (q_lens, Lq))]
        as_given, clamped = ([torch.tensor(x, dtype=torch.int32, device=hip_device) for x in pair] for pair in ((k_lens, q_lens), within))
        want = sage_ops.attn_fwd(ws, torch.empty_like(q), k_lens=clamped[0], q_lens=clamped[1])
        for lens in (as_given, clamped):
            _spoil(q, ws)
            assert torch.equal(sage_ops.sageattn(q, k, v, k_lens=lens[0], q_lens=lens[1]), want), (k_lens, q_lens)
        assert torch.equal(sage_ops.attn_fwd(ws, torch.empty_like(q), k_lens=as_given[0], q_lens=as_given[1]), want), (k_lens, q_lens)
        for b, (n_k, n_q) in enumerate(zip(*within)):
            assert (want[b, n_q:] == 0).all() and (n_k > 0 or (want[b] == 0).all())


@pytest.mark.parametrize("kw", [dict(), dict(is_causal=True), dict(mask=True), dict(mask=True, is_causal=True), dict(mask=True, wg_waves=8), dict(wg_waves=4),
                                dict(wg_waves=8), dict(smooth_v=True), dict(pwl_exp2=True), dict(tile_skip=True)], ids=lambda kw: "-".join(map(str, kw)) or "plain")
# (one launch; the attention kernel quantizes Q; Q quantized apart, keys in runs; a last block whose waves share the keys)
@pytest.mark.parametrize("H,Lq,Lk,D", [(4, 100, 200, 128), (4, 100, 200, 64), (64, 400, 600, 128), (64, 400, 600, 64), (2, 600, 1100, 128), (16, 300, 1100, 128)])
def test_rows_that_do_not_count_are_zeros_whatever_they_hold(hip_device, H, Lq, Lk, D, kw):
    """Infinities and NaN in the padding rows of q, and infinite values: the rows that do not count are written as zeros, the
    others as ever."""
    print(f"case H={H} Lq={Lq} Lk={Lk} D={D} {kw}", flush=True)
    kw = dict(kw)
    g = torch.Generator(device=hip_device).manual_seed(Lq + D)
    q, k, v = (torch.randn((3, n, H, D), generator=g, device=hip_device).bfloat16() for n in (Lq, Lk, Lk))
    if kw.pop("mask", False):
        kw["block_mask"] = (torch.rand((-(-Lq // 128), -(-Lk // 64)), generator=g, device=hip_device) < 0.6).to(torch.int8)
        kw["block_mask"][:, 0] = 1
    q_lens = [Lq, Lq - 5, 33]
    kw["q_lens"] = torch.tensor(q_lens, dtype=torch.int32, device=hip_device)

    def call():
        if "wg_waves" not in kw:
            return sage_ops.sageattn(q, k, v, **kw)
        ws = sage_ops.workspace_for(q, k)
        sage_ops.quant_q(q, ws, D**-0.5), sage_ops.quant_k(k, ws, True), sage_ops.quant_v(v, ws)
        return sage_ops.attn_fwd(ws, torch.full_like(q, float("nan")), **kw)

    want = call()
    for b, n in enumerate(q_lens):
        q[b, n:, 0], q[b, n:, 1, 3] = float("inf"), float("-inf")
        q[b, n + 1 :: 3] = float("nan")
    for _ in range(2):
        got = call()
        for b, n in enumerate(q_lens):
            assert (got[b, n:] == 0).all(), f"entry {b}: {int((got[b, n:] != 0).sum())} values of the padding are not zero"
            if want is not None:
                assert torch.equal(got[b, :n], want[b, :n]), f"entry {b}: rows that count have changed"
        v[:, Lk // 2, 0, 1], want = float("inf"), None
