"""Calls with few keys and many query rows, whose tiles stay in LDS, against the stage-wise entry points on the same inputs
(the general kernel on a quantized Q): the same operations in the same order, so the same bits."""

import pytest
import torch

from ksanadit_amd import sage_ops

pytestmark = pytest.mark.gpu


def _by_stages(q, k, v, **kw):
    ws = sage_ops.workspace_for(q, k)
    sage_ops.quant_q(q, ws, q.shape[-1] ** -0.5), sage_ops.quant_k(k, ws, True), sage_ops.quant_v(v, ws, kw.pop("smooth_v", False))
    return sage_ops.attn_fwd(ws, torch.empty_like(q), **kw)


def _inputs(hip_device, B, Hq, Hkv, Lq, Lk, D, dtype, seed):
    g = torch.Generator(device=hip_device).manual_seed(seed)
    q, k, v = (torch.randn((B, n, h, D), generator=g, device=hip_device) for n, h in ((Lq, Hq), (Lk, Hkv), (Lk, Hkv)))
    k += 2.0 * torch.randn((1, 1, Hkv, D), generator=g, device=hip_device)
    return (t.to(dtype) for t in (q, k, v))


# keys: one tile, ragged ones, odd and even numbers of tiles, the most that stay; rows: whole blocks, one row more, parts of
# equal and of unequal numbers of blocks, a workgroup for two rounds of heads
@pytest.mark.parametrize("Lk", [1, 64, 77, 128, 191, 256, 300, 448, 511, 512])
@pytest.mark.parametrize("B,Hq,Hkv,Lq,D,dtype", [(1, 40, 40, 16384, 128, torch.bfloat16), (2, 64, 16, 4097, 128, torch.float16),
                                                 (4, 128, 128, 1025, 64, torch.bfloat16)])
def test_same_bits_as_the_general_kernel(hip_device, B, Hq, Hkv, Lq, Lk, D, dtype):
    print(f"case B={B} Hq={Hq} Lq={Lq} Lk={Lk} D={D} {dtype}", flush=True)
    q, k, v = _inputs(hip_device, B, Hq, Hkv, Lq, Lk, D, dtype, Lk)
    assert torch.equal(sage_ops.sageattn(q, k, v), _by_stages(q, k, v))


def test_means_strides_values_that_are_not_finite_and_capture(hip_device):
    B, H, Lq, Lk = 1, 40, 14001, 200
    q, k, v = _inputs(hip_device, B, 2 * H, 2 * H, Lq, Lk, 128, torch.bfloat16, 5)
    q[0, 7, 3] = float("inf")
    q[0, 14000, 4] = float("nan")
    q, k, v = q[:, :, ::2], k[:, :, ::2], v[:, :, ::2] + 1.0
    got, want = sage_ops.sageattn(q, k, v), _by_stages(q.contiguous(), k.contiguous(), v.contiguous())
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.nan_to_num(got), torch.nan_to_num(want))
    q = torch.nan_to_num(q, nan=0.0, posinf=1.0)
    want = _by_stages(q.contiguous(), k.contiguous(), v.contiguous(), smooth_v=True)
    assert torch.equal(sage_ops.sageattn(q, k, v, smooth_v=True), want)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = sage_ops.sageattn(q, k, v, smooth_v=True)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
