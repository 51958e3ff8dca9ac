"""The sparse-linear backend's whole call against the entry points it joins, called one after the other on the same inputs:
statistics, codes, averages, map, attention and both passes of the linear branch do the same operations in the same order
there, so the results are the same bits."""

import pytest
import torch

from ksanadit_amd import sage_ops

pytestmark = pytest.mark.gpu


def _one_by_one(q, k, v, keep, w, b):
    ws = sage_ops.workspace_for(q, k)
    pooled_q, pooled_k = sage_ops.quant_qk_pooled(q, k, ws, 128**-0.5)
    sage_ops.quant_v(v, ws)
    sparse = sage_ops.attn_fwd(ws, torch.empty_like(q), block_mask=sage_ops.sla_block_map(pooled_q, pooled_k, keep))
    return sage_ops.sla_linear(q, k, v, w, b, add=sparse)


# chunks of 256 rows: part of one, one, one and a row, several, 63, 64 (from where a launch in between finishes the statistics)
@pytest.mark.parametrize("B,H,L", [(1, 1, 1), (2, 3, 63), (1, 2, 256), (2, 2, 257), (1, 3, 1000), (2, 24, 1100), (1, 1, 63 * 256), (1, 2, 63 * 256 + 1)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_whole_call_is_its_parts(hip_device, B, H, L, dtype):
    print(f"case B={B} H={H} L={L} {dtype}", flush=True)
    g = torch.Generator().manual_seed(L)
    q, k, v = (torch.randn((B, L, H, 128), generator=g) for _ in range(3))
    k += 2.0 * torch.randn((1, 1, H, 128), generator=g)
    w, b = torch.randn((128, 128), generator=g) * 0.05, torch.randn(128, generator=g)
    q, k, v, w, b = (t.to(dtype).to(hip_device) for t in (q, k, v, w, b))
    nk = -(-L // 64)
    for keep in sorted({0, min(1, nk), max(1, nk // 10), nk}):
        for bias in (b, None):
            got = sage_ops.sla_forward(q, k, v, keep, w, bias)
            assert torch.equal(got, _one_by_one(q, k, v, keep, w, bias)), (keep, bias is None)


def test_strided_inputs_and_capture(hip_device):
    g = torch.Generator().manual_seed(4)
    wide = [torch.randn((2, 900, 5, 128), generator=g).to(torch.bfloat16).to(hip_device) for _ in range(3)]
    q, k, v = (t[:, 100:800, 1:4] for t in wide)
    w = (torch.randn((128, 128), generator=g) * 0.05).to(torch.bfloat16).to(hip_device)
    want = _one_by_one(q.contiguous(), k.contiguous(), v.contiguous(), 2, w, None)
    assert torch.equal(sage_ops.sla_forward(q, k, v, 2, w), want)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = sage_ops.sla_forward(q, k, v, 2, w)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        assert torch.equal(sage_ops.sla_forward(q, k, v, 2, w), want)
