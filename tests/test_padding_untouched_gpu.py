"""Batches with lengths of their own, workspace unseen: blocks of rows or keys that take no part are not quantized.  Against the
stage-wise entry points, which quantize everything: the statistics are the same, so the results are the same bits."""

import pytest
import torch

from ksanadit_amd import sage_ops

pytestmark = pytest.mark.gpu


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
        got = sage_ops.sageattn(q, k, v, **kw)
        torch.empty_like(got).fill_(float("nan"))  # what the allocator hands out next is not a finished result
        assert torch.equal(got, sage_ops.attn_fwd(ws, torch.empty_like(q), **kw)), (k_lens, q_lens)
