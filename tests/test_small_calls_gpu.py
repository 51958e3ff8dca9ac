"""Calls of at most 256 keys without a workspace of their own run in one launch; with one they take the general path
(quantizers, then the attention kernel).  Both do the same operations in the same order on the same values, so every
comparison is bit for bit."""

import ctypes

import pytest
import torch

from ksanadit_amd import _capi, sage_ops

pytestmark = pytest.mark.gpu


def _tensors(B, Lq, Lk, Hq, Hkv, D, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn((B, n, h, D), generator=g) for n, h in ((Lq, Hq), (Lk, Hkv), (Lk, Hkv)))
    k += 2.0 * torch.randn((1, 1, Hkv, D), generator=g)
    q[torch.rand(q.shape, generator=g) < 1e-2] *= 20.0
    return tuple(t.to(dtype) for t in (q, k, v))


def _same(q, k, v, **kw):
    assert sage_ops._CallPlan(q, k, v).one_launch
    small = sage_ops.sageattn(q, k, v, **kw)
    general = sage_ops.sageattn(q, k, v, workspace=sage_ops.workspace_for(q, k), **kw)
    assert torch.equal(small, general)
    return small


@pytest.mark.parametrize("Lk", [1, 31, 32, 33, 63, 64, 65, 96, 128, 129, 192, 200, 255, 256])
@pytest.mark.parametrize("Lq", [1, 33, 128, 130, 300])
@pytest.mark.parametrize("causal", [False, True], ids=["dense", "causal"])
@pytest.mark.parametrize("D,dtype", [(128, torch.bfloat16), (128, torch.float16), (64, torch.bfloat16)])
def test_one_launch_gives_the_general_path_bits(hip_device, Lk, Lq, causal, D, dtype):
    print(f"case Lq={Lq} Lk={Lk} causal={causal} D={D} {dtype}", flush=True)
    q, k, v = (t.to(hip_device) for t in _tensors(2, Lq, Lk, 4, 2, D, dtype, 1000 * Lq + Lk))
    _same(q, k, v, is_causal=causal)


@pytest.mark.parametrize("Lq,Lk", [(40, 70), (200, 256), (129, 33)])
def test_counts_layouts_and_unsmoothed_keys(hip_device, Lq, Lk):
    """Key and query counts per batch entry (none, one, all), strided inputs, the [B, H, L, D] layout, keys as they are."""
    print(f"case Lq={Lq} Lk={Lk}", flush=True)
    q, k, v = (t.to(hip_device) for t in _tensors(3, Lq, Lk, 4, 4, 128, torch.bfloat16, 7 * Lq + Lk))
    out = _same(q, k, v, k_lens=[0, 1, Lk], q_lens=[Lq, Lq - 5, 1])
    assert (out[0] == 0).all() and (out[1, Lq - 5 :] == 0).all() and (out[2, 1:] == 0).all() and torch.isfinite(out.float()).all()
    _same(q, k, v, k_lens=[Lk // 2, Lk, 3], is_causal=True)
    _same(q, k, v, smooth_k=False)
    hnd = [t.transpose(1, 2) for t in (q, k, v)]
    assert torch.equal(sage_ops.sageattn(*hnd, tensor_layout="HND").transpose(1, 2), sage_ops.sageattn(q, k, v))
    wide = [torch.cat([t, t], dim=3)[..., :128] for t in (q, k, v)]
    assert torch.equal(sage_ops.sageattn(*wide), sage_ops.sageattn(q, k, v))


@pytest.mark.parametrize("what", ["infinite query", "infinite key", "zero keys", "zero values", "large values"])
def test_values_at_the_ends(hip_device, what):
    print(f"case {what}", flush=True)
    q, k, v = _tensors(1, 70, 100, 2, 2, 128, torch.bfloat16, 5)
    if what == "infinite query":
        q[0, 3, 0, 5] = float("inf")
    elif what == "infinite key":
        k[0, 9, 1, 5] = float("inf")
    elif what == "zero keys":
        k.zero_()
    elif what == "zero values":
        v.zero_()
    else:
        v *= 1e30
    q, k, v = (t.to(hip_device) for t in (q, k, v))
    small = sage_ops.sageattn(q, k, v)
    general = sage_ops.sageattn(q, k, v, workspace=sage_ops.workspace_for(q, k))
    assert torch.equal(torch.isnan(small), torch.isnan(general))
    assert torch.equal(torch.nan_to_num(small.float()), torch.nan_to_num(general.float()))


def test_which_calls_take_one_launch(hip_device):
    """Up to 256 keys and a bounded number of query blocks; options send a call down the general path."""
    def scratch(B, H, Lq, Lk, flags):
        shape, layout = _capi.workspace_layout(B, H, H, Lq, Lk, 128)
        n = ctypes.c_uint64(1)
        _capi.check(_capi.load().ksana_sage_forward_scratch(ctypes.byref(shape), flags, ctypes.byref(n)), "scratch")
        assert n.value in (0, layout.total_bytes)
        return n.value

    both = _capi.FLAG_Q_UNSTORED | _capi.FLAG_WS_UNSTORED
    assert scratch(2, 64, 32, 32, both) == 0 and scratch(1, 1, 1, 256, both) == 0
    assert scratch(4, 64, 256, 64, both) == 0 and scratch(1, 1, 256 * 256, 64, both) == 0
    assert scratch(1, 1, 1, 257, both) != 0 and scratch(4, 64, 257, 64, both) != 0 and scratch(1, 257, 1, 64, both) != 0
    for flags in (0, _capi.FLAG_Q_UNSTORED, _capi.FLAG_WS_UNSTORED, both | _capi.FLAG_PWL_EXP2, both | _capi.FLAG_SMOOTH_V,
                  both | _capi.FLAG_TILE_SKIP, both | _capi.FLAG_WG_4_WAVES):
        assert scratch(2, 64, 32, 32, flags) != 0
    q, k, v = (t.to(hip_device) for t in _tensors(1, 50, 60, 2, 2, 128, torch.bfloat16, 3))
    plain = sage_ops.sageattn(q, k, v)
    assert torch.equal(plain, sage_ops.sageattn(q, k, v, tile_skip=True))
    assert torch.equal(plain, sage_ops.sageattn(q, k, v, out_dtype=torch.bfloat16))


def test_captured_and_replayed(hip_device):
    q, k, v = (t.to(hip_device) for t in _tensors(2, 77, 150, 4, 4, 128, torch.bfloat16, 11))
    want = sage_ops.sageattn(q, k, v)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = sage_ops.sageattn(q, k, v)
    for i in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), i
        assert torch.equal(sage_ops.sageattn(q, k, v), want)


@pytest.mark.parametrize("pairs,Lq", [((1, 4), 65), ((2, 64), 64), ((2, 64), 65), ((2, 64), 97), ((2, 64), 130), ((2, 64), 257), ((4, 64), 33), ((4, 64), 225)])
@pytest.mark.parametrize("Lk", [32, 33, 97, 160])
@pytest.mark.parametrize("D", [64, 128])
def test_every_size_of_workgroup(hip_device, pairs, Lq, Lk, D):
    """32, 64, 128 and 256 query rows a workgroup (the fewest that leave a compute unit to each), with row groups that are part
    full or empty, and last tiles of at most 32 keys, of which the second half is left out."""
    (B, H), dtype = pairs, torch.float16 if Lk & 1 else torch.bfloat16
    print(f"case {pairs} Lq={Lq} Lk={Lk} D={D}", flush=True)
    q, k, v = (t.to(hip_device) for t in _tensors(B, Lq, Lk, H, H // 2, D, dtype, Lq + Lk + D))
    _same(q, k, v)
    _same(q, k, v, is_causal=True, k_lens=[Lk - 7 * b for b in range(B)], q_lens=[max(0, Lq - 40 * b) for b in range(B)])


@pytest.mark.parametrize("Lk", [40, 300])
def test_calls_without_options_and_the_general_call(hip_device, Lk):
    """A repeated call without options takes a shorter way to the library than one with an option that changes nothing
    (``out_dtype`` = the inputs' dtype): same result, same layout, whatever the layout and the kinds of its scalars."""
    print(f"case {Lk}", flush=True)
    q, k, v = (t.to(hip_device) for t in _tensors(2, 50, Lk, 4, 2, 128, torch.bfloat16, Lk))
    wide = [torch.cat([t, t], dim=3)[..., :128] for t in (q, k, v)]
    one = [t[:1] for t in (q, k, v)]
    odd = [t.as_strided((1, *t.shape[1:]), (8, *t.stride()[1:])) for t in (q, k, v)]  # an entry's stride nobody uses
    swapped = [t.transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k, v)]
    for tensors in ([q, k, v], wide, one, odd, swapped, [t.half() for t in (q, k, v)], [torch.nn.Parameter(t) for t in (q, k, v)]):
        for kw in ({}, {"sm_scale": 0.11}, {"sm_scale": 0.07, "is_causal": True}, {"smooth_k": False}, {"is_causal": 1, "sm_scale": 1}):
            want = sage_ops.sageattn(*tensors, **kw, out_dtype=tensors[0].dtype)
            for _ in range(2):
                out = sage_ops.sageattn(*tensors, **kw)
                assert torch.equal(out, want) and out.stride() == want.stride() and out.dtype == want.dtype and type(out) is torch.Tensor
    scale = torch.tensor(0.1)
    first = sage_ops.sageattn(q, k, v, sm_scale=scale)
    scale.fill_(0.3)  # a scale that is a tensor is read in every call
    assert torch.equal(sage_ops.sageattn(q, k, v, sm_scale=scale), sage_ops.sageattn(q, k, v, sm_scale=scale.item()))
    assert not torch.equal(sage_ops.sageattn(q, k, v, sm_scale=scale), first)
    for i in range(20):  # more settings than are kept
        assert torch.equal(sage_ops.sageattn(q, k, v, sm_scale=0.01 * i), sage_ops.sageattn(q, k, v, sm_scale=0.01 * i, out_dtype=q.dtype)), i
    named = [t.refine_names("B", "L", "H", "D") for t in (q, k, v)]  # names of the input are no names of the result, in any call
    for _ in range(2):
        out = sage_ops.sageattn(*named)
        assert not out.has_names() and torch.equal(out, sage_ops.sageattn(q, k, v))
    empty = q[:, :0]
    for _ in range(2):
        assert sage_ops.sageattn(empty, k, v).shape == empty.shape
