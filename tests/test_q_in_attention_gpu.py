"""Q quantized by the attention kernel itself (calls that bring no workspace, from one full round of workgroups and 257 keys
on) against Q quantized into the caller's workspace, which is pinned to the oracle bit for bit in test_quant_gpu.py: the
same result bits."""

import ctypes

import pytest
import torch

from ksanadit_amd import _capi, sage_ops

pytestmark = pytest.mark.gpu


def _tensors(hip_device, B, Lq, Lk, Hq, Hkv, D, dtype, strided=False):
    g = torch.Generator(device=hip_device).manual_seed(Lq + 7 * Lk + D)

    def draw(L, H):
        x = torch.randn((B, L, H + (1 if strided else 0), D), generator=g, device=hip_device)
        x = torch.where(torch.rand(x.shape, generator=g, device=hip_device) < 2e-3, x * 20.0, x)
        return x.to(dtype)[:, :, :H]

    return draw(Lq, Hq), draw(Lk, Hkv), draw(Lk, Hkv)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,Lq,Lk,Hq,Hkv,D,kw", [
    (2, 1, 257, 128, 32, 128, {}), (2, 33, 300, 128, 128, 64, {}), (1, 257, 300, 128, 128, 64, dict(pwl_exp2=True)),
    (1, 300, 300, 128, 64, 128, dict(is_causal=True)), (1, 300, 300, 128, 16, 64, dict(is_causal=True)),
    (2, 200, 330, 128, 128, 128, dict(tile_skip=True)), (1, 300, 300, 128, 128, 128, dict(smooth_v=True)),
    (1, 1000, 64 * 33, 65, 65, 128, {}),  # whole and cut query blocks in one grid (8 waves)
    (2, 500, 700, 64, 64, 128, dict(k_lens=[700, 65], q_lens=[500, 131])),
    (1, 33, 256 * 64, 256, 2, 128, {}), (1, 33, 256 * 64 + 1, 256, 2, 128, {}),  # 256 tiles, and one more: through memory again
    (1, 255, 300, 255, 255, 128, {}),  # one workgroup short of a round: through memory
    (1, 260, 500, 128, 128, 128, "mask")])  # (through memory)
def test_same_bits_as_through_the_workspace(hip_device, B, Lq, Lk, Hq, Hkv, D, kw, dtype):
    print(f"case B={B} Lq={Lq} Lk={Lk} Hq={Hq} Hkv={Hkv} D={D} {kw} {dtype}", flush=True)
    for strided in (False, True):
        q, k, v = _tensors(hip_device, B, Lq, Lk, Hq, Hkv, D, dtype, strided)
        q[:, 0, 0] = 0  # a row whose scale is zero
        args = dict(kw) if kw != "mask" else {}
        if kw == "mask":
            g = torch.Generator().manual_seed(1)
            args["block_mask"] = (torch.rand((B, Hq, -(-Lq // 128), -(-Lk // 64)), generator=g) < 0.6).to(torch.int8)
        want = sage_ops.sageattn(q, k, v, workspace=sage_ops.workspace_for(q, k), **args)
        assert torch.equal(sage_ops.sageattn(q, k, v, **args), want)


def test_rows_that_are_not_finite(hip_device):
    print("case rows with inf and NaN", flush=True)
    q, k, v = _tensors(hip_device, 1, 300, 500, 128, 128, 128, torch.bfloat16)
    q[0, 5, 0, 7], q[0, 70, 1, 127], q[0, 299, 0, 64] = float("inf"), float("nan"), -float("inf")
    want = sage_ops.sageattn(q, k, v, workspace=sage_ops.workspace_for(q, k))
    out = sage_ops.sageattn(q, k, v)
    finite = torch.isfinite(q).all(-1)
    assert torch.equal(out[finite], want[finite]) and torch.isfinite(out[finite]).all()
    assert torch.equal(torch.isnan(out), torch.isnan(want))


@pytest.mark.parametrize("Hq,Lk,unstored,o_dtype,leaves_q", [
    (256, 257, True, torch.bfloat16, True), (256, 257, False, torch.bfloat16, False), (256, 256, True, torch.bfloat16, False),
    (255, 257, True, torch.bfloat16, False), (256, 257, True, torch.float16, False)])
def test_which_calls_leave_the_codes_unwritten(hip_device, Hq, Lk, unstored, o_dtype, leaves_q):
    if torch.cuda.get_device_properties(hip_device).multi_processor_count != 256:
        pytest.skip("the sizes are those of a chip of 256 compute units")
    print(f"case Hq={Hq} Lk={Lk} unstored={unstored} {o_dtype}", flush=True)
    q, k, v = _tensors(hip_device, 1, 33, Lk, Hq, Hq, 128, torch.bfloat16)
    ws, out = sage_ops.workspace_for(q, k), torch.empty(q.shape, dtype=o_dtype, device=hip_device)
    ws.blob.fill_(0x7F)
    st = [_capi.Strides(*t.stride()) for t in (q, k, v, out)]
    rc = _capi.load().ksana_sage_forward_varlen(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), sage_ops._DTYPES[q.dtype], sage_ops._DTYPES[o_dtype], *st,
        ctypes.byref(ws.shape), None, None, None, None, None, 128**-0.5, 1, 0, _capi.FLAG_Q_UNSTORED if unstored else 0, ws.blob.data_ptr(),
        torch.cuda.current_stream(hip_device).cuda_stream)
    assert rc == _capi.OK
    assert bool((ws.q_i8 == 0x7F).all()) == leaves_q
