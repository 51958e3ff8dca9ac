"""Q, K and V quantized together (the first launches of a whole call) against the separate quantizers, which are pinned
to the oracle bit for bit in test_quant_gpu.py and test_prep_gpu.py: the same bits in every area of the workspace."""

import pytest
import torch

from ksanadit_amd import sage_ops

pytestmark = pytest.mark.gpu

AREAS = ("q_i8", "q_scale", "k_tiles", "k_scale", "k_mean", "v_tiles", "v_scale", "v_mean")


def _compare(hip_device, B, Lq, Lk, Hq, Hkv, D, dtype, smooth_k=True, prep=None, strided=False):
    g = torch.Generator(device=hip_device).manual_seed(Lq + 7 * Lk + D)

    def draw(L, H):
        x = torch.randn((B, L, H + (1 if strided else 0), D), generator=g, device=hip_device)
        x = x + 2.0 * torch.randn((H + (1 if strided else 0), D), generator=g, device=hip_device)
        return x.to(dtype)[:, :, :H]

    q, k, v = draw(Lq, Hq), draw(Lk, Hkv), draw(Lk, Hkv)
    v[:, :, 0, 3] = 0  # a channel that is zero throughout
    k[:, : min(64, Lk), 0] = 0
    ws, want = sage_ops.workspace_for(q, k), sage_ops.workspace_for(q, k)
    ws.blob.fill_(0x7F), want.blob.fill_(0x7F)
    out = sage_ops.sageattn(q, k, v, workspace=ws, smooth_k=smooth_k, prep=prep)
    sage_ops.quant_qk(q, k, want, D**-0.5, smooth_k, prep=prep)
    sage_ops.quant_v(v, want)
    for name in AREAS:
        assert torch.equal(getattr(ws, name).view(torch.uint8), getattr(want, name).view(torch.uint8)), name
    assert sage_ops.quant_status(ws) == (0, 0)
    assert torch.equal(out, sage_ops.attn_fwd(want, torch.empty_like(out)))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,Lq,Lk,Hq,Hkv,D,smooth_k", [
    (2, 32, 32, 4, 4, 128, True), (1, 1, 1, 1, 1, 128, True), (1, 300, 256, 2, 1, 128, True), (1, 40, 256, 2, 2, 64, False),
    (1, 129, 257, 3, 3, 128, True), (2, 513, 1560, 4, 2, 128, True), (1, 100, 640, 2, 2, 64, True), (1, 64, 700, 2, 2, 128, False),
    (1, 200, 16384, 2, 2, 128, True), (1, 64, 16385, 1, 1, 128, True), (1, 128, 8300, 16, 16, 128, True),
    (1, 128, 20000, 24, 12, 128, True), (1, 128, 17000, 1, 1, 64, False),
    (1, 128, 4096 - 64, 16, 16, 128, True), (1, 128, 4096 + 64, 16, 16, 128, True)])  # 2016 and 2080 tiles: one and two a workgroup
def test_together_gives_the_separate_quantizers_bits(hip_device, B, Lq, Lk, Hq, Hkv, D, smooth_k, dtype):
    print(f"case B={B} Lq={Lq} Lk={Lk} Hq={Hq} Hkv={Hkv} D={D} smooth_k={smooth_k} {dtype}", flush=True)
    _compare(hip_device, B, Lq, Lk, Hq, Hkv, D, dtype, smooth_k)
    _compare(hip_device, B, Lq, Lk, Hq, Hkv, D, dtype, smooth_k, strided=True)


@pytest.mark.parametrize("txt,img,weights,tables", [(5, 60, True, True), (256, 1000, True, True), (300, 400, False, True), (13, 3000, True, False)])
def test_together_with_the_joint_block_step(hip_device, txt, img, weights, tables):
    print(f"case txt={txt} img={img} weights={weights} tables={tables}", flush=True)
    g = torch.Generator(device=hip_device).manual_seed(txt)
    ws = [1.0 + 0.2 * torch.randn(128, generator=g, device=hip_device) if weights else None for _ in range(4)]
    ang = torch.rand((txt + img, 64), generator=g, device=hip_device) * 6.0
    tab = torch.polar(torch.ones_like(ang), ang) if tables else None
    prep = sage_ops.QwenPrep(txt, *ws, 1e-6, img_freqs=None if tab is None else tab[:img].contiguous(),
                             txt_freqs=None if tab is None else tab[img:].contiguous())
    _compare(hip_device, 2, txt + img, txt + img, 3, 3, 128, torch.bfloat16, True, prep)


@pytest.mark.parametrize("B,txt,img,H", [
    (1, 56, 13576, 24), (1, 56, 13676, 24),    # 159.75 and 160.9 MB of K and V: the last size in two stages, separate kernels
    (1, 100, 16284, 1), (1, 100, 16285, 1),    # 64 chunks of keys, and one row more
    (1, 100, 5340, 24), (1, 100, 5468, 24)])   # 4080 and (an odd number a head) 4176 tiles: one and two a workgroup of stage 2
def test_together_with_the_joint_block_step_at_its_limits(hip_device, B, txt, img, H):
    print(f"case B={B} txt={txt} img={img} H={H}", flush=True)
    g = torch.Generator(device=hip_device).manual_seed(img)
    ws = [1.0 + 0.2 * torch.randn(128, generator=g, device=hip_device) for _ in range(4)]
    ang = torch.rand((txt + img, 64), generator=g, device=hip_device) * 6.0
    tab = torch.polar(torch.ones_like(ang), ang)
    prep = sage_ops.QwenPrep(txt, *ws, 1e-6, img_freqs=tab[:img].contiguous(), txt_freqs=tab[img:].contiguous())
    _compare(hip_device, B, txt + img, txt + img, H, H, 128, torch.bfloat16, True, prep)


@pytest.mark.parametrize("B,txt,img,Hq,Hkv,weights,tables,dtype", [
    (2, 52, 1284, 24, 24, True, True, torch.bfloat16), (2, 52, 1228, 24, 24, True, True, torch.bfloat16),  # 1104 and 1008 workgroups: several heads, one
    (2, 13, 1401, 27, 27, True, True, torch.float16),      # heads that leave both groups incomplete, ragged lengths
    (3, 200, 1700, 18, 9, False, True, torch.bfloat16), (2, 0, 2500, 21, 21, True, False, torch.bfloat16)])
def test_the_joint_block_step_on_several_heads_per_item(hip_device, B, txt, img, Hq, Hkv, weights, tables, dtype):
    print(f"case B={B} txt={txt} img={img} Hq={Hq} Hkv={Hkv} weights={weights} tables={tables} {dtype}", flush=True)
    g = torch.Generator(device=hip_device).manual_seed(img)
    ws = [1.0 + 0.2 * torch.randn(128, generator=g, device=hip_device) if weights else None for _ in range(4)]
    ang = torch.rand((txt + img, 64), generator=g, device=hip_device) * 6.0
    tab = torch.polar(torch.ones_like(ang), ang) if tables else None
    prep = sage_ops.QwenPrep(txt, *ws, 1e-6, img_freqs=None if tab is None else tab[:img].contiguous(),
                             txt_freqs=None if tab is None or txt == 0 else tab[img:].contiguous())
    _compare(hip_device, B, txt + img, txt + img, Hq, Hkv, 128, dtype, True, prep)


@pytest.mark.parametrize("img", [8136, 8137])    # 192 MB of K and V: the last size in two stages, and separate kernels
def test_together_with_the_joint_block_step_at_192_mb(hip_device, img):
    print(f"case img={img}", flush=True)
    B, txt, H = 2, 56, 24
    assert (2 * B * (txt + img) * H * 128 * 2 <= 192 << 20) == (img == 8136)
    ang = torch.rand((txt + img, 64), generator=torch.Generator(device=hip_device).manual_seed(img), device=hip_device) * 6.0
    tab = torch.polar(torch.ones_like(ang), ang)
    prep = sage_ops.QwenPrep(txt, None, None, None, None, 1e-6, img_freqs=tab[:img].contiguous(), txt_freqs=tab[img:].contiguous())
    _compare(hip_device, B, txt + img, txt + img, H, H, 128, torch.bfloat16, True, prep)


# K and V in one launch, K of several chunks and of one, other numbers of keys and heads; 5760 workgroups: a launch each, their
# counters cleared by Q's; no norm of k or of q: K's statistic is not there yet, or Q's kernel is another one
@pytest.mark.parametrize("B,Lq,Lk,Hq,Hkv,norm,rotation", [
    (1, 300, 300, 12, 12, "qk", "wan"), (2, 1000, 1000, 3, 3, "qk", "comfy"), (2, 200, 520, 4, 4, "qk", None), (1, 520, 70, 8, 4, "qk", None),
    (1, 15360, 15360, 48, 48, "qk", "wan"), (1, 640, 640, 4, 4, "q", "wan"), (1, 640, 640, 4, 4, "k", "wan")])
def test_the_row_norm_step_in_whole_calls(hip_device, B, Lq, Lk, Hq, Hkv, norm, rotation):
    print(f"case B={B} Lq={Lq} Lk={Lk} Hq={Hq} Hkv={Hkv} {norm} {rotation}", flush=True)
    g = torch.Generator(device=hip_device).manual_seed(Lk)
    wq, wk = (1.0 + 0.2 * torch.randn(h * 128, generator=g, device=hip_device) if n in norm else None for n, h in (("q", Hq), ("k", Hkv)))
    kw = {}
    if rotation == "wan":
        ang = torch.rand((1024, 64), generator=g, device=hip_device, dtype=torch.float64) * 6.0
        kw = dict(freqs=torch.polar(torch.ones_like(ang), ang), grid_sizes=[(Lq // 20, 4, 5)] * B)
    if rotation == "comfy":
        kw = dict(comfy_freqs=torch.randn((Lq - 7, 64, 2, 2), generator=g, device=hip_device))
    _compare(hip_device, B, Lq, Lk, Hq, Hkv, 128, torch.bfloat16, True, sage_ops.WanPrep(wq, wk, 1e-6, **kw))


# 1140 and 1152, 1536 and 1584, 5376 and 5424 workgroups: one launch for K and V below 1.5 rounds of 768 and from 2 to 7
@pytest.mark.parametrize("B,Lk,H", [(1, 24300, 6), (1, 24400, 6), (2, 8192, 12), (2, 8200, 12), (1, 28672, 24), (1, 28700, 24)])
def test_the_row_norm_step_where_one_launch_starts_and_ends(hip_device, B, Lk, H):
    print(f"case B={B} Lk={Lk} H={H}", flush=True)
    g = torch.Generator(device=hip_device).manual_seed(Lk)
    wq, wk = (1.0 + 0.2 * torch.randn(H * 128, generator=g, device=hip_device) for _ in range(2))
    ang = torch.rand((1024, 64), generator=g, device=hip_device, dtype=torch.float64) * 6.0
    prep = sage_ops.WanPrep(wq, wk, 1e-6, freqs=torch.polar(torch.ones_like(ang), ang), grid_sizes=[(2, 4, 5)] * B)
    _compare(hip_device, B, 40, Lk, H, H, 128, torch.bfloat16, True, prep)


def _inputs(hip_device, B, Lk, Hq, Hkv, D, dtype):
    g = torch.Generator(device=hip_device).manual_seed(Lk + D)
    k = torch.randn((B, Lk, Hkv, D), generator=g, device=hip_device) + 2.0 * torch.randn((Hkv, D), generator=g, device=hip_device)
    q, v = (torch.randn((B, n, h, D), generator=g, device=hip_device) for n, h in ((128, Hq), (Lk, Hkv)))
    return q.to(dtype), k.to(dtype), v.to(dtype)


def _same_areas(ws, want):
    for name in AREAS:
        assert torch.equal(getattr(ws, name).view(torch.uint8), getattr(want, name).view(torch.uint8)), name


@pytest.mark.parametrize("B,Lk,Hq,Hkv,D,dtype,smooth_k", [
    (1, 16385, 1, 1, 128, torch.bfloat16, True), (2, 17000, 4, 2, 128, torch.float16, True), (1, 16641, 2, 2, 64, torch.bfloat16, True),
    (2, 8500, 24, 24, 128, torch.bfloat16, True), (1, 20000, 2, 2, 128, torch.bfloat16, False)])
def test_the_meeting_launch_stays_exact_when_its_waits_run_out(hip_device, quant_settings, B, Lk, Hq, Hkv, D, dtype, smooth_k):
    """K's and V's chunks share one launch and one area of counters; with a negative bound every workgroup but the last
    arrivers of its head's K and V takes the statistic from the input."""
    print(f"case B={B} Lk={Lk} Hq={Hq} Hkv={Hkv} D={D} {dtype} smooth_k={smooth_k}", flush=True)
    q, k, v = _inputs(hip_device, B, Lk, Hq, Hkv, D, dtype)
    ws, want = sage_ops.workspace_for(q, k), sage_ops.workspace_for(q, k)
    ws.blob.fill_(0x7F), want.blob.fill_(0x7F)
    sage_ops.quant_qk(q, k, want, D**-0.5, smooth_k)
    sage_ops.quant_v(v, want)
    for bound in (-1, 0):  # 0: which workgroups give up depends on timing
        quant_settings(wait_ticks=bound)
        sage_ops.sageattn(q, k, v, workspace=ws, smooth_k=smooth_k)
        status = sage_ops.quant_status(ws)
        if bound < 0:
            assert status == (1 if smooth_k else 0, 1)  # without a mean to take off K waits for nobody
        _same_areas(ws, want)
        assert not sage_ops.one_read_state()["demoted"]  # test-mode bounds switch nothing off
    quant_settings(wait_ticks=200000)
    sage_ops.sageattn(q, k, v, workspace=ws, smooth_k=smooth_k)
    assert sage_ops.quant_status(ws) == (0, 0)
    _same_areas(ws, want)


def test_an_expired_bound_of_the_meeting_launch_switches_it_off(hip_device, quant_settings):
    print("case expired bound, whole call", flush=True)
    q, k, v = _inputs(hip_device, 1, 20000, 8, 8, 128, torch.bfloat16)
    ws, want = sage_ops.workspace_for(q, k), sage_ops.workspace_for(q, k)
    sage_ops.quant_qk(q, k, want, 128**-0.5)
    sage_ops.quant_v(v, want)
    quant_settings(wait_ticks=1)  # 10 ns: any workgroup that finds its head's flag down twice gives up
    sage_ops.sageattn(q, k, v, workspace=ws)
    _same_areas(ws, want)
    if sage_ops.quant_status(ws) == (0, 0):
        pytest.skip("no workgroup had to wait for its head in this run")
    assert sage_ops.one_read_state()["demoted"]
    ws.blob.fill_(0x7F)
    sage_ops.sageattn(q, k, v, workspace=ws)  # the separate two-pass kernels: nobody waits
    assert sage_ops.quant_status(ws) == (0, 0)
    _same_areas(ws, want)


@pytest.mark.parametrize("Lk,qwen,smooth_v,waits", [
    (16384, False, False, {"v": (0, 0), "": (0, 0), "k": (0, 0), "kv": (0, 0)}),   # two stages: nobody waits
    (16385, False, False, {"v": (1, 1), "": (0, 0), "k": (1, 0), "kv": (1, 1)}),   # one launch with "v", separate kernels without
    (41000, False, False, {"v": (0, 1), "": (0, 0), "k": (1, 0), "kv": (1, 1)}),   # more than 160 chunks: separate kernels
    (16385, True, False, {"v": (1, 1), "": (1, 0), "k": (1, 0), "kv": (1, 1)}),    # with a folded step K tries to read once
    (3000, False, True, {"v": (0, 0), "": (0, 0), "k": (1, 0), "kv": (1, 0)})])    # V smoothing: separate kernels, V in passes
def test_which_settings_make_whole_calls_wait(hip_device, quant_settings, Lk, qwen, smooth_v, waits):
    """The routes of ``ksana_sage_configure``'s letters, seen through the status words of calls whose workgroups never look at
    a flag: 1 where a stage's workgroups meet."""
    q, k, v = _inputs(hip_device, 1, Lk, 1, 1, 128, torch.bfloat16)
    prep = None
    if qwen:
        q, w = k.flip(1), torch.ones(128, device=hip_device)
        prep = sage_ops.QwenPrep(5, w, w, w, w, 1e-6)
    ws = sage_ops.workspace_for(q, k)
    for letters, status in waits.items():
        print(f"case Lk={Lk} qwen={qwen} smooth_v={smooth_v} letters={letters!r}", flush=True)
        quant_settings(one_read=letters, wait_ticks=-1)
        ws.blob.fill_(0x7F)
        sage_ops.sageattn(q, k, v, workspace=ws, prep=prep, smooth_v=smooth_v)
        assert sage_ops.quant_status(ws) == status, letters
