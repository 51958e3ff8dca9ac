"""The attention calls this package is timed on: what a diffusion transformer (and the package's other users) ask of it.

``listed()`` are fixed cases, ``draw(rng)`` gives more of the same ranges, ``prepare`` makes what a caller holds before
the call, ``run`` is one call through the public entry points, ``work`` counts the bytes and operations the call cannot
do without and ``tolerance`` says how far two correct implementations may differ.

Kinds of call:

* ``op``      the operator a block holds, ``pick_attn_op(config)(heads, head size)`` -> ``op(q, k, v)``, dense or causal;
* ``cross``   the same operator with a short key sequence (video tokens attend to text tokens);
* ``wan``     ``wan_self_attention`` on raw projections: token-row RMSNorm and 3-axis rotation folded in;
* ``qwen``    ``sageattn`` on the joint text + image sequence with the per-head RMSNorm and rotation folded in;
* ``varlen``  ``sageattn`` on a padded batch with a key count and a query count per batch entry;
* ``radial``  the radial block-sparse backend's operator;
* ``sla``     the sparse-linear backend's operator with the block's linear layer.
"""

import math

import torch

from ksanadit_amd import KsanaAttentionBackend, KsanaAttentionConfig, pick_attn_op
from ksanadit_amd.config import KsanaRadialSageAttentionConfig, KsanaSageSLAConfig
from ksanadit_amd.sage_ops import QwenPrep, WanPrep, sageattn, wan_self_attention

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
DEVICE = "cuda"


def listed():
    return [
        # A unit-test-sized call: nothing but the path's latency (launches and host work).
        dict(name="unit_fp16", kind="op", B=2, H=64, Hkv=64, Lq=32, Lk=32, D=128, dtype="fp16", outliers=0.0, causal=False),
        # One latent frame of a 480p video (30 x 52 tokens): the first block of a streaming generation, image models at
        # small sizes; still near the latency of the call.
        dict(name="one_frame_480p", kind="op", B=1, H=40, Hkv=40, Lq=1560, Lk=1560, D=128, dtype="bf16", outliers=0.0, causal=False),
        # Joint text + image attention of a 1024 x 1024 image, conditional and unconditional pass as one batch.
        dict(name="joint_image_pair", kind="qwen", B=2, H=24, txt=256, img=4096, D=128, dtype="bf16"),
        # Every video token attends to the 512 text tokens: once per block, next to the self-attention.
        dict(name="cross_text_480p", kind="cross", B=1, H=40, Hkv=40, Lq=32760, Lk=512, D=128, dtype="bf16", outliers=0.0, causal=False),
        # A padded batch of unequal prompts, odd lengths, fp16, grouped key/value heads.
        dict(name="padded_batch", kind="varlen", B=3, H=24, Hkv=8, Lq=3001, Lk=4099, D=128, dtype="fp16", smooth_v=False),
        # Causal attention over a ragged sequence with grouped key/value heads (streaming video, text encoders).
        dict(name="causal_ragged", kind="op", B=1, H=32, Hkv=8, Lq=8191, Lk=8191, D=128, dtype="bf16", outliers=0.0, causal=True),
        # The other head size the interface serves.
        dict(name="head_size_64", kind="op", B=2, H=16, Hkv=16, Lq=9001, Lk=9001, D=64, dtype="bf16", outliers=0.0, causal=False),
        # 720p video self-attention of the 5B model from its raw projections.
        dict(name="wan5b_720p_projections", kind="wan", B=1, H=24, frames=31, height=22, width=40, D=128, dtype="bf16"),
        # 480p, 81-frame video self-attention of the 14B model: the shape the path is quoted on, values with outliers.
        dict(name="wan14b_480p", kind="op", B=1, H=40, Hkv=40, Lq=32760, Lk=32760, D=128, dtype="bf16", outliers=1e-3, causal=False),
        # The same model at 720p: the longest sequence.
        dict(name="wan14b_720p", kind="op", B=1, H=40, Hkv=40, Lq=75600, Lk=75600, D=128, dtype="bf16", outliers=1e-3, causal=False),
        # The radial backend on a latent grid it accepts (21 frames of 64 x 112 latents).
        dict(name="radial_video", kind="radial", B=1, H=40, frames=21, latent_h=64, latent_w=112, D=128, dtype="bf16"),
        # The sparse-linear backend at the 480p shape, a tenth of the key blocks kept.
        dict(name="sparse_linear_480p", kind="sla", B=1, H=40, L=32760, D=128, dtype="bf16", topk=0.1),
    ]


def _log_int(rng, lo, hi):
    """An integer spread evenly over its logarithm; odd as often as even."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _heads(rng):
    hq = rng.choice((1, 8, 12, 16, 24, 32, 40, 64))
    return hq, hq // rng.choice([g for g in (1, 1, 1, 2, 4) if hq % g == 0])


def _shortened(case, keys, most):
    """The case with the sizes named in ``keys`` scaled down until its pairs of tokens cost at most ``most`` operations."""
    while _dense_flops(case) > most:
        for key in keys:
            case[key] = max(1, case[key] * 9 // 10)
    return case


def draw(rng):
    kind = rng.choice(("op", "op", "op", "cross", "wan", "qwen", "varlen", "radial", "sla"))
    dtype = rng.choice(("bf16", "bf16", "fp16"))
    if kind == "op":
        h, hkv = _heads(rng)
        length = _log_int(rng, 32, 75600)
        case = dict(kind=kind, B=rng.choice((1, 1, 2, 4)), H=h, Hkv=hkv, Lq=length, Lk=length, D=rng.choice((128, 128, 128, 64)),
                    dtype=dtype, outliers=rng.choice((0.0, 1e-3)), causal=rng.random() < 0.25)
        return _shortened(case, ("Lq", "Lk"), 8e13)
    if kind == "cross":
        h, hkv = _heads(rng)
        case = dict(kind=kind, B=rng.choice((1, 2)), H=h, Hkv=hkv, Lq=_log_int(rng, 1000, 75600), Lk=_log_int(rng, 77, 1024), D=128,
                    dtype=dtype, outliers=0.0, causal=False)
        return _shortened(case, ("Lq",), 2e13)
    if kind == "wan":
        frames, height, width = rng.randint(1, 31), rng.randint(12, 45), rng.randint(16, 80)
        case = dict(kind=kind, B=rng.choice((1, 1, 2)), H=rng.choice((12, 24, 40)), frames=frames, height=height, width=width, D=128,
                    dtype="bf16")
        return _shortened(case, ("frames",) if frames > 8 else ("frames", "height", "width"), 6e13)
    if kind == "qwen":
        return dict(kind=kind, B=rng.choice((1, 2)), H=24, txt=_log_int(rng, 13, 1024), img=_log_int(rng, 256, 16384), D=128, dtype="bf16")
    if kind == "varlen":
        h, hkv = _heads(rng)
        case = dict(kind=kind, B=rng.randint(2, 6), H=h, Hkv=hkv, Lq=_log_int(rng, 100, 16384), Lk=_log_int(rng, 100, 16384), D=128,
                    dtype=dtype, smooth_v=rng.random() < 0.25)
        return _shortened(case, ("Lq", "Lk"), 3e13)
    if kind == "radial":
        case = dict(kind=kind, B=1, H=rng.choice((12, 24, 40)), frames=rng.randint(3, 21), latent_h=16 * rng.randint(2, 5),
                    latent_w=16 * rng.randint(2, 7), D=128, dtype=dtype)
        return _shortened(case, ("frames",), 6e13)
    case = dict(kind=kind, B=rng.choice((1, 1, 2)), H=rng.choice((12, 24, 40)), L=_log_int(rng, 2000, 60000), D=128, dtype=dtype,
                topk=rng.choice((0.05, 0.1, 0.15, 0.25)))
    return _shortened(case, ("L",), 6e13)


def _lengths(case):
    if case["kind"] == "wan":
        n = case["frames"] * case["height"] * case["width"]
    elif case["kind"] == "qwen":
        n = case["txt"] + case["img"]
    elif case["kind"] == "radial":
        n = case["frames"] * (case["latent_h"] // 2) * (case["latent_w"] // 2)
    elif case["kind"] == "sla":
        n = case["L"]
    else:
        return case["Lq"], case["Lk"]
    return n, n


def _dense_flops(case):
    lq, lk = _lengths(case)
    return 4.0 * case["B"] * case["H"] * lq * lk * case["D"]


def _batch_lens(case):
    """Key and query counts of a padded batch: the first entry is full, the others fall off to about half."""
    B, lq, lk = case["B"], case["Lq"], case["Lk"]
    share = [1.0 - 0.55 * b / max(1, B - 1) for b in range(B)]
    return [max(1, int(lk * s)) for s in share], [max(1, int(lq * s)) for s in share]


def _values(g, shape, dtype, offset_std=0.0, outliers=0.0, text=0):
    """fp32 N(0, 1) rounded to ``dtype``; ``offset_std``: plus an offset per (head, channel), as keys have; ``outliers``:
    that share of the entries times 20; the first ``text`` tokens with a standard deviation of 3."""
    x = torch.randn(shape, generator=g, device=DEVICE, dtype=torch.float32)
    if text:
        x[:, :text] *= 3.0
    if offset_std:
        x += torch.randn(shape[2:], generator=g, device=DEVICE) * offset_std
    if outliers:
        x = torch.where(torch.rand(shape, generator=g, device=DEVICE) < outliers, x * 20.0, x)
    return x.to(dtype)


def _rope_table(rows, dim):
    f = torch.outer(torch.arange(rows, dtype=torch.float64), 1.0 / torch.pow(10000.0, torch.arange(0, dim, 2, dtype=torch.float64) / dim))
    return torch.polar(torch.ones_like(f), f)


def prepare(case, seed):
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    kind, B, H, D, dtype = case["kind"], case["B"], case["H"], case["D"], DTYPES[case["dtype"]]
    hkv = case.get("Hkv", H)
    lq, lk = _lengths(case)
    outliers, text = case.get("outliers", 0.0), case.get("txt", 0)
    state = {"kind": kind, "heads": H}
    state["q"] = _values(g, (B, lq, H, D), dtype, 0.0, outliers, text)
    state["k"] = _values(g, (B, lk, hkv, D), dtype, 2.0, outliers, text)
    state["v"] = _values(g, (B, lk, hkv, D), dtype, 0.0, 0.0, text)

    def weight(n):
        return 1.0 + 0.2 * torch.randn(n, generator=g, device=DEVICE)

    if kind in ("op", "cross"):
        config = KsanaAttentionConfig(backend=KsanaAttentionBackend.SAGE_ATTN)
        state["op"] = pick_attn_op(config)(num_heads=H, head_size=D, num_kv_heads=hkv, causal=case["causal"])
    elif kind == "wan":  # projections are [B, L, H * D]; the rotation table is the model's [1024, D / 2] buffer
        for name in "qkv":
            state[name] = state[name].flatten(2)
        freqs = torch.cat([_rope_table(1024, D - 4 * (D // 6)), _rope_table(1024, 2 * (D // 6)), _rope_table(1024, 2 * (D // 6))], dim=1)
        grid = [(case["frames"], case["height"], case["width"])] * B
        state["prep"] = WanPrep(weight(H * D), weight(H * D), 1e-6, freqs.to(DEVICE), grid)
    elif kind == "qwen":
        table = _rope_table(lq, D).to(torch.complex64).to(DEVICE)
        state["prep"] = QwenPrep(text, weight(D), weight(D), weight(D), weight(D), 1e-6,
                                 img_freqs=table[: lq - text].contiguous(), txt_freqs=table[lq - text :].contiguous())
    elif kind == "varlen":
        k_lens, q_lens = _batch_lens(case)
        state["k_lens"] = torch.tensor(k_lens, dtype=torch.int32, device=DEVICE)
        state["q_lens"] = torch.tensor(q_lens, dtype=torch.int32, device=DEVICE)
        state["smooth_v"] = case["smooth_v"]
    elif kind == "radial":
        state["op"] = pick_attn_op(KsanaRadialSageAttentionConfig())(num_heads=H, head_size=D, causal=False)
        state["kwargs"] = dict(k_lens=torch.tensor([lk] * B, device=DEVICE), step_iter=9, block_id=7,
                               latent_shape=[B, 16, case["frames"], case["latent_h"], case["latent_w"]])
    else:
        state["op"] = pick_attn_op(KsanaSageSLAConfig(topk=case["topk"]))(num_heads=H, head_size=D, causal=False)
        proj = torch.nn.Linear(D, D, bias=True, device=DEVICE)
        with torch.no_grad():
            proj.weight.copy_(torch.randn(D, D, generator=g, device=DEVICE) * 0.05)
            proj.bias.copy_(torch.randn(D, generator=g, device=DEVICE) * 0.05)
        state["proj"] = proj.to(dtype).requires_grad_(False)
    return state


def run(state):
    kind, q, k, v = state["kind"], state["q"], state["k"], state["v"]
    if kind in ("op", "cross"):
        return state["op"](q, k, v)
    if kind == "wan":
        return wan_self_attention(q, k, v, state["heads"], state["prep"])
    if kind == "qwen":
        return sageattn(q, k, v, prep=state["prep"])
    if kind == "varlen":
        return sageattn(q, k, v, k_lens=state["k_lens"], q_lens=state["q_lens"], smooth_v=state["smooth_v"])
    if kind == "radial":
        return state["op"](q, k, v, **state["kwargs"])
    return state["op"](q, k, v, proj_l=state["proj"])


def _radial_pairs(case):
    """Token pairs of the radial pattern: every query sees the first frame, its own frame, and a band that narrows with
    the distance in frames (never under one block of 128), at frame distances that thin out once the band is that narrow."""
    n, frames, block, decay = (case["latent_h"] // 2) * (case["latent_w"] // 2), case["frames"], 128, 0.02
    total = 0
    for i in range(frames):
        for j in range(frames):
            dist = abs(i - j)
            if j == 0 or dist == 0:
                total += n * n
                continue
            reach = 2 ** n.bit_length() / 2 ** dist.bit_length()
            if reach < block and dist % int(block / reach):
                continue
            width = min(n, n // 2 if dist == 1 else max(reach * decay, block))
            total += n * n - (n - width) ** 2
    return total


def work(case):
    """Operations: a multiply-add counts as 2; QK^T and PV over the token pairs that take part.  Bytes: q, k, v read once
    and the result written once."""
    B, H, D = case["B"], case["H"], case["D"]
    hkv = case.get("Hkv", H)
    lq, lk = _lengths(case)
    nbytes = 2.0 * D * B * (2 * lq * H + 2 * lk * hkv)
    flops = _dense_flops(case)
    if case.get("causal"):
        flops *= (lq + 1) / (2.0 * lq)
    elif case["kind"] == "varlen":
        k_lens, q_lens = _batch_lens(case)
        flops = 4.0 * H * D * sum(a * b for a, b in zip(k_lens, q_lens))
        nbytes = 2.0 * D * (B * lq * H + sum(q_lens) * H + 2 * sum(k_lens) * hkv)
    elif case["kind"] == "radial":
        flops = 4.0 * B * H * D * _radial_pairs(case)
    elif case["kind"] == "sla":
        blocks = -(-lk // 64)
        keep = min(blocks, int(case["topk"] * blocks))
        # the kept blocks, the scores of the pooled blocks, sum(phi(k)^T v), phi(q) times it and its row sum
        flops = flops * keep / blocks + 2.0 * B * H * -(-lq // 128) * blocks * D + 4.0 * B * H * lq * D * D + 4.0 * B * H * lq * D
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Probabilities and values are multiplied as e4m3 (three mantissa bits): one rounding to it is 2.6 % (root mean
    square) of what is rounded, and over zero-mean values that share of the rounding reaches the result.  Two correct
    implementations round the probabilities against reference points of their own."""
    return {"rel": 0.03, "max": 0.5}
