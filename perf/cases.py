"""Performance cases of the LTX-2.5 audio-video DiT path: what a denoising program has this framework do.

Each case is one call (or one short sequence of calls) that a program makes through the public entry points of
ltxk / ltx_nn / ltx_dit / ltx_te / torch_rng, at the widths of the 48-block checkpoint configuration: video stream 4096
wide (32 heads of 128), audio stream 2048 wide (32 heads of 64), FFN 4x, text context 1024 tokens, latents 128 channels.
121 frames at 512x768 make a 16x16x24 latent grid (6144 video tokens) and 126 audio tokens; 97 frames at 704x480 make
13x22x15 = 4290 video tokens and 101 audio tokens at 24 frames a second.  The guidance batch is four passes.

The cases are mostly the model's single layers, each with its own tolerance; `model` is a whole LTXModel call (velocities
of both streams) and `text_encoder` a whole EmbeddingsProcessor call.
"""
import math
import pathlib
import sys
import zlib

import numpy as np
import torch

sys.path.insert(0, str(pathlib.Path(__file__).resolve().parents[1] / "ltx-nv_amd"))

DEV = "cuda"
EPS = 1e-6
BF16 = torch.bfloat16
VIDEO, AUDIO = 4096, 2048
HEADS = 32
VIDEO_MAX_POS, TIME_MAX_POS = [20, 2048, 2048], [20]


def listed():
    return [
        # One latent's noise and one Euler update in fp32 (121 frames at 512x768): the smallest call, launch-bound.
        dict(name="noise_euler_fp32", kind="noise", batch=1, tokens=6144, dtype="float32"),
        # The norm + AdaLN modulation in front of the first video self-attention of a step.
        dict(name="norm_video", kind="norm", batch=1, tokens=6144, dim=VIDEO, residual=False, two=False, indexed=False),
        # Text-attention residual + the two A2V/V2A modulations of the same row, on a ragged video length.
        dict(name="residual_norm_ragged", kind="norm", batch=1, tokens=4290, dim=VIDEO, residual=True, two=True,
             indexed=False),
        # Video self-attention of one block: the largest layer of a step.
        dict(name="self_attn_video", kind="self", stream="video", batch=1, frames=16, height=16, width=24),
        # Audio self-attention of one block: few tokens, latency counts.
        dict(name="self_attn_audio", kind="self", stream="audio", batch=1, audio=126),
        # Video to text cross-attention, ragged video length.
        dict(name="text_attn_video", kind="text", stream="video", batch=1, tokens=4290, text=1024),
        # Audio to video attention: many queries over few keys.
        dict(name="a2v_attn", kind="a2v", batch=1, frames=16, height=16, width=24, audio=126),
        # Video to audio attention in the guidance batch: few queries over many keys.
        dict(name="v2a_attn_b4", kind="v2a", batch=4, frames=16, height=16, width=24, audio=126),
        # The video feed-forward of one block.
        dict(name="ffn_video", kind="ffn", batch=1, tokens=6144, dim=VIDEO, bias=False),
        # The tail of a guided step: x0 of four passes, guidance with rescale, Euler.
        dict(name="guide_video", kind="guide", tokens=6144),
        # Prompt features of 1024 tokens (49 hidden states) through the projections and both connectors.
        dict(name="text_encoder", kind="te", tokens=1024, kept=724, layers=49, blocks=2),
        # One transformer call of the guided loop (cond, uncond, STG-perturbed, modality-isolated), two blocks deep.
        dict(name="model_b4", kind="model", batch=4, frames=16, height=16, width=24, audio=126, text=1024, blocks=2),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, most):
    while True:
        f, h, w = rng.randint(2, 16), rng.randint(4, 24), rng.randint(4, 30)
        if 64 <= f * h * w <= most:
            return dict(frames=f, height=h, width=w)


def draw(rng):
    kind = rng.choice(["noise", "norm", "self", "self", "text", "a2v", "v2a", "ffn", "guide", "te", "model"])
    if kind == "noise":
        return dict(kind=kind, batch=rng.choice([1, 2, 4]), tokens=_log_int(rng, 100, 8192),
                    dtype=rng.choice(["float32", "bfloat16"]))
    if kind == "norm":
        return dict(kind=kind, batch=rng.choice([1, 2, 4]), tokens=_log_int(rng, 32, 6144), dim=rng.choice([VIDEO, AUDIO]),
                    residual=rng.random() < 0.7, two=rng.random() < 0.4, indexed=rng.random() < 0.25)
    if kind == "self":
        b = rng.choice([1, 1, 2, 4])
        if rng.random() < 0.3:
            return dict(kind=kind, stream="audio", batch=b, audio=_log_int(rng, 16, 512))
        return dict(kind=kind, stream="video", batch=b, **_grid(rng, 6144 if b == 1 else 3072))
    if kind == "text":
        return dict(kind=kind, stream=rng.choice(["video", "video", "audio"]), batch=rng.choice([1, 2, 4]),
                    tokens=_log_int(rng, 64, 6144), text=_log_int(rng, 64, 1024))
    if kind in ("a2v", "v2a"):
        return dict(kind=kind, batch=rng.choice([1, 4]), **_grid(rng, 6144), audio=_log_int(rng, 16, 256))
    if kind == "ffn":
        dim = rng.choice([VIDEO, VIDEO, AUDIO])
        return dict(kind=kind, batch=rng.choice([1, 2]), tokens=_log_int(rng, 32, 6144), dim=dim, bias=dim == AUDIO)
    if kind == "guide":
        return dict(kind=kind, tokens=_log_int(rng, 32, 8192))
    if kind == "te":
        s = 128 * rng.randint(1, 8)
        return dict(kind=kind, tokens=s, kept=rng.randint(s // 8, s), layers=49, blocks=rng.randint(1, 2))
    return dict(kind="model", batch=rng.choice([1, 4]), **_grid(rng, 3072), audio=_log_int(rng, 16, 160),
                text=_log_int(rng, 64, 1024), blocks=rng.randint(1, 2))


# --------------------------------------------------------------------------------------------------------------------
# Inputs, from the seed and a name alone
# --------------------------------------------------------------------------------------------------------------------


def _rand(seed, name, shape, std=1.0, mean=0.0, dtype=BF16):
    g = torch.Generator(device=DEV).manual_seed((seed * 1000003 + zlib.crc32(name.encode())) % (2**62))
    return torch.randn(*shape, device=DEV, generator=g).mul_(std).add_(mean).to(dtype)


def _param(seed, name, shape):
    """A weight by its name: projections and biases N(0, 0.02^2), modulation tables N(0, 0.2^2), and q/k norm weights
    near 1.5, so that attention scores spread as a trained model's do (std about 2) instead of nearly uniform."""
    if name.endswith(("q_norm.weight", "k_norm.weight")):
        return _rand(seed, name, shape, 0.1, 1.5)
    if "scale_shift_table" in name:
        return _rand(seed, name, shape, 0.2)
    if "learnable_registers" in name:
        return _rand(seed, name, shape, 1.0)
    return _rand(seed, name, shape, 0.02)


def _module(make, seed, prefix=""):
    """The module with its parameters on the GPU in bf16, drawn by name."""
    with torch.device("meta"):
        m = make()
    m = m.to(BF16).to_empty(device=DEV).eval().requires_grad_(False)
    for name, p in m.named_parameters():
        p.copy_(_param(seed, prefix + name, p.shape))
    return m


def _dims(case):
    return case["frames"], case["height"], case["width"]


def _tokens(case):
    """Video tokens of a latent grid (the audio stream's, where a case has no grid)."""
    return math.prod(_dims(case)) if "frames" in case else case["audio"]


def _video_positions(batch, grid):
    """Pixel-space [start, end) bounds of every latent token, time in seconds at 24 frames a second."""
    idx = torch.stack(torch.meshgrid(*[torch.arange(n, device=DEV) for n in grid], indexing="ij")).reshape(3, -1).float()
    bounds = torch.stack([idx, idx + 1], -1) * torch.tensor([8.0, 32.0, 32.0], device=DEV).view(3, 1, 1)
    bounds[0] = (bounds[0] - 7).clamp(min=0) / 24.0
    return bounds.unsqueeze(0).expand(batch, -1, -1, -1).contiguous()


def _audio_positions(batch, n):
    i = torch.arange(n, dtype=torch.float32, device=DEV)
    return torch.stack([(i * 4 - 3).clamp(min=0) * 160 / 16000, (i * 4 + 1) * 160 / 16000], -1)[None, None] \
        .expand(batch, 1, -1, -1).contiguous()


def _stream_dims(stream):
    return (VIDEO, HEADS, VIDEO // HEADS) if stream == "video" else (AUDIO, HEADS, AUDIO // HEADS)


def _positions(case, stream):
    if stream == "video":
        return _video_positions(case["batch"], _dims(case)), VIDEO_MAX_POS
    return _audio_positions(case["batch"], case["audio"]), TIME_MAX_POS


def _indexed_rows(case):
    """A keyframe-conditioned step has two timestep rows: the first tenth of the tokens carries the conditioning one."""
    b, t = case["batch"], case["tokens"]
    first = torch.arange(b * t, device=DEV) % t < max(1, t // 10)
    return torch.where(first, 0, 1).to(torch.int32)


def _guide_inputs(case, seed):
    t = case["tokens"]
    latent = _rand(seed, "latent", (1, t, 128))
    base = _rand(seed, "velocity", (1, t, 128), dtype=torch.float32)
    vel = (base + 0.2 * _rand(seed, "spread", (4, t, 128), dtype=torch.float32)).to(BF16)
    return latent, vel, torch.full((4, t, 1), 0.725, device=DEV)


GUIDE = dict(cfg_scale=3.0, stg_scale=1.0, modality_scale=3.0, rescale_scale=0.7)
SIGMA, DT = 0.725, -0.03125


def _model_inputs(case, seed):
    b, tv, ta, s = case["batch"], _tokens(case), case["audio"], case["text"]
    n = case["blocks"]
    # the passes of a guided step share the latent; the unconditional pass has the negative prompt's context
    x = {k: _rand(seed, k + "_latent", (1, t, 128)).repeat(b, 1, 1) for k, t in (("video", tv), ("audio", ta))}
    ctx = {}
    for k, d in (("video", VIDEO), ("audio", AUDIO)):
        pos, neg = (_rand(seed, k + which, (1, s, d)) for which in ("_pos", "_neg"))
        ctx[k] = torch.cat([neg if i == 1 else pos for i in range(b)])
    keep = torch.ones(4, n, b)
    if b == 4:
        keep[0:2, n - 1, 2] = 0   # the STG-perturbed pass skips self-attention in the last block
        keep[2:4, :, 3] = 0       # the modality-isolated pass skips A2V and V2A
    kf = torch.zeros(b, tv, 1, device=DEV)
    kf[:, :case["height"] * case["width"]] = 1.0
    return x, ctx, keep, kf


# --------------------------------------------------------------------------------------------------------------------
# prepare / run
# --------------------------------------------------------------------------------------------------------------------


@torch.no_grad()
def prepare(case, seed):
    import ltx_dit
    import ltx_nn
    import ltx_te
    import ltxk

    kind = case["kind"]
    b = case.get("batch", 1)
    s = {"case": case, "seed": seed}
    if kind == "noise":
        s["shape"] = (b, case["tokens"], 128)
        s["v"] = _rand(seed, "v", s["shape"], dtype=getattr(torch, case["dtype"]))
    elif kind == "norm":
        d, t = case["dim"], case["tokens"]
        s["x"] = _rand(seed, "x", (b, t, d))
        s["f"] = _rand(seed, "f", (b, t, d)) if case["residual"] else None
        s["table"] = _rand(seed, "table", (9, d), 0.2)
        s["emb"] = _rand(seed, "emb", (1, 2, 9 * d) if case["indexed"] else (b, 1, 9 * d), 0.1)
        s["index"] = ltxk.TimestepIndex(_indexed_rows(case), 2) if case["indexed"] else None
    elif kind == "self":
        dim, h, dh = _stream_dims(case["stream"])
        pos, max_pos = _positions(case, case["stream"])
        s["attn"] = _module(lambda: ltx_nn.Attention(dim, None, h, dh, EPS, True), seed)
        s["x"] = _rand(seed, "x", (b, pos.shape[2], dim))
        s["pe"] = ltx_nn.precompute_freqs_cis_compact(pos, dim, max_pos=max_pos, num_attention_heads=h)
    elif kind == "text":
        dim, h, dh = _stream_dims(case["stream"])
        s["attn"] = _module(lambda: ltx_nn.Attention(dim, dim, h, dh, EPS, True), seed)
        s["x"] = _rand(seed, "x", (b, case["tokens"], dim))
        s["context"] = _rand(seed, "context", (b, case["text"], dim))
    elif kind in ("a2v", "v2a"):
        qd, cd = (VIDEO, AUDIO) if kind == "a2v" else (AUDIO, VIDEO)
        s["attn"] = _module(lambda: ltx_nn.Attention(qd, cd, HEADS, AUDIO // HEADS, EPS, True), seed)
        vpos, apos = _video_positions(b, _dims(case))[:, 0:1], _audio_positions(b, case["audio"])
        vpe, ape = (ltx_nn.precompute_freqs_cis_compact(p, AUDIO, max_pos=TIME_MAX_POS, num_attention_heads=HEADS)
                    for p in (vpos, apos))
        video, audio = _rand(seed, "video", (b, _tokens(case), VIDEO)), _rand(seed, "audio", (b, case["audio"], AUDIO))
        s["x"], s["context"], s["pe"], s["k_pe"] = (video, audio, vpe, ape) if kind == "a2v" else (audio, video, ape, vpe)
    elif kind == "ffn":
        s["ffn"] = _module(lambda: ltx_nn.FeedForward(case["dim"], case["dim"], bias=case["bias"]), seed)
        s["x"] = _rand(seed, "x", (b, case["tokens"], case["dim"]))
    elif kind == "guide":
        s["latent"], s["velocity"], s["timesteps"] = _guide_inputs(case, seed)
    elif kind == "te":
        t = case["tokens"]
        s["hidden"] = tuple(_rand(seed, "hidden%d" % i, (1, t, 3840), 1.0 + 0.1 * i) for i in range(case["layers"]))
        s["mask"] = (torch.arange(t, device=DEV) >= t - case["kept"]).long().view(1, t)
        s["proc"] = _module(lambda: ltx_te.EmbeddingsProcessor(
            ltx_te.FeatureExtractorV2(3840, case["layers"] - 1, VIDEO, AUDIO),
            ltx_te.Embeddings1DConnector(HEADS, 128, case["blocks"], [4096], 128, False, True),
            ltx_te.Embeddings1DConnector(HEADS, 64, case["blocks"], [4096], 128, False, True)), seed)
    else:
        cfg = ltx_dit.DiTConfig(num_layers=case["blocks"])
        m = _module(lambda: ltx_dit.LTXModel(cfg), seed)
        x, ctx, keep, kf = _model_inputs(case, seed)
        sig = torch.full((b,), SIGMA, device=DEV)
        mods = {}
        for k, pre, pos in (("video", m.video_pre, _video_positions(b, _dims(case))),
                            ("audio", m.audio_pre, _audio_positions(b, case["audio"]))):
            ts = torch.full((b, x[k].shape[1], 1), SIGMA, device=DEV)
            # a denoising loop analyses its masks and positions once and hands the derived forms in
            mods[k] = ltx_dit.Modality(latent=x[k], sigma=sig, timesteps=ts, positions=pos, context=ctx[k],
                                       keyframes_mask=kf if k == "video" else None,
                                       timestep_rows=ltx_dit.timestep_rows(ts), rope_tables=pre.rope_tables(pos))
        s["model"], s["video"], s["audio"] = m, mods["video"], mods["audio"]
        s["keep"] = ltx_dit.PerturbationTable.of(keep.to(DEV, BF16)) if b == 4 else None
    return s


def run(state):
    import ltxk
    import torch_rng

    case = state["case"]
    kind = case["kind"]
    with torch.inference_mode():
        if kind == "noise":
            x = torch_rng.TorchRNG(state["seed"], DEV).randn(*state["shape"], dtype=state["v"].dtype)
            return ltxk.euler_update(x, state["v"], -0.125)
        if kind == "norm":
            def ada(row):
                return ltxk.AdaRef(state["table"], row, state["emb"], index=state["index"])

            more = dict(shift2=ada(3), scale2=ada(4)) if case["two"] else {}
            if case["residual"]:
                return ltxk.add_norm_modulate(state["x"], state["f"], gate=ada(2), shift=ada(0), scale=ada(1), eps=EPS,
                                              **more)
            return ltxk.norm_modulate(state["x"], shift=ada(0), scale=ada(1), eps=EPS, **more)
        if kind == "self":
            return state["attn"](state["x"], pe=state["pe"])
        if kind == "text":
            return state["attn"](state["x"], context=state["context"])
        if kind in ("a2v", "v2a"):
            return state["attn"](state["x"], context=state["context"], pe=state["pe"], k_pe=state["k_pe"])
        if kind == "ffn":
            return state["ffn"](state["x"])
        if kind == "guide":
            den, nxt, _ = ltxk.guide(state["latent"], state["velocity"], state["timesteps"], **GUIDE, sigma=SIGMA, dt=DT)
            return den, nxt
        if kind == "te":
            video, audio, _ = state["proc"].process_hidden_states(state["hidden"], state["mask"])
            return video, audio
        return state["model"](state["video"], state["audio"], state["keep"])


# --------------------------------------------------------------------------------------------------------------------
# work / tolerance
# --------------------------------------------------------------------------------------------------------------------


def _attn_work(b, tq, tk, qd, cd, inner, rope=True):
    flops = 2.0 * b * (tq * qd * inner * 2 + 2 * tk * cd * inner + tq * qd * HEADS) + 4.0 * b * tq * tk * inner
    same = tq == tk and qd == cd and rope
    data = 2.0 * (b * tq * qd * 2 + (0 if same else b * tk * cd) + 2 * inner * (qd + cd))
    return data, flops


def work(case):
    kind, b = case["kind"], case.get("batch", 1)
    if kind == "noise":
        n = b * case["tokens"] * 128
        return {"bytes": 2.0 * n * (4 if case["dtype"] == "float32" else 2), "flops": 40.0 * n}
    if kind == "norm":
        n = b * case["tokens"] * case["dim"]
        tensors = 2 + (2 if case["residual"] else 0) + (1 if case["two"] else 0)
        return {"bytes": 2.0 * n * tensors, "flops": 8.0 * n}
    if kind == "self":
        dim, _, _ = _stream_dims(case["stream"])
        t = _tokens(case)
        data, flops = _attn_work(b, t, t, dim, dim, dim)
    elif kind == "text":
        dim, _, _ = _stream_dims(case["stream"])
        data, flops = _attn_work(b, case["tokens"], case["text"], dim, dim, dim, rope=False)
    elif kind == "a2v":
        data, flops = _attn_work(b, _tokens(case), case["audio"], VIDEO, AUDIO, AUDIO)
    elif kind == "v2a":
        data, flops = _attn_work(b, case["audio"], _tokens(case), AUDIO, VIDEO, AUDIO)
    elif kind == "ffn":
        d, t = case["dim"], b * case["tokens"]
        data, flops = 2.0 * (2 * t * d + 8 * d * d), 16.0 * t * d * d
    elif kind == "guide":
        data, flops = 2.0 * case["tokens"] * 128 * 7, 40.0 * case["tokens"] * 128
    elif kind == "te":
        t, k = case["tokens"], 3840 * case["layers"]
        data = 2.0 * (t * k + k * (VIDEO + AUDIO) + t * (VIDEO + AUDIO))
        flops = 2.0 * t * k * (VIDEO + AUDIO)
        for d in (VIDEO, AUDIO):
            data += case["blocks"] * 2.0 * 12 * d * d
            flops += case["blocks"] * (24.0 * t * d * d + 4.0 * t * t * d)
    else:
        tv, ta, s = _tokens(case), case["audio"], case["text"]
        data = flops = 0.0
        for qt, kt, qd, cd, inner, rope in ((tv, tv, VIDEO, VIDEO, VIDEO, True), (tv, s, VIDEO, VIDEO, VIDEO, False),
                                            (ta, ta, AUDIO, AUDIO, AUDIO, True), (ta, s, AUDIO, AUDIO, AUDIO, False),
                                            (tv, ta, VIDEO, AUDIO, AUDIO, True), (ta, tv, AUDIO, VIDEO, AUDIO, True)):
            flops += case["blocks"] * _attn_work(b, qt, kt, qd, cd, inner, rope)[1]
            data += case["blocks"] * 4.0 * inner * (qd + cd)
        for t, d in ((tv, VIDEO), (ta, AUDIO)):
            flops += case["blocks"] * 16.0 * b * t * d * d
            data += case["blocks"] * 16.0 * d * d + 2.0 * b * (256 * t + s * d)
    return {"bytes": data, "flops": flops}


def tolerance(case):
    kind = case["kind"]
    if kind == "noise":
        # one fp32 ulp of the normal's formula, or (bf16) a rounding that falls the other way
        return {"rel": 1e-6} if case["dtype"] == "float32" else {"rel": 1e-3}
    # four times the measured distance of the bf16 results from the 64-bit ones: norm 0.0024, guide 0.009, ffn 0.003,
    # te 0.0056, model 0.0095, an attention layer 0.0069 to 0.0093
    return {"rel": {"norm": 1e-2, "guide": 3.6e-2, "ffn": 1.2e-2, "te": 2.3e-2, "model": 4e-2}.get(kind, 3.6e-2)}


# --------------------------------------------------------------------------------------------------------------------
# exact: the same results in 64 bits from plain torch
# --------------------------------------------------------------------------------------------------------------------


def _lin64(p, name, x):
    y = x @ p(name + ".weight").T
    bias = p(name + ".bias")
    return y if bias is None else y + bias


class _Params:
    """Weights by name in 64 bits; shapes come from `shapes` (name -> shape), a missing name is None."""

    def __init__(self, seed, shapes, prefix=""):
        self.seed, self.shapes, self.prefix = seed, shapes, prefix

    def __call__(self, name):
        shape = self.shapes.get(self.prefix + name)
        return None if shape is None else _param(self.seed, self.prefix + name, shape).double()

    def at(self, prefix):
        return _Params(self.seed, self.shapes, self.prefix + prefix)


def _attn_shapes(pre, qd, cd, inner, gated=True):
    s = {}
    for n, o, i in (("to_q", inner, qd), ("to_k", inner, cd), ("to_v", inner, cd), ("to_out", qd, inner)):
        s[pre + n + ".weight"], s[pre + n + ".bias"] = (o, i), (o,)
    if gated:
        s[pre + "to_gate_logits.weight"], s[pre + "to_gate_logits.bias"] = (HEADS, qd), (HEADS,)
    s[pre + "q_norm.weight"] = s[pre + "k_norm.weight"] = (inner,)
    return s


def _ffn_shapes(pre, d, bias):
    s = {pre + "proj_in.weight": (4 * d, d), pre + "proj_out.weight": (d, 4 * d)}
    if bias:
        s[pre + "proj_in.bias"], s[pre + "proj_out.bias"] = (4 * d,), (d,)
    return s


def _rms64(x, w=None):
    y = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS)
    return y if w is None else y * w


def _tables64(pos, dim, max_pos):
    """cos, sin (B, T, dim/2) of split rotation: positions (B, A, T, 2) bounds or (B, A, T); axis fastest, front padding."""
    mid = pos.double().mean(-1) if pos.ndim == 4 else pos.double()
    n_axes = mid.shape[1]
    count = dim // (2 * n_axes)
    # the frequencies are defined in fp32 (rounded from fp64), as are the positions' fractions
    freq = torch.from_numpy(np.power(10000.0, np.linspace(0.0, 1.0, count)) * math.pi / 2).float().double().to(DEV)
    frac = torch.stack([mid[:, a] / max_pos[a] for a in range(n_axes)], -1)
    ang = (freq * (frac.unsqueeze(-1) * 2 - 1)).transpose(-1, -2).flatten(2)
    ang = torch.nn.functional.pad(ang, (dim // 2 - ang.shape[-1], 0))
    return ang.cos(), ang.sin()


def _rope64(x, tables):
    if tables is None:
        return x
    b, t, d = x.shape
    c, s = (v.view(v.shape[0], t, HEADS, -1) for v in tables)
    x1, x2 = x.view(b, t, HEADS, 2, -1).unbind(3)
    return torch.stack([x1 * c - x2 * s, x2 * c + x1 * s], 3).reshape(b, t, d)


def _attn64(p, x, ctx=None, pe=None, k_pe=None, keep=None):
    ctx = x if ctx is None else ctx
    v = _lin64(p, "to_v", ctx)
    q = _rope64(_rms64(_lin64(p, "to_q", x), p("q_norm.weight")), pe)
    k = _rope64(_rms64(_lin64(p, "to_k", ctx), p("k_norm.weight")), k_pe if k_pe is not None else pe)
    b, t, inner = q.shape
    dh = inner // HEADS
    out = torch.empty_like(q)
    for i in range(b):
        for h in range(HEADS):
            j = slice(h * dh, (h + 1) * dh)
            for r in range(0, t, 4096):
                rows = slice(r, r + 4096)
                out[i, rows, j] = torch.softmax(q[i, rows, j] @ k[i, :, j].T / math.sqrt(dh), -1) @ v[i, :, j]
    if keep is not None:
        out = out * keep + v * (1 - keep)
    if p("to_gate_logits.weight") is not None:
        out = (out.view(b, t, HEADS, dh) * (2 * torch.sigmoid(_lin64(p, "to_gate_logits", x))).unsqueeze(-1)).flatten(2)
    return _lin64(p, "to_out", out)


def _ffn64(p, x):
    return _lin64(p, "proj_out", torch.nn.functional.gelu(_lin64(p, "proj_in", x), approximate="tanh"))


def _noise64(n, seed):
    """Philox4x32-10 normals in torch's grid-stride layout on this device, in 64 bits from the fp32 (u, v) pair."""
    props = torch.cuda.get_device_properties(0)
    threads = 256 * min(-(-n // 256), props.multi_processor_count * (props.max_threads_per_multi_processor // 256))
    m32 = 0xFFFFFFFF
    rounds = -(-n // (4 * threads))
    it = torch.arange(rounds, device=DEV).view(-1, 1).expand(rounds, threads).reshape(-1)
    tid = torch.arange(threads, device=DEV).view(1, -1).expand(rounds, threads).reshape(-1)
    c = [it & m32, it >> 32, tid & m32, tid >> 32]
    k0, k1 = seed & m32, (seed >> 32) & m32
    for r in range(10):
        if r:
            k0, k1 = (k0 + 0x9E3779B9) & m32, (k1 + 0xBB67AE85) & m32
        p0, p1 = c[0] * 0xD2511F53, c[2] * 0xCD9E8D57
        c = [((p1 >> 32) & m32) ^ c[1] ^ k0, p1 & m32, ((p0 >> 32) & m32) ^ c[3] ^ k1, p0 & m32]
    lanes = []
    for x, y in ((c[0], c[1]), (c[2], c[3])):
        u = (x.float() * 2.3283064e-10 + 2.3283064e-10).double()
        v = (y.float() * 1.46291807e-09 + 1.46291807e-09).double()
        amp = torch.sqrt(-2 * torch.log(u))
        lanes += [amp * torch.sin(v), amp * torch.cos(v)]
    return torch.stack(lanes).view(4, rounds, threads).transpose(0, 1).reshape(-1)[:n]


def _norm64(case, seed):
    b, t, d = case["batch"], case["tokens"], case["dim"]
    x = _rand(seed, "x", (b, t, d)).double()
    table = _rand(seed, "table", (9, d), 0.2).double()
    emb = _rand(seed, "emb", (1, 2, 9 * d) if case["indexed"] else (b, 1, 9 * d), 0.1).double()
    if case["indexed"]:
        emb = emb[0][_indexed_rows(case).long()].view(b, t, 9 * d)

    def ada(row):
        return table[row] + emb[..., row * d:(row + 1) * d]

    out = []
    if case["residual"]:
        x = x + _rand(seed, "f", (b, t, d)).double() * ada(2)
        out.append(x)
    y = _rms64(x)
    out.append(y * (1 + ada(1)) + ada(0))
    if case["two"]:
        out.append(y * (1 + ada(4)) + ada(3))
    return out[0] if len(out) == 1 else tuple(out)


def _guide64(case, seed):
    latent, vel, ts = (t.double() for t in _guide_inputs(case, seed))
    c, u, p, m = (latent - vel * ts).unbind(0)
    pred = c + 2.0 * (c - u) + 1.0 * (c - p) + 2.0 * (c - m)
    pred = pred * (0.7 * c.std() / pred.std() + 0.3)
    return pred.unsqueeze(0), latent + (latent - pred) / SIGMA * DT


def _te64(case, seed):
    t, n = case["tokens"], case["layers"]
    shapes = {}
    for k, d in (("video", VIDEO), ("audio", AUDIO)):
        shapes["feature_extractor.%s_aggregate_embed.weight" % k] = (d, 3840 * n)
        shapes["feature_extractor.%s_aggregate_embed.bias" % k] = (d,)
        shapes["%s_connector.learnable_registers" % k] = (128, d)
        for i in range(case["blocks"]):
            shapes.update(_attn_shapes("%s_connector.blocks.%d.attn1." % (k, i), d, d, d, gated=False))
            shapes.update(_ffn_shapes("%s_connector.blocks.%d.ff." % (k, i), d, True))
    p = _Params(seed, shapes)
    hid = torch.stack([_rms64(_rand(seed, "hidden%d" % i, (t, 3840), 1.0 + 0.1 * i).double()) for i in range(n)], -1)
    feat = hid.flatten(1)[t - case["kept"]:]
    out = []
    for k, d in (("video", VIDEO), ("audio", AUDIO)):
        regs = p("%s_connector.learnable_registers" % k)
        x = regs[torch.arange(t, device=DEV) % 128].clone()
        x[:case["kept"]] = _lin64(p, "feature_extractor.%s_aggregate_embed" % k, feat * math.sqrt(d / 3840))
        x = x.unsqueeze(0)
        pe = _tables64(torch.arange(t, device=DEV).view(1, 1, t), d, [4096])
        for i in range(case["blocks"]):
            q = p.at("%s_connector.blocks.%d." % (k, i))
            x = x + _attn64(q.at("attn1."), _rms64(x), pe=pe)
            x = x + _ffn64(q.at("ff."), _rms64(x))
        out.append(_rms64(x))
    return tuple(out)


def _adaln64(p, t):
    freq = torch.exp(-math.log(10000) * torch.arange(128, dtype=torch.float64, device=DEV) / 128)
    a = t.double()[:, None] * freq
    silu = torch.nn.functional.silu
    h = silu(_lin64(p, "emb.timestep_embedder.linear_1", torch.cat([a.cos(), a.sin()], -1)))
    emb = _lin64(p, "emb.timestep_embedder.linear_2", h)
    return _lin64(p, "linear", silu(emb)), emb


def _model_shapes(blocks):
    s = {}

    def lin(name, o, i):
        s[name + ".weight"], s[name + ".bias"] = (o, i), (o,)

    def adaln(name, d, n):
        lin(name + ".emb.timestep_embedder.linear_1", d, 256)
        lin(name + ".emb.timestep_embedder.linear_2", d, d)
        lin(name + ".linear", n * d, d)

    s["keyframes_abs_pos_embedding"] = (1, VIDEO)
    for pre, k, d, gate in (("", "video", VIDEO, "a2v"), ("audio_", "audio", AUDIO, "v2a")):
        lin(pre + "patchify_proj", d, 128)
        lin(pre + "proj_out", 128, d)
        s[pre + "scale_shift_table"] = (2, d)
        adaln(pre + "adaln_single", d, 9)
        adaln(pre + "prompt_adaln_single", d, 2)
        adaln("av_ca_%s_scale_shift_adaln_single" % k, d, 4)
        adaln("av_ca_%s_gate_adaln_single" % gate, d, 1)
    for i in range(blocks):
        b = "blocks.%d." % i
        for pre, d, k in (("", VIDEO, "video"), ("audio_", AUDIO, "audio")):
            s.update(_attn_shapes(b + pre + "attn1.", d, d, d))
            s.update(_attn_shapes(b + pre + "attn2.", d, d, d))
            s.update(_ffn_shapes(b + pre + "ff.", d, d == AUDIO))
            s[b + pre + "scale_shift_table"] = (9, d)
            s[b + pre + "prompt_scale_shift_table"] = (2, d)
            s[b + "scale_shift_table_a2v_ca_" + k] = (5, d)
        s.update(_attn_shapes(b + "audio_to_video_attn.", VIDEO, AUDIO, AUDIO))
        s.update(_attn_shapes(b + "video_to_audio_attn.", AUDIO, VIDEO, AUDIO))
    return s


def _model64(case, seed):
    b, n = case["batch"], case["blocks"]
    p = _Params(seed, _model_shapes(n))
    lat, ctx, keep, kf = _model_inputs(case, seed)
    keep = keep.to(DEV).double()
    t = torch.full((1,), SIGMA * 1000.0, device=DEV)
    st = {}
    for pre, k, d, gate, pos, mp in (("", "video", VIDEO, "a2v", _video_positions(b, _dims(case)), VIDEO_MAX_POS),
                                     ("audio_", "audio", AUDIO, "v2a", _audio_positions(b, case["audio"]), TIME_MAX_POS)):
        x = _lin64(p, pre + "patchify_proj", lat[k].double())
        if k == "video":
            x = x + (kf > 0).double() * p("keyframes_abs_pos_embedding")
        ts, emb = _adaln64(p.at(pre + "adaln_single."), t)
        st[k] = dict(x=x, ts=ts.view(9, d), emb=emb.view(d), ctx=ctx[k].double(),
                     prompt=_adaln64(p.at(pre + "prompt_adaln_single."), t)[0].view(2, d),
                     css=_adaln64(p.at("av_ca_%s_scale_shift_adaln_single." % k), t)[0].view(4, d),
                     cgate=_adaln64(p.at("av_ca_%s_gate_adaln_single." % gate), t)[0].view(d),
                     pe=_tables64(pos[:1], d, mp), cpe=_tables64(pos[:1, 0:1], AUDIO, TIME_MAX_POS))
    v, a = st["video"], st["audio"]
    for i in range(n):
        q = p.at("blocks.%d." % i)
        mask = [keep[j, i].view(b, 1, 1) for j in range(4)]
        for o, pre, m in ((v, "", mask[0]), (a, "audio_", mask[1])):
            r = q(pre + "scale_shift_table") + o["ts"]
            o["rows"] = r
            x = o["x"]
            x = x + _attn64(q.at(pre + "attn1."), _rms64(x) * (1 + r[1]) + r[0], pe=o["pe"], keep=m) * r[2]
            kv = q(pre + "prompt_scale_shift_table") + o["prompt"]
            x = x + _attn64(q.at(pre + "attn2."), _rms64(x) * (1 + r[7]) + r[6], o["ctx"] * (1 + kv[1]) + kv[0]) * r[8]
            o["x"] = x
        av = {}
        for o, k in ((v, "video"), (a, "audio")):
            tab = q("scale_shift_table_a2v_ca_" + k)
            r = torch.cat([tab[:4] + o["css"], (tab[4] + o["cgate"]).unsqueeze(0)])
            y = _rms64(o["x"])
            av[k] = (y * (1 + r[0]) + r[1], y * (1 + r[2]) + r[3], r[4])
        v["x"] = v["x"] + _attn64(q.at("audio_to_video_attn."), av["video"][0], av["audio"][0], v["cpe"], a["cpe"]) \
            * av["video"][2] * mask[2]
        a["x"] = a["x"] + _attn64(q.at("video_to_audio_attn."), av["audio"][1], av["video"][1], a["cpe"], v["cpe"]) \
            * av["audio"][2] * mask[3]
        for o, pre in ((v, ""), (a, "audio_")):
            r = o["rows"]
            o["x"] = o["x"] + _ffn64(q.at(pre + "ff."), _rms64(o["x"]) * (1 + r[4]) + r[3]) * r[5]
    out = []
    for o, pre in ((v, ""), (a, "audio_")):
        r = p(pre + "scale_shift_table") + o["emb"]
        x = torch.nn.functional.layer_norm(o["x"], (o["x"].shape[-1],), eps=EPS) * (1 + r[1]) + r[0]
        out.append(_lin64(p, pre + "proj_out", x))
    return tuple(out)


@torch.no_grad()
def exact(case, seed):
    kind, b = case["kind"], case.get("batch", 1)
    if kind == "noise":
        shape = (b, case["tokens"], 128)
        v = _rand(seed, "v", shape, dtype=getattr(torch, case["dtype"])).double()
        x = _noise64(math.prod(shape), seed).view(shape)
        return x.to(getattr(torch, case["dtype"])).double() - 0.125 * v
    if kind == "norm":
        return _norm64(case, seed)
    if kind == "self":
        dim, _, _ = _stream_dims(case["stream"])
        pos, max_pos = _positions(case, case["stream"])
        p = _Params(seed, _attn_shapes("", dim, dim, dim))
        return _attn64(p, _rand(seed, "x", (b, pos.shape[2], dim)).double(), pe=_tables64(pos, dim, max_pos))
    if kind == "text":
        dim, _, _ = _stream_dims(case["stream"])
        p = _Params(seed, _attn_shapes("", dim, dim, dim))
        return _attn64(p, _rand(seed, "x", (b, case["tokens"], dim)).double(),
                       _rand(seed, "context", (b, case["text"], dim)).double())
    if kind in ("a2v", "v2a"):
        qd, cd = (VIDEO, AUDIO) if kind == "a2v" else (AUDIO, VIDEO)
        p = _Params(seed, _attn_shapes("", qd, cd, AUDIO))
        video = _rand(seed, "video", (b, _tokens(case), VIDEO)).double()
        audio = _rand(seed, "audio", (b, case["audio"], AUDIO)).double()
        vpe = _tables64(_video_positions(b, _dims(case))[:, 0:1], AUDIO, TIME_MAX_POS)
        ape = _tables64(_audio_positions(b, case["audio"]), AUDIO, TIME_MAX_POS)
        return _attn64(p, video, audio, vpe, ape) if kind == "a2v" else _attn64(p, audio, video, ape, vpe)
    if kind == "ffn":
        p = _Params(seed, _ffn_shapes("", case["dim"], case["bias"]))
        return _ffn64(p, _rand(seed, "x", (b, case["tokens"], case["dim"])).double())
    if kind == "guide":
        return _guide64(case, seed)
    if kind == "te":
        return _te64(case, seed)
    return _model64(case, seed)
