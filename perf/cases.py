"""The work a restoration program has this framework do, as measurable cases.

A case is a dict of plain values; "kind" says which entry points it calls:

  attention   the window attention layer on a fused QKV blob (s2_awa_forward)
  qkv         the QKV projection and the window attention (s2_awa_qkv_forward)
  mlp         MLP up + GELU, MLP down with the gated residual sum in its epilogue
  swiglu      the v3 MLP: SwiGLU gate/up, down
  linear      one SharedLinear over both token streams
  block       a whole DiT block: norms, modulation, QKV + attention, out, MLP, residual sums
  sampler     one sampler step around the DiT: patches in, timestep, guided Euler update out
  conv        the VAE's causal 3-D convolution over two consecutive slices of a video
  mha         the VAE's self attention over one latent frame

Weights and activations have the distributions of the repository's benchmark:
activations N(0, 1), weights N(0, 0.02) for the DiT and N(0, 1 / fan-in) for
the VAE, norm weights 1 + N(0, 0.02).
"""
import math

import numpy as np
import torch

from seedvr2_ncnn_amd import capi

PAIRS = 21                # rotary pairs per axis at head dim 128
TYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}


def listed():
    return [
        # The layer alone as a graph calls it on fp32 blobs: a 512 x 512 image's
        # 32 x 32 token grid, one frame; a few launches of a few microseconds.
        dict(name="attention_small", kind="attention", t=1, h=32, w=32, heads=8, dim=64, pairs=10,
             tt=1, th=8, tw=8, shifted=0, text=64, dtype="fp32"),
        # A 1024 x 1024 image (one frame of 64 x 64 tokens) in the 3B model,
        # one of its shifted-window blocks.
        dict(name="qkv_image", kind="qkv", t=1, h=64, w=64, heads=20, shifted=1, text=64),
        # The 720p video of the benchmark: 21 frames, 6 x 45 x 80 tokens, 3B.
        dict(name="qkv_video", kind="qkv", t=6, h=45, w=80, heads=20, shifted=0, text=64),
        # The 3B MLP on an odd-sized image (33 x 45 tokens), rows that fill no tile.
        dict(name="mlp_image", kind="mlp", rows=1485, text=64, hidden=2560, inner=10240),
        # The same on the 720p video: the largest projections of a block.
        dict(name="mlp_video", kind="mlp", rows=21600, text=64, hidden=2560, inner=10240),
        # The v3 model's MLP on a short clip (5 frames of 640 x 480: 2 x 30 x 40 tokens).
        dict(name="swiglu_clip", kind="swiglu", rows=2400, text=64, hidden=2560, inner=3456),
        # The out projection on fp32 blobs, the type of the layers' host surface,
        # on one frame of 720p (45 x 80 tokens) with an odd prompt length.
        dict(name="linear_fp32", kind="linear", rows=3600, text=77, k=2560, n=2560, dtype="fp32"),
        # A whole block on a 768 x 768 image (48 x 48 tokens): what one of the
        # 32 steps of a restoration of a photograph is made of.
        dict(name="block_image", kind="block", t=1, h=48, w=48, heads=20, shifted=0, text=64),
        # The DiT's frontend and tail at the 720p latent, guidance with rescale.
        dict(name="sampler_step", kind="sampler", t=6, h=90, w=160, scale=6.5, rescale=0.7),
        # The VAE's 512-channel layers at latent resolution (720p), slice by slice.
        dict(name="conv_latent", kind="conv", cin=512, cout=512, frames=1, h=90, w=160, dtype="bf16"),
        # The decoder's full-resolution layers, four frames a slice.
        dict(name="conv_full", kind="conv", cin=128, cout=128, frames=4, h=720, w=1280, dtype="bf16"),
        # The VAE's attention over one 720p latent frame.
        dict(name="mha_latent", kind="mha", seq=14400, width=512, dtype="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["attention", "qkv", "mlp", "swiglu", "linear", "block", "sampler", "conv",
                       "mha"])
    text = rng.choice([64, 64, 58, 77, 16])
    if kind == "attention":
        heads, dim, pairs = rng.choice([(8, 64, 10), (20, 128, 21), (24, 128, 21)])
        tt, th, tw = rng.choice([(1, 8, 8), (4, 3, 3)])
        return dict(kind=kind, t=_log(rng, 1, 3), h=_log(rng, 16, 64), w=_log(rng, 16, 64),
                    heads=heads, dim=dim, pairs=pairs, tt=tt, th=th, tw=tw,
                    shifted=rng.randrange(2), text=text, dtype=rng.choice(["fp32", "bf16", "fp16"]))
    if kind in ("qkv", "block"):
        return dict(kind=kind, t=_log(rng, 1, 5), h=_log(rng, 16, 45), w=_log(rng, 16, 80),
                    heads=rng.choice([20, 24]), shifted=rng.randrange(2), text=text)
    if kind == "mlp":
        hidden = rng.choice([2560, 3072])
        return dict(kind=kind, rows=_log(rng, 256, 15000), text=text, hidden=hidden,
                    inner=4 * hidden)
    if kind == "swiglu":
        return dict(kind=kind, rows=_log(rng, 256, 21600), text=text, hidden=2560, inner=3456)
    if kind == "linear":
        hidden = rng.choice([2560, 3072])
        k, n = rng.choice([(hidden, hidden), (hidden, 3 * hidden), (4 * hidden, hidden)])
        return dict(kind=kind, rows=_log(rng, 256, 15000), text=text, k=k, n=n,
                    dtype=rng.choice(["fp32", "bf16", "fp16"]))
    if kind == "sampler":
        return dict(kind=kind, t=_log(rng, 1, 6), h=2 * _log(rng, 16, 45), w=2 * _log(rng, 16, 80),
                    scale=rng.choice([1.0, 6.5, 7.5]), rescale=rng.choice([0.0, 0.7]))
    if kind == "conv":
        # channels with the resolution the VAE runs them at, as parts of 720p
        cin, cout, frames, part = rng.choice([(512, 512, 1, 8), (512, 512, 2, 4), (512, 256, 4, 2),
                                              (256, 256, 4, 2), (256, 128, 4, 1), (128, 128, 4, 1),
                                              (128, 3, 4, 1), (3, 128, 4, 1)])
        size = math.exp(rng.uniform(math.log(0.3), 0.0))
        h, w = (max(12, int(n * size / part)) for n in (720, 1280))
        if cin * cout > 128 * 128 and part < 4:
            h, w = int(h * 0.7), int(w * 0.7)
        return dict(kind=kind, cin=cin, cout=cout, frames=frames, h=h, w=w,
                    dtype=rng.choice(["bf16", "bf16", "fp16", "fp32"]))
    return dict(kind=kind, seq=_log(rng, 256, 14400), width=512,
                dtype=rng.choice(["bf16", "bf16", "fp32"]))


# ---- what a program has in hand before the call ------------------------------

class _Random:
    """Seeded device tensors, in one order for a case and a seed."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(int(seed))

    def __call__(self, *shape, std=1.0, mean=0.0, dtype=torch.float32):
        x = torch.randn(*shape, generator=self.gen, device="cuda")
        return x.mul_(std).add_(mean).to(dtype)

    def weight(self, n, k):
        return self(n, k, std=0.02, dtype=torch.bfloat16)

    def bias(self, n):
        return self(n, std=0.02)


def _freqs(pairs):
    f = 10000.0 ** (-np.arange(pairs, dtype=np.float64) / pairs)
    return torch.from_numpy(f.astype(np.float32)).cuda()


def _attention_inputs(case, seed):
    r = _Random(seed)
    dtype, width = TYPES[case["dtype"]], 3 * case["heads"] * case["dim"]
    return dict(video=r(case["t"] * case["h"] * case["w"], width, dtype=dtype),
                text=r(case["text"], width, dtype=dtype),
                norms=r(4, case["dim"], std=0.02, mean=1.0), freqs=_freqs(case["pairs"]))


def _qkv_inputs(case, seed):
    r = _Random(seed)
    d = 128 * case["heads"]
    bf = torch.bfloat16
    return dict(xv=r(case["t"] * case["h"] * case["w"], d, dtype=bf), xt=r(case["text"], d, dtype=bf),
                w=r.weight(3 * d, d), b=r.bias(3 * d), norms=r(4, 128, std=0.02, mean=1.0),
                freqs=_freqs(PAIRS))


def _mlp_inputs(case, seed):
    r = _Random(seed)
    d, f, m, t = case["hidden"], case["inner"], case["rows"], case["text"]
    bf = torch.bfloat16
    return dict(xv=r(m, d, dtype=bf), xt=r(t, d, dtype=bf), up=r.weight(f, d), bup=r.bias(f),
                dn=r.weight(d, f), bdn=r.bias(d), rv=r(m, d), rt=r(t, d),
                gate=r(1, d, std=0.1))


def _swiglu_inputs(case, seed):
    r = _Random(seed)
    d, f = case["hidden"], case["inner"]
    bf = torch.bfloat16
    return dict(xv=r(case["rows"], d, dtype=bf), xt=r(case["text"], d, dtype=bf),
                wg=r.weight(f, d), wu=r.weight(f, d), bg=r.bias(f), bu=r.bias(f),
                dn=r.weight(d, f), bdn=r.bias(d))


def _linear_inputs(case, seed):
    r = _Random(seed)
    dtype = TYPES[case["dtype"]]
    return dict(xv=r(case["rows"], case["k"], dtype=dtype), xt=r(case["text"], case["k"], dtype=dtype),
                w=r.weight(case["n"], case["k"]), b=r.bias(case["n"]))


MODULATION = ("a_shift", "a_scale", "a_gate", "m_shift", "m_scale", "m_gate")


def _block_inputs(case, seed):
    r = _Random(seed)
    d = 128 * case["heads"]
    s = dict(rv=r(case["t"] * case["h"] * case["w"], d), rt=r(case["text"], d),
             w=r.weight(3 * d, d), b=r.bias(3 * d), norms=r(4, 128, std=0.02, mean=1.0),
             freqs=_freqs(PAIRS), o=r.weight(d, d), bo=r.bias(d), up=r.weight(4 * d, d),
             bup=r.bias(4 * d), dn=r.weight(d, 4 * d), bdn=r.bias(d))
    for k in MODULATION:
        s[k] = r(1, d, std=0.1, mean=1.0 if k.endswith("scale") else 0.0)
    return s


def _sampler_inputs(case, seed):
    r = _Random(seed)
    t, h, w = case["t"], case["h"], case["w"]
    patches = t * (h // 2) * (w // 2)
    positive = r(patches, 64)
    return dict(noise=r(16, t * h * w), condition=r(16, t * h * w), positive=positive,
                negative=None if case["scale"] == 1.0 else positive * 0.9 + 0.3 * r(patches, 64))


def _conv_inputs(case, seed):
    r = _Random(seed)
    cin, cout = case["cin"], case["cout"]
    n = case["frames"] * case["h"] * case["w"]
    n4 = (n + 7) // 8 * 8
    return dict(wts=r(3, cout, cin, 3, 3, std=(cin * 27) ** -0.5), bias=r(cout, std=0.1),
                x0=r(cin, n4, dtype=TYPES[case["dtype"]]), x1=r(cin, n4, dtype=TYPES[case["dtype"]]))


def _mha_inputs(case, seed):
    r = _Random(seed)
    e = case["width"]
    s = dict(x=r(case["seq"], e, dtype=TYPES[case["dtype"]]))
    for n in ("q", "k", "v", "o"):
        s["w" + n], s["b" + n] = r(e, e, std=e ** -0.5), r(e, std=0.1)
    return s


INPUTS = dict(attention=_attention_inputs, qkv=_qkv_inputs, mlp=_mlp_inputs, swiglu=_swiglu_inputs,
              linear=_linear_inputs, block=_block_inputs, sampler=_sampler_inputs,
              conv=_conv_inputs, mha=_mha_inputs)


def _plan(case, state, dim, pairs, target):
    config = capi.awa_config(case["heads"], dim, target, case["shifted"], 1e-5, pairs)
    plan = capi.AwaPlan(config, [(case["t"], case["h"], case["w"])], [case["text"]])
    plan.cache_rope(state["freqs"])
    state["plan"] = plan
    state["ws"] = torch.empty(plan.info.workspace_bytes, dtype=torch.uint8, device="cuda")


def prepare(case, seed):
    kind = case["kind"]
    s = INPUTS[kind](case, seed)
    bf = torch.bfloat16
    if kind == "attention":
        _plan(case, s, case["dim"], case["pairs"], (case["tt"], case["th"], case["tw"]))
    elif kind in ("qkv", "block"):
        _plan(case, s, 128, PAIRS, (4, 3, 3))
    if kind == "block":
        # the blobs between the block's layers
        d = 128 * case["heads"]
        for n, width in (("h", d), ("a", d), ("y", d), ("m", 4 * d)):
            s[n + "v"] = torch.empty(s["rv"].shape[0], width, dtype=bf, device="cuda")
            s[n + "t"] = torch.empty(case["text"], width, dtype=bf, device="cuda")
    elif kind == "mlp":
        s["hv"] = torch.empty(case["rows"], case["inner"], dtype=bf, device="cuda")
        s["ht"] = torch.empty(case["text"], case["inner"], dtype=bf, device="cuda")
    elif kind == "swiglu":
        s["packed"], s["bpacked"] = capi.swiglu_pack_weight(s["wg"], s["wu"], s["bg"], s["bu"])
    elif kind == "conv":
        config = capi.conv3d_config(num_output=case["cout"], num_input=case["cin"], kernel_t=3,
                                    kernel_h=3, kernel_w=3, pad_h=1, pad_w=1, head_frames=2,
                                    bias_term=1)
        s["conv"] = capi.Conv3d(config, s.pop("wts"), s.pop("bias"))
    elif kind == "mha":
        s["mha"] = capi.Mha(1, *(s.pop(k) for k in ("wq", "bq", "wk", "bk", "wv", "bv", "wo", "bo")))
    s["case"] = case
    return s


# ---- one pass -----------------------------------------------------------------

def _run_attention(c, s):
    n = c["heads"] * c["dim"]
    v, t = s["video"], s["text"]
    return capi.awa_forward(s["plan"], s["norms"], s["freqs"], v[:, :n], v[:, n:2 * n], v[:, 2 * n:],
                            t[:, :n], t[:, n:2 * n], t[:, 2 * n:], workspace=s["ws"])


def _run_qkv(c, s):
    return capi.awa_qkv_forward(s["plan"], s["xv"], s["xt"], s["w"], s["b"], s["norms"], s["freqs"],
                                workspace=s["ws"])


def _run_mlp(c, s):
    capi.shared_linear(s["xv"], s["xt"], s["up"], s["bup"], capi.ACT_GELU, y_video=s["hv"],
                       y_text=s["ht"])
    return capi.shared_linear_residual(s["hv"], s["ht"], s["dn"], s["bdn"], [c["rows"]], [c["text"]],
                                       s["rv"], s["rt"], s["gate"],
                                       out_video=torch.empty_like(s["rv"]),
                                       out_text=torch.empty_like(s["rt"]))


def _run_swiglu(c, s):
    hv, ht = capi.shared_linear(s["xv"], s["xt"], s["packed"], s["bpacked"], capi.ACT_SWIGLU)
    return capi.shared_linear(hv, ht, s["dn"], s["bdn"])


def _run_linear(c, s):
    return capi.shared_linear(s["xv"], s["xt"], s["w"], s["b"])


def _run_block(c, s):
    vr, tr = [s["rv"].shape[0]], [c["text"]]
    ov, ot = torch.empty_like(s["rv"]), torch.empty_like(s["rt"])
    capi.ada_in(s["rv"], s["rt"], vr, tr, s["a_shift"], s["a_scale"], out_video=s["hv"],
                out_text=s["ht"])
    capi.awa_qkv_forward(s["plan"], s["hv"], s["ht"], s["w"], s["b"], s["norms"], s["freqs"],
                         workspace=s["ws"], out_video=s["av"], out_text=s["at"])
    capi.shared_linear(s["av"], s["at"], s["o"], s["bo"], y_video=s["yv"], y_text=s["yt"])
    capi.ada_out_in(s["rv"], s["rt"], s["yv"], s["yt"], vr, tr, s["a_gate"], s["m_shift"],
                    s["m_scale"], h_video=s["hv"], h_text=s["ht"], out_video=ov, out_text=ot)
    capi.shared_linear(s["hv"], s["ht"], s["up"], s["bup"], capi.ACT_GELU, y_video=s["mv"],
                       y_text=s["mt"])
    capi.shared_linear(s["mv"], s["mt"], s["dn"], s["bdn"], y_video=s["yv"], y_text=s["yt"])
    return capi.ada_out(ov, ot, s["yv"], s["yt"], vr, tr, s["m_gate"])


def _run_sampler(c, s):
    t, h, w = c["t"], c["h"], c["w"]
    # a one-step sampler: the latent starts as the noise, which the program keeps
    latent = s["noise"].clone()
    patches = capi.latent_patches(latent, s["condition"], t, h, w, t * h * w)
    embedding = capi.timestep_embedding([1000.0])
    capi.denoise_update(s["positive"], s["negative"], t, h, w, c["scale"], c["rescale"], -1.0,
                        latent, t * h * w)
    return patches, embedding, latent


def _run_conv(c, s):
    # a video's first slice, then the next one on the frames the first one left
    conv, n = s["conv"], c["frames"] * c["h"] * c["w"]
    y0, _ = conv.forward(s["x0"], c["frames"], c["h"], c["w"], keep_memory=True)
    y1, _ = conv.forward(s["x1"], c["frames"], c["h"], c["w"], use_memory=True, keep_memory=True,
                         reuse_memory_buffer=True)
    return y0, y1


def _run_mha(c, s):
    return s["mha"].forward(s["x"])


RUN = dict(attention=_run_attention, qkv=_run_qkv, mlp=_run_mlp, swiglu=_run_swiglu,
           linear=_run_linear, block=_run_block, sampler=_run_sampler, conv=_run_conv, mha=_run_mha)


def run(state):
    return RUN[state["case"]["kind"]](state["case"], state)


# ---- what a pass cannot do without -------------------------------------------

def _axis(n, extent, shifted):
    """Windows of one axis: a regular grid, or one moved by half a window."""
    if not shifted:
        return [(lo, min(lo + extent, n)) for lo in range(0, n, extent)]
    if extent >= n:
        return [(0, n)]
    edges = [0]
    k = 1
    while edges[-1] < n:
        edges.append(min((2 * k - 1) * extent // 2, n))
        k += 1
    return [(lo, hi) for lo, hi in zip(edges, edges[1:]) if hi > lo]


def _windows(t, h, w, target, shifted):
    """(t, h, w) bounds of the windows: the grid is cut as one of about 3600
    tokens a frame would be into target windows."""
    s = math.sqrt(3600.0 / (h * w))
    sizes = [-(-min(t, 30) // target[0]), -(-round(h * s) // target[1]), -(-round(w * s) // target[2])]
    bounds = [_axis(n, e, shifted) for n, e in zip((t, h, w), sizes)]
    return [(a, b, c) for c in bounds[2] for b in bounds[1] for a in bounds[0]]


def _target(case):
    return (case["tt"], case["th"], case["tw"]) if case["kind"] == "attention" else (4, 3, 3)


def _attention_flops(case, dim):
    total = 0
    for win in _windows(case["t"], case["h"], case["w"], _target(case), case["shifted"]):
        n = math.prod(hi - lo for lo, hi in win) + case["text"]
        total += 4 * case["heads"] * dim * n * n
    return total


def work(case):
    kind = case["kind"]
    size = {"fp32": 4}.get(case.get("dtype"), 2)
    if kind == "attention":
        m = case["t"] * case["h"] * case["w"] + case["text"]
        return dict(bytes=4 * m * case["heads"] * case["dim"] * size,
                    flops=_attention_flops(case, case["dim"]))
    if kind == "qkv":
        d = 128 * case["heads"]
        m = case["t"] * case["h"] * case["w"] + case["text"]
        return dict(bytes=2 * (2 * m * d + 3 * d * d),
                    flops=2 * m * d * 3 * d + _attention_flops(case, 128))
    if kind == "block":
        d = 128 * case["heads"]
        m = case["t"] * case["h"] * case["w"] + case["text"]
        return dict(bytes=2 * 12 * d * d + 8 * m * d,
                    flops=2 * m * d * 12 * d + _attention_flops(case, 128))
    if kind == "mlp":
        m, d, f = case["rows"] + case["text"], case["hidden"], case["inner"]
        return dict(bytes=10 * m * d + 4 * d * f, flops=4 * m * d * f)
    if kind == "swiglu":
        m, d, f = case["rows"] + case["text"], case["hidden"], case["inner"]
        return dict(bytes=4 * m * d + 6 * d * f, flops=6 * m * d * f)
    if kind == "linear":
        m, k, n = case["rows"] + case["text"], case["k"], case["n"]
        return dict(bytes=size * m * (k + n) + 2 * n * k, flops=2 * m * k * n)
    if kind == "sampler":
        tokens = case["t"] * case["h"] * case["w"]
        # noise, condition, one or two predictions in; patches and the latent out
        return dict(bytes=tokens * 4 * (16 + 16 + (16 if case["scale"] == 1.0 else 32) + 33 + 16),
                    flops=10 * 16 * tokens)
    if kind == "conv":
        n = case["frames"] * case["h"] * case["w"]
        cin, cout = case["cin"], case["cout"]
        return dict(bytes=2 * n * (cin + cout) * size + 2 * 27 * cin * cout,
                    flops=2 * 2 * n * 27 * cin * cout)
    e, n = case["width"], case["seq"]
    return dict(bytes=2 * n * e * size + 8 * e * e, flops=8 * n * e * e + 4 * n * n * e)


def tolerance(case):
    """About four times the distance of a pass from exact(): bf16 operands of
    the products, and 16-bit outputs; fp32 in the sampler."""
    kind = case["kind"]
    if kind == "sampler":
        return {"rel": 1e-6}
    return {"rel": dict(attention=1.4e-2, qkv=1.7e-2, mlp=1.5e-3, swiglu=1e-2, linear=7e-3,
                        block=2e-3, conv=1e-2, mha=1.4e-2)[kind]}


# ---- the same in 64 bits -------------------------------------------------------

def _rms(x, eps=1e-5):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _rotate(x, pos, freqs):
    """x [tokens, heads, dim], pos [tokens, 3]: pairs of each axis's slice turned."""
    p = freqs.numel()
    out = x.clone()
    for axis in range(3):
        angle = (pos[:, axis, None] * freqs)[:, None, :]
        a, b = (x[..., 2 * p * axis + i:2 * p * (axis + 1):2] for i in (0, 1))
        out[..., 2 * p * axis:2 * p * (axis + 1):2] = a * angle.cos() - b * angle.sin()
        out[..., 2 * p * axis + 1:2 * p * (axis + 1):2] = a * angle.sin() + b * angle.cos()
    return out


def _exact_attention(case, video, text, norms, freqs, dim):
    """video [tokens, 3 * inner], text likewise, in 64 bits; (video, text) contexts."""
    t, h, w, heads, lt = (case[k] for k in ("t", "h", "w", "heads", "text"))
    norms, freqs = norms.double(), freqs.double()
    q, k, v = (x.reshape(-1, heads, dim) for x in video.chunk(3, 1))
    tq, tk, tv = (x.reshape(-1, heads, dim) for x in text.chunk(3, 1))
    tpos = torch.arange(lt, device="cuda", dtype=torch.float64)[:, None].expand(lt, 3)
    tq = _rotate(_rms(tq) * norms[2], tpos, freqs)
    tk = _rotate(_rms(tk) * norms[3], tpos, freqs)
    out_v = torch.empty(t * h * w, heads * dim, dtype=torch.float64, device="cuda")
    out_t = torch.zeros(lt, heads * dim, dtype=torch.float64, device="cuda")
    token = torch.arange(t * h * w, device="cuda").view(t, h, w)
    windows = _windows(t, h, w, _target(case), case["shifted"])
    for (t0, t1), (h0, h1), (w0, w1) in windows:
        src = token[t0:t1, h0:h1, w0:w1].reshape(-1)
        axes = (torch.arange(n, device="cuda", dtype=torch.float64) for n in (t1 - t0, h1 - h0, w1 - w0))
        pos = torch.stack(torch.meshgrid(*axes, indexing="ij"), -1).reshape(-1, 3)
        pos[:, 0] += lt
        qq = torch.cat([_rotate(_rms(q[src]) * norms[0], pos, freqs), tq]).transpose(0, 1)
        kk = torch.cat([_rotate(_rms(k[src]) * norms[1], pos, freqs), tk]).permute(1, 2, 0)
        vv = torch.cat([v[src], tv]).transpose(0, 1).contiguous()
        ctx = torch.softmax(qq.contiguous() @ kk.contiguous() / math.sqrt(dim), -1) @ vv
        ctx = ctx.transpose(0, 1).reshape(-1, heads * dim)
        n = src.numel()
        out_v[src] = ctx[:n]
        out_t += ctx[n:] / len(windows)
    return out_v, out_t


def _gelu(x):
    return 0.5 * x * (1 + torch.erf(x / math.sqrt(2.0)))


def _linear(x, w, b):
    return x @ w.double().t().contiguous() + b.double()


def _exact_conv(case, s):
    frames, h, w = case["frames"], case["h"], case["w"]
    cin, cout, n = case["cin"], case["cout"], frames * h * w
    wts = s["wts"].double()
    # both slices as one video behind two copies of its first frame, padded by a pixel
    x = torch.cat([s["x0"][:, :n], s["x1"][:, :n]], 1).view(cin, 2 * frames, h, w)
    outs = []
    for half in range(2):
        y = torch.empty(cout, frames, h * w, dtype=torch.float64, device="cuda")
        for f in range(frames):
            acc = s["bias"].double()[:, None].expand(cout, h * w).clone()
            for tap in range(3):
                frame = x[:, max(0, half * frames + f + tap - 2)].double()
                frame = torch.nn.functional.pad(frame, (1, 1, 1, 1))
                for ky in range(3):
                    for kx in range(3):
                        acc += wts[tap, :, :, ky, kx].contiguous() @ \
                            frame[:, ky:ky + h, kx:kx + w].reshape(cin, h * w)
            y[:, f] = acc
        outs.append(y.view(cout, n))
    return tuple(outs)


def _exact_mha(case, s):
    x = s["x"].double()
    q, k, v = (_linear(x, s["w" + n], s["b" + n]) for n in "qkv")
    kt = k.t().contiguous()
    out = torch.empty_like(x)
    for rows in torch.arange(x.shape[0], device="cuda").split(2048):
        p = torch.softmax(q[rows] @ kt / math.sqrt(case["width"]), -1)
        out[rows] = _linear(p @ v, s["wo"], s["bo"])
    return out


def _exact_sampler(case, s):
    t, h, w = case["t"], case["h"], case["w"]
    noise = s["noise"].double()
    # patches: 2 x 2 tokens of [latent 16 | condition 16 | 1]
    tokens = torch.cat([noise, s["condition"].double(), torch.ones_like(noise[:1])])
    patches = tokens.view(33, t, h // 2, 2, w // 2, 2).permute(1, 2, 4, 3, 5, 0).reshape(-1, 132)
    # the phase is one of 32 bits by definition: frequencies and phases are rounded, sines are not
    steps = torch.arange(128, device="cuda", dtype=torch.float32)
    freq = torch.exp((-math.log(10000.0) * steps / 128).double()).float()
    phase = (1000.0 * freq).double()
    embedding = torch.cat([phase.sin(), phase.cos()])[None]
    pred = s["positive"].double()
    if s["negative"] is not None:
        neg = s["negative"].double()
        cfg = neg + case["scale"] * (pred - neg)
        if case["rescale"]:
            cfg = cfg * (case["rescale"] * pred.std() / cfg.std() + (1 - case["rescale"]))
        pred = cfg
    planes = pred.view(t, h // 2, w // 2, 2, 2, 16).permute(5, 0, 1, 3, 2, 4).reshape(16, -1)
    return patches, embedding, noise - planes


def exact(case, seed):
    kind = case["kind"]
    s = INPUTS[kind](case, seed)
    if kind == "attention":
        return _exact_attention(case, s["video"].double(), s["text"].double(), s["norms"], s["freqs"],
                                case["dim"])
    if kind == "qkv":
        return _exact_attention(case, _linear(s["xv"].double(), s["w"], s["b"]),
                                _linear(s["xt"].double(), s["w"], s["b"]), s["norms"], s["freqs"], 128)
    if kind == "mlp":
        return tuple(s["r" + n].double() + s["gate"].double() *
                     _linear(_gelu(_linear(s["x" + n].double(), s["up"], s["bup"])), s["dn"], s["bdn"])
                     for n in "vt")
    if kind == "swiglu":
        out = []
        for n in "vt":
            x = s["x" + n].double()
            g = _linear(x, s["wg"], s["bg"])
            out.append(_linear(g * torch.sigmoid(g) * _linear(x, s["wu"], s["bu"]), s["dn"], s["bdn"]))
        return tuple(out)
    if kind == "linear":
        return tuple(_linear(s["x" + n].double(), s["w"], s["b"]) for n in "vt")
    if kind == "block":
        m = {k: s[k].double() for k in MODULATION}
        res = [s["rv"].double(), s["rt"].double()]
        qkv = [_linear(_rms(x) * m["a_scale"] + m["a_shift"], s["w"], s["b"]) for x in res]
        ctx = _exact_attention(case, *qkv, s["norms"], s["freqs"], 128)
        res = [x + m["a_gate"] * _linear(a, s["o"], s["bo"]) for x, a in zip(res, ctx)]
        hid = [_gelu(_linear(_rms(x) * m["m_scale"] + m["m_shift"], s["up"], s["bup"])) for x in res]
        return tuple(x + m["m_gate"] * _linear(y, s["dn"], s["bdn"]) for x, y in zip(res, hid))
    if kind == "sampler":
        return _exact_sampler(case, s)
    if kind == "conv":
        return _exact_conv(case, s)
    return _exact_mha(case, s)
