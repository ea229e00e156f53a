"""VAEChunkedMHA on the GPU (src/seedvr2/vae_chunked_mha.cpp:223-281: ncnn
MultiHeadAttention over one blob) against the CPU oracle.

The device runs the projections and both attention products in bf16 with
fp32 accumulation (scores and exponentials are formed in fp32; the weights of V
are rounded to bf16, and in long sequences divided by their sum afterwards).  The
bar is the path's: max-abs <= 2e-2 and cosine >=
0.9999 against the fp32-input oracle.  Sequences of VAE size are checked on
a spread of query rows (the oracle computes only those rows)."""
import ctypes

import numpy as np
import pytest

import oracle
from common import assert_close, bf16_round
from seedvr2_ncnn_amd import capi

pytestmark = pytest.mark.gpu


def _weights(g, qdim, embed):
    w = lambda *s: (g.standard_normal(s) / np.sqrt(s[-1])).astype(np.float32)
    b = lambda n: (0.1 * g.standard_normal(n)).astype(np.float32)
    return [w(embed, qdim), b(embed), w(embed, qdim), b(embed), w(embed, qdim), b(embed),
            w(qdim, embed), b(qdim)]


def _device(heads, ws, scale=None):
    import torch
    return capi.Mha(heads, *[torch.from_numpy(a).cuda() for a in ws], scale=scale)


def _run(mha, x, dtype=None, out_dtype=None):
    import torch
    t = torch.from_numpy(x).cuda()
    if dtype is not None:
        t = t.to(dtype)
    y = mha.forward(t, out_dtype=out_dtype)
    torch.cuda.synchronize()
    return y.float().cpu().numpy()


@pytest.mark.parametrize("seq,qdim,heads", [(1, 64, 1), (37, 64, 2), (200, 128, 4), (1000, 512, 1),
                                            (333, 256, 2)])
def test_mha_matches_oracle(seq, qdim, heads):
    g = np.random.default_rng(seq + qdim)
    x = g.standard_normal((seq, qdim)).astype(np.float32)
    ws = _weights(g, qdim, qdim)
    got = _run(_device(heads, ws), x)
    ref = oracle.mha(x, heads, *ws, threads=16)
    assert_close(got, ref)


def test_mha_explicit_scale_and_16bit_blobs():
    import torch
    g = np.random.default_rng(2)
    x = g.standard_normal((300, 128)).astype(np.float32)
    ws = _weights(g, 128, 128)
    mha = _device(2, ws, scale=0.3)
    for dt, odt in ((torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32)):
        xs = torch.from_numpy(x).to(dt).float().numpy()    # the stored values
        got = _run(mha, xs, dtype=dt, out_dtype=odt)
        assert_close(got, oracle.mha(xs, 2, *ws, scale=0.3, threads=16))


def test_mha_16bit_outputs_round_the_fp32_output():
    """bf16 and fp16 outputs are the round-to-nearest-even of the fp32
    output of the same call (one rounding of the fp32 result)."""
    import torch
    g = np.random.default_rng(12)
    x = bf16_round(g.standard_normal((333, 256)).astype(np.float32))
    ws = _weights(g, 256, 256)
    mha = _device(2, ws)
    outs = {odt: _run(mha, x, dtype=torch.bfloat16, out_dtype=odt)
            for odt in (torch.float32, torch.bfloat16, torch.float16)}
    ref = outs[torch.float32]
    np.testing.assert_array_equal(outs[torch.bfloat16], bf16_round(ref))
    np.testing.assert_array_equal(outs[torch.float16], ref.astype(np.float16).astype(np.float32))
    assert_close(ref, oracle.mha(x, 2, *ws, threads=16))


def test_mha_vae_frame_rows():
    """One 720p latent frame (90 x 160 = 14,400 tokens, 512 channels, one
    head): 64 query rows spread over the sequence against the oracle."""
    g = np.random.default_rng(9)
    seq, qdim = 14400, 512
    x = g.standard_normal((seq, qdim)).astype(np.float32)
    ws = _weights(g, qdim, qdim)
    got = _run(_device(1, ws), x)
    rows = np.linspace(0, seq - 1, 64).astype(np.int32)
    ref = oracle.mha(x, 1, *ws, rows=rows, threads=16, fast=True)
    assert_close(got[rows], ref)


# ---- exponentials in the score product's epilogue (long sequences) --------------

def _reference_weights(g, kind, heads):
    """64 channels a head.  plain: scores near zero.  shifted: q and k share a
    constant channel of 40, so every score is near 200 and the exponentials
    need a reference.  general: q's constant channel is another than k's, so
    the scores are near zero but far below |q| |k| and no reference shows it.
    kind may name one of these per head."""
    e = 64 * heads
    ws = _weights(g, e, e)
    for h, of_head in enumerate([kind] * heads if isinstance(kind, str) else kind):
        if of_head != "plain":
            for i, c in ((0, 0), (2, 0 if of_head == "shifted" else 1)):
                for ch in (0, 1):
                    ws[i][64 * h + ch] = 0
                    ws[i + 1][64 * h + ch] = 40 if ch == c else 0
    return ws


@pytest.mark.parametrize("seq,heads", [(1024, 1), (1601, 1), (4096, 2), (4609, 2)])
@pytest.mark.parametrize("kind", ["plain", "shifted", "general"])
def test_mha_long_sequences(seq, heads, kind):
    g = np.random.default_rng(seq + heads)
    x = g.standard_normal((seq, 64 * heads)).astype(np.float32)
    ws = _reference_weights(g, kind, heads)
    got = _run(_device(heads, ws), x)
    rows = np.concatenate([np.arange(3), g.integers(0, seq, 24), np.arange(seq - 3, seq)]).astype(np.int32)
    assert_close(got[rows], oracle.mha(x, heads, *ws, rows=rows, threads=16, fast=True))


@pytest.mark.parametrize("seq,heads", [(1024, 1), (4096, 2)])
def test_mha_weights_of_a_row_sum_to_one(seq, heads):
    """Values that are the same for every key come back as they are: what a row's
    weights are divided by is the sum of the bf16 weights themselves.  Scores
    of standard deviation 2.5, so that a few keys hold most of a row.  The
    output projection averages 512 channels of different values, so the
    rounding of the concatenated heads (rms 2^-9 / sqrt 3 a channel) is left with
    5e-5; eight of these."""
    import torch
    g = np.random.default_rng(seq)
    e = 512
    x = g.standard_normal((seq, e)).astype(np.float32)
    x[:, 0] = 1.0
    ws = _weights(g, e, e)
    ws[0] *= 2.5
    c = bf16_round(g.uniform(1, 2, e).astype(np.float32))
    ws[4] = np.zeros((e, e), np.float32)
    ws[4][:, 0] = c
    ws[5] = np.zeros(e, np.float32)
    ws[6] = np.tile(bf16_round((1 / (e * c)).astype(np.float32)), (e, 1))
    ws[7] = np.zeros(e, np.float32)
    want = float(ws[6][0].astype(np.float64) @ c)
    got = _run(_device(heads, ws), bf16_round(x), dtype=torch.bfloat16, out_dtype=torch.float32)
    assert np.abs(got.astype(np.float64) / want - 1).max() <= 4e-4


# (constant channel of q and k, the same channel in both, size of the values):
# scores at their bound, with values that a sum of unnormalised weights has no
# room for; scores about 170 and 125 powers of two below it, with values whose
# products with weights that small are, or nearly are, no normal numbers
@pytest.mark.parametrize("const,same,size", [(40, True, 1e6), (40, True, 1e12), (40, True, 1e30),
                                             (29, False, 1e-16), (25, False, 1e-7)])
def test_mha_large_and_small_values(const, same, size):
    g = np.random.default_rng(int(const + np.log10(size) + 50))
    x = g.standard_normal((1100, 64)).astype(np.float32)
    ws = _weights(g, 64, 64)
    for i, c in ((0, 0), (2, 0 if same else 1)):
        ws[i][:2] = 0
        ws[i + 1][:2] = 0
        ws[i + 1][c] = const
    for i in (4, 5):
        ws[i] = (ws[i] * size).astype(np.float32)
    ws[6] = (ws[6] / size).astype(np.float32)
    rows = np.arange(0, 1100, 37).astype(np.int32)
    assert_close(_run(_device(1, ws), x)[rows], oracle.mha(x, 1, *ws, rows=rows, threads=16))


@pytest.mark.parametrize("kinds", [("general", "plain"), ("plain", "general"),
                                   ("shifted", "general", "plain"), ("general", "shifted")])
def test_mha_heads_of_different_kinds(kinds):
    """The flag, the row sums and the row scale are one head's at a time: what a
    head leaves in them must not reach the next one.  The output projection
    keeps the heads' channels apart, so each is compared by itself."""
    seq, heads = 4096, len(kinds)
    g = np.random.default_rng(sum(map(len, kinds)))
    x = g.standard_normal((seq, 64 * heads)).astype(np.float32)
    ws = _reference_weights(g, kinds, heads)
    ws[6] *= np.kron(np.eye(heads), np.ones((64, 64))).astype(np.float32) * np.sqrt(heads)
    got = _run(_device(heads, ws), x)
    rows = np.arange(0, seq, 151).astype(np.int32)
    ref = oracle.mha(x, heads, *ws, rows=rows, threads=16, fast=True)
    for h in range(heads):
        assert_close(got[rows, 64 * h:64 * h + 64], ref[:, 64 * h:64 * h + 64])


@pytest.mark.parametrize("seq,heads", [(64, 1), (320, 2), (1024, 1), (4096, 2)])
def test_mha_bf16_rows_read_in_place(seq, heads):
    """bf16 rows that need no padding are not staged: the same bits as for the
    same values given as fp32 (which are), x as it was, also with out = x."""
    import torch
    g = np.random.default_rng(seq)
    e = 64 * heads
    mha = _device(heads, _weights(g, e, e))
    x = torch.from_numpy(g.standard_normal((seq, e)).astype(np.float32)).cuda().bfloat16()
    kept = x.clone()
    ref = mha.forward(x.float(), out_dtype=torch.bfloat16)
    got = mha.forward(x)
    torch.cuda.synchronize()
    assert torch.equal(got, ref) and torch.equal(x, kept)
    ptr, n = ctypes.byref(mha.config), ctypes.c_size_t()
    capi.check(capi.lib().s2_mha_workspace_bytes(ptr, seq, ctypes.byref(n)))
    work = torch.empty(n.value, dtype=torch.uint8, device="cuda")
    capi.check(capi.lib().s2_mha_forward(
        ptr, mha.prepared.data_ptr(), x.data_ptr(), capi.DTYPE_BF16, seq, x.data_ptr(),
        capi.DTYPE_BF16, work.data_ptr(), n.value, torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert torch.equal(x, ref)


def test_mha_long_sequence_nan_reaches_every_row():
    g = np.random.default_rng(3)
    x = g.standard_normal((4700, 64)).astype(np.float32)
    x[4321, 7] = np.nan
    assert np.isnan(_run(_device(1, _weights(g, 64, 64)), x)).all()


# ---- the ncnn-surface layer (vae_chunked_mha.h:12-50) --------------------------

FP16_TAG = np.frombuffer(np.uint32(0x01306B47).tobytes(), np.float32)


def _fp16_blob(a):
    """ncnn's tagged fp16 weight: the tag, then the halves padded to 4 bytes."""
    h = np.asarray(a, np.float16).ravel()
    if h.size % 2:
        h = np.concatenate([h, np.zeros(1, np.float16)])
    return np.concatenate([FP16_TAG, h.view(np.float32)])


def _layer(embed, heads, qdim, ws, scale=None, fp16_out_weight=False):
    from common import Layer
    wq, bq, wk, bk, wv, bv, wo, bo = ws
    params = f"0={embed} 1={heads} 2={embed * qdim} 3={qdim} 4={qdim} 20=64"
    if scale is not None:
        params += f" 6={scale}"
    tag0 = np.zeros(1, np.float32)   # raw fp32 tag of a type-0 blob
    out_w = _fp16_blob(wo) if fp16_out_weight else np.concatenate([tag0, wo.ravel()])
    blobs = [tag0, wq, bq, tag0, wk, bk, tag0, wv, bv, out_w, bo]
    layer = Layer("SeedVR2ChunkedMHA", params, weights=blobs)
    assert layer.create_code == 0
    assert layer.create_pipeline() == 0
    return layer


@pytest.mark.parametrize("device", [False, True])
def test_layer_forward(device):
    import torch
    g = np.random.default_rng(12)
    x = g.standard_normal((500, 128)).astype(np.float32)
    ws = _weights(g, 128, 128)
    layer = _layer(128, 2, 128, ws)
    dt = torch.bfloat16 if device else None
    xs = torch.from_numpy(x).to(torch.bfloat16).float().numpy() if device else x
    code, got = layer.forward_rows(xs, 128, device=device, dtype=dt)
    assert code == 0
    assert_close(got, oracle.mha(xs, 2, *ws, threads=16))


def test_layer_fp16_weights_and_scale():
    g = np.random.default_rng(13)
    x = g.standard_normal((64, 64)).astype(np.float32)
    ws = _weights(g, 64, 64)
    ws[6] = ws[6].astype(np.float16).astype(np.float32)   # what the fp16 blob stores
    layer = _layer(64, 1, 64, ws, scale=0.2, fp16_out_weight=True)
    code, got = layer.forward_rows(x, 64)
    assert code == 0
    assert_close(got, oracle.mha(x, 1, *ws, scale=0.2, threads=16))


def test_layer_rejects_wrong_width():
    g = np.random.default_rng(14)
    ws = _weights(g, 64, 64)
    layer = _layer(64, 1, 64, ws)
    assert layer.forward_rows(np.zeros((8, 32), np.float32), 32)[0] == -1
