"""The GEMM's epilogues at the edges of the parts a wave writes (128 rows by 64
columns, in quarters of 32 rows or, fp32, eighths of 16): rows and columns that
end inside, at and just past them, with the text stream beginning in the same
tile.  The projection is compared with float64 on the same bf16 operands within
the bound of an fp32 sum of k products, (k + 2) 2^-24 of the sum of their
magnitudes; 16-bit outputs must be the rounding of the fp32 output, and the
residual epilogue the projection followed by ada_out, bit for bit."""
import pytest

from seedvr2_ncnn_amd import capi

pytestmark = pytest.mark.gpu

ROWS = [(1, 0), (31, 3), (33, 16), (127, 1), (129, 15), (250, 17), (257, 33)]
COLS = [8, 72, 136, 264]


def _inputs(mv, mt, k, n):
    import torch
    gen = torch.Generator(device="cuda").manual_seed(1000 * mv + n)
    draw = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    xt = draw(mt, k).bfloat16() if mt else None
    return draw, draw(mv, k).bfloat16(), xt, (0.1 * draw(n, k)).bfloat16(), 0.1 * draw(n)


@pytest.mark.parametrize("mv,mt", ROWS)
@pytest.mark.parametrize("n", COLS + [12, 7, 288, 261])
def test_plain_outputs(mv, mt, n):
    # (rows of whole 64-byte sectors: 288; of 16-byte chunks that share sectors:
    # COLS, and 12 in fp32; of single elements: 12 in 16 bits, 7, 261)
    import torch
    k = 128
    _, xv, xt, w, b = _inputs(mv, mt, k, n)
    full = capi.shared_linear(xv, xt, w, b, out_dtype=torch.float32)
    for x, y in zip((xv, xt), full):
        if x is None:
            continue
        xd, wd = x.double(), w.double().t().contiguous()
        bound = (k + 2) * 2.0 ** -24 * (xd.abs() @ wd.abs() + b.abs().double())
        assert ((y.double() - (xd @ wd + b.double())).abs() <= bound).all()
    for dt in (torch.bfloat16, torch.float16):
        half = capi.shared_linear(xv, xt, w, b, out_dtype=dt)
        for y, h in zip(full, half):
            assert h is None or torch.equal(h, y.to(dt))


@pytest.mark.parametrize("mv,mt", ROWS)
@pytest.mark.parametrize("n", COLS)
@pytest.mark.parametrize("dtype", ["float32", "bfloat16", "float16"])
def test_residual_equals_projection_and_ada_out(mv, mt, n, dtype):
    import torch
    draw, xv, xt, w, b = _inputs(mv, mt, 64, n)
    dt = getattr(torch, dtype)
    rv, rt = draw(mv, n).to(dt), draw(mt, n).to(dt) if mt else None
    split = mv // 3   # two samples, the first one's rows ending inside a part
    vr, tr = [split, mv - split], [mt // 2, mt - mt // 2] if mt else None
    gate = draw(2, n)
    got = capi.shared_linear_residual(xv, xt, w, b, vr, tr, rv, rt, gate,
                                      out_video=torch.empty_like(rv),
                                      out_text=torch.empty_like(rt) if mt else None)
    yv, yt = capi.shared_linear(xv, xt, w, b)
    ref = capi.ada_out(rv.clone(), rt.clone() if mt else None, yv, yt, vr, tr, gate)
    torch.cuda.synchronize()
    assert torch.equal(got[0], ref[0])
    assert not mt or torch.equal(got[1], ref[1])


@pytest.mark.parametrize("mv,mt", ROWS + [(128, 64), (192, 0), (200, 300), (0, 40),
                                          ((128, 300, 212), (40, 130, 200)),
                                          ((127, 129, 384), (128, 1, 63)),
                                          ((500, 0, 140), (64, 0, 64))])
@pytest.mark.parametrize("n", [8, 264])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16", "float16"])
@pytest.mark.parametrize("own_gates", [False, True])
def test_residual_samples_and_streams_of_a_wave(mv, mt, n, dtype, own_gates):
    """A wave goes over its 128 rows once for each sample of each stream in them:
    one sample, and three whose ends lie on and off the waves' edges, one of
    them empty; rows of either stream that fill no wave."""
    import torch
    if isinstance(mv, tuple):
        vr, tr, mv, mt = list(mv), list(mt), sum(mv), sum(mt)
    else:
        vr, tr = [mv], [mt] if mt else None
    draw, xv, xt, w, b = _inputs(mv, mt, 64, n)
    dt = getattr(torch, dtype)
    rv, rt = draw(mv, n).to(dt), draw(mt, n).to(dt) if mt else None
    gate, gates = draw(len(vr), n), dict(video_gate=draw(n), text_gate=draw(n)) if own_gates else {}
    got = capi.shared_linear_residual(xv, xt, w, b, vr, tr, rv, rt, gate,
                                      out_video=torch.empty_like(rv),
                                      out_text=torch.empty_like(rt) if mt else None, **gates)
    yv, yt = capi.shared_linear(xv, xt, w, b)
    ref = capi.ada_out(rv.clone(), rt.clone() if mt else None, yv, yt, vr, tr, gate, **gates)
    torch.cuda.synchronize()
    assert torch.equal(got[0], ref[0])
    assert not mt or torch.equal(got[1], ref[1])
