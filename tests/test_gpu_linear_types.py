"""fp32 and fp16 activations on the 256-tile GEMM (k a multiple of 64): the
kernel rounds them to bf16 between global memory and LDS and then adds the
same 32-k products in the same order as for bf16 activations, so the result
equals, bit for bit, that of the rounded activations given as bf16 (which
tests/test_gpu_linear.py checks against the oracle)."""
import pytest

from seedvr2_ncnn_amd import capi

pytestmark = pytest.mark.gpu

# one row; a video tail off an 8-row group with text rows in its tile; two,
# four and six 32-k steps (the pipeline's start and end); n that ends inside a
# wave's columns; a split tail; rows past two tiles
CASES = [(1, 0, 64, 64), (37, 5, 128, 40), (250, 70, 192, 260), (257, 3, 64, 512),
         (300, 40, 2560, 1000), (600, 1, 1088, 2560)]


@pytest.mark.parametrize("mv,mt,k,n", CASES)
@pytest.mark.parametrize("act", [capi.ACT_NONE, capi.ACT_GELU])
def test_equals_the_rounded_activations_as_bf16(mv, mt, k, n, act):
    import torch
    gen = torch.Generator(device="cuda").manual_seed(mv + k)
    draw = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    xv, xt = draw(mv, k), draw(mt, k) if mt else None
    w, b = (0.02 * draw(n, k)).bfloat16(), 0.02 * draw(n)
    for dt in (torch.float32, torch.float16):
        v, t = xv.to(dt), xt.to(dt) if mt else None
        got = capi.shared_linear(v, t, w, b, act, out_dtype=torch.float32)
        ref = capi.shared_linear(v.bfloat16(), t.bfloat16() if mt else None, w, b, act,
                                 out_dtype=torch.float32)
        torch.cuda.synchronize()
        assert torch.equal(got[0], ref[0])
        assert not mt or torch.equal(got[1], ref[1])


# n that no 16-byte row piece covers (7: element stores in every type; 12: in the
# 16-bit ones), one 16-byte piece, and a split tail
@pytest.mark.parametrize("mv,mt,k,n", [(37, 5, 128, 7), (130, 3, 192, 12), (257, 3, 64, 8),
                                       (300, 40, 2560, 1000)])
@pytest.mark.parametrize("dtype", ["float32", "float16"])
def test_outputs_bias_and_entry_points(mv, mt, k, n, dtype):
    """Every output type, with and without a bias, through both entry points: the
    bits of the rounded activations given as bf16, and 16-bit outputs the
    rounding of the fp32 one."""
    import torch
    gen = torch.Generator(device="cuda").manual_seed(n)
    draw = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    dt = getattr(torch, dtype)
    xs = [draw(mv, k).to(dt), draw(mt, k).to(dt)]
    w, b = (0.02 * draw(n, k)).bfloat16(), 0.02 * draw(n)
    for bias in (b, None):
        full = capi.shared_linear(*xs, w, bias, out_dtype=torch.float32)
        for odt in (torch.float32, torch.bfloat16, torch.float16):
            ref = capi.shared_linear(*[x.bfloat16() for x in xs], w, bias, out_dtype=odt)
            for noalloc in (False, True):
                got = capi.shared_linear(*xs, w, bias, out_dtype=odt, noalloc=noalloc)
                for y, r, f in zip(got, ref, full):
                    assert torch.equal(y, r) and torch.equal(y, f.to(odt))


@pytest.mark.parametrize("dtype", ["float32", "float16"])
def test_capture_on_a_stream_that_nobody_owns(dtype):
    """A shape whose tail is split, captured before any call on the stream: the
    call needs no scratch there (none can be made under capture) and every
    replay is the rounded operands' product within the bound of an fp32 sum of k
    products, (k + 2) 2^-24 of the sum of their magnitudes."""
    import torch
    mv, k, n = 300, 2560, 1000
    gen = torch.Generator(device="cuda").manual_seed(8)
    draw = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    x, w, b = draw(mv, k).to(getattr(torch, dtype)), (0.02 * draw(n, k)).bfloat16(), 0.02 * draw(n)
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        y, _ = capi.shared_linear(x, None, w, b, out_dtype=torch.float32)
    wd = w.double().t().contiguous()
    for i in range(3):
        x.copy_(draw(mv, k))
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        xd = x.bfloat16().double()
        bound = (k + 2) * 2.0 ** -24 * (xd.abs() @ wd.abs() + b.abs().double())
        assert ((y.double() - (xd @ wd + b.double())).abs() <= bound).all()
