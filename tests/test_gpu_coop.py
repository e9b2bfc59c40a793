"""Launches with few rows: the kernels whose waves split the summed dimension (the library's pick
there), against the block kernels of the tile tables on the same inputs: row counts around tiles and
steps, every head dim, layouts, scales, both masks."""

import pytest
import torch

pytestmark = pytest.mark.gpu
U = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}
STRESS = [(1, 16, 200, 64), (1, 8, 1024, 64), (2, 8, 500, 64)]


def _rand(shape, dtype, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(shape, device="cuda", dtype=dtype, generator=g)


def _compare(q, k, v, do, causal, scale):
    """O within one rounding of every P and of itself (u relative each, |v| at most 6 here), M
    within P's rounding in log2; gradients of one (O, M): the same rounded P and dS summed in float32
    in another order, so one rounding at the store plus float32 noise."""
    from tattn.api import _backward, _forward

    u = U[q.dtype]
    o, m = _forward(q, k, v, causal, scale)
    ob, mb = _forward(q, k, v, causal, scale, config={"id": 1})
    assert (o.float() - ob.float()).abs().max().item() <= 3 * u * v.float().abs().max().item()
    assert (m - mb).abs().max().item() <= 2 * u / 0.69
    got = _backward(q, k, v, o, m, do, causal, scale)
    want = _backward(q, k, v, o, m, do, causal, scale, config={"dkdv": 0, "dq": 0})
    for name, a, b in zip(("dq", "dk", "dv"), got, want):
        a, b = a.float(), b.float()
        assert ((a - b).abs() <= 2 * u * b.abs() + 1e-5 * (1 + b.abs().max())).all(), name
    again = _backward(q, k, v, o, m, do, causal, scale)
    assert all(torch.equal(a, b) for a, b in zip(got, again))
    assert torch.equal(_forward(q, k, v, causal, scale, save_lse=False)[0], o)


SHAPES = [(4, 8, 129), (3, 11, 160), (2, 16, 255), (1, 16, 257), (2, 5, 513), (1, 7, 1000), (1, 3, 2049)]


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [16, 32, 64, 128])
def test_the_shapes_below_run_these_kernels(d, causal):
    """Forward and dQ everywhere but at 129 rows of head dim 64; dK/dV (which head dim 128 does not have) from 257
    rows on, and on short rows of head dims 16 and 32. Layouts, scales (the forward but at 0) and stress as well."""
    from tattn import _lib

    def coop(kernel, shape, **kw):
        return _lib.picked(kernel, shape, _lib.F16, causal, **kw) == _lib.PICK_COOP

    for z, h, n in SHAPES:
        if (n, d) != (129, 64):
            assert coop(_lib.K_FWD, (z, h, n, d)) and coop(_lib.K_BWD_DQ, (z, h, n, d))
        if d < 128 and (n >= 257 or d < 64):
            assert coop(_lib.K_BWD_DKDV, (z, h, n, d))
    for kernel in (_lib.K_FWD, _lib.K_BWD_DQ, _lib.K_BWD_DKDV):
        assert coop(kernel, (2, 8, 400, 64))
        assert coop(kernel, (2, 8, 400, 64), scale=0.0) == (kernel != _lib.K_FWD)
        assert all(coop(kernel, shape) for shape in STRESS[1:])
    assert all(coop(_lib.K_FWD, shape) for shape in (*STRESS, (2, 16, 200, 64)))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [16, 32, 64, 128])
@pytest.mark.parametrize("z,h,n", SHAPES)
def test_coop_kernels_match_the_block_kernels(z, h, n, d, causal, dtype):
    q, k, v, do = (_rand((z, h, n, d), dtype, n + s) for s in range(4))
    _compare(q, k, v, do, causal, d ** -0.5)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("scale", [-0.125, 0.0, 0.5])
def test_coop_scales(scale, causal):
    q, k, v, do = (_rand((2, 8, 400, 64), torch.float16, 50 + s) for s in range(4))
    _compare(q, k, v, do, causal, scale)


@pytest.mark.parametrize("causal", [False, True])
def test_coop_layouts(causal):
    """Token-major, interleaved, and broadcast key / value views."""
    tok = [_rand((2, 400, 8, 64), torch.float16, 70 + s).transpose(1, 2) for s in range(4)]
    _compare(*tok, causal, 0.125)
    packed = _rand((2, 400, 4, 8, 64), torch.float16, 80)
    _compare(*(t.transpose(1, 2) for t in packed.unbind(2)), causal, 0.125)
    q, do = (_rand((2, 8, 400, 64), torch.float16, 90 + s) for s in range(2))
    k, v = (_rand((1, 1, 400, 64), torch.float16, 95 + s).expand(2, 8, 400, 64) for s in range(2))
    _compare(q, k, v, do, causal, 0.125)


@pytest.mark.parametrize("causal", [False, True])
def test_coop_infinite_and_nan_scores_stay_in_their_rows(causal):
    from tattn.api import _forward

    q, k, v = (_rand((2, 16, 200, 64), torch.float16, 30 + s) for s in range(3))
    q[0, 1, 77, 5] = float("nan")
    q[1, 2, 130] = 60000.0  # overflows to infinite scores
    o, m = _forward(q, k, v, causal, 0.125)
    ob, mb = _forward(q, k, v, causal, 0.125, config={"id": 1})
    assert torch.equal(torch.isfinite(o), torch.isfinite(ob)) and torch.equal(torch.isfinite(m), torch.isfinite(mb))
    assert torch.isnan(o[0, 1, 77]).all() and torch.isfinite(o[0, 0]).all()


def _exact(q, k, v, do, causal, scale):
    q, k, v, do = (t.double() for t in (q, k, v, do))
    s = torch.matmul(q, k.transpose(-1, -2).contiguous()) * scale
    if causal:
        s = s.masked_fill(torch.ones(s.shape[-2:], dtype=torch.bool, device=s.device).triu(1), float("-inf"))
    p = torch.softmax(s, -1)
    o = torch.matmul(p, v)
    ds = (torch.matmul(do, v.transpose(-1, -2).contiguous()) - (do * o).sum(-1, keepdim=True)) * p * scale
    grads = torch.matmul(ds, k), torch.matmul(ds.transpose(-1, -2).contiguous(), q), \
        torch.matmul(p.transpose(-1, -2).contiguous(), do)
    return o, torch.logsumexp(s, -1) / 0.6931471805599453, grads


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("z,h,n,d", [(2, 16, 255, 32), (1, 16, 300, 64), (1, 7, 1000, 64), (1, 7, 1000, 128), (1, 3, 2049, 16)])
def test_coop_gradients_are_no_further_from_float64(z, h, n, d, causal, dtype):
    """Whole pipeline against float64, beside the block kernels': the same rounded operands in another order
    of sums. The errors are those of 50,000 and more roundings, so the norms of two sets agree to about 1%."""
    from tattn.api import _backward, _forward

    q, k, v, do = (_rand((z, h, n, d), dtype, 700 + s) for s in range(4))
    scale = d ** -0.5
    o, m = _forward(q, k, v, causal, scale)
    ob, mb = _forward(q, k, v, causal, scale, config={"id": 1})
    got = (o, *_backward(q, k, v, o, m, do, causal, scale))
    old = (ob, *_backward(q, k, v, ob, mb, do, causal, scale, config={"dkdv": 0, "dq": 0}))
    ref_o, _, grads = _exact(q, k, v, do, causal, scale)
    for name, a, b, r in zip(("o", "dq", "dk", "dv"), got, old, (ref_o, *grads)):
        assert (a.double() - r).norm().item() <= 1.02 * (b.double() - r).norm().item(), name


def _stress(kind, shape, dtype):
    """The softmax stress test's inputs over more heads: near one-hot rows, a row max that rises (or falls)
    with every key block, rows of very different magnitude."""
    z, h, n, d = shape
    g = torch.Generator().manual_seed(123 + n)
    q, k, v, do = (torch.randn(shape, generator=g) for _ in range(4))
    if kind == "peaked":
        q, k = 10 * q, 10 * k
    elif kind in ("rising", "falling"):
        u = torch.randn(d, generator=g)
        u = u / u.norm()
        ramp = torch.linspace(-6.0, 6.0, n) * (1 if kind == "rising" else -1)
        q = 4.0 * u.expand(shape).clone()
        k = k * 0.1 + ramp[None, None, :, None] * u * 2.0
    else:
        q = q * torch.logspace(-2, 1.3, n)[None, None, :, None]
    return [t.to("cuda", dtype) for t in (q, k, v, do)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("kind", ["peaked", "rising", "falling", "mixed"])
@pytest.mark.parametrize("shape", STRESS, ids=lambda s: "x".join(map(str, s)))
def test_coop_softmax_stress(shape, kind, causal, dtype):
    """Per wave: the seed from tile 0, the sum check, the rescale and its undo, and the merge of waves whose
    maxima differ. O within one rounding of every P and of itself and M within P's rounding of float64;
    gradients against the reference's algorithm on the same O and M, each element within one flip of every rounded
    P or dS that it sums (two half ulps of each), one rounding at the store and float32 noise. That allowance is
    per element; a flat one is no property of a kernel here: over 8 x 1,024 peaked rows the block
    kernels exceed the flat allowance of the 2 x 1,024 test as well (by 2.0e-3 in fp16)."""
    from helpers import emulated_backward
    from tattn.api import _backward, _forward

    q, k, v, do = _stress(kind, shape, dtype)
    u, scale = U[dtype], 0.125
    o, m = _forward(q, k, v, causal, scale)
    ref_o, ref_m, _ = _exact(q, k, v, do, causal, scale)
    assert (o.double() - ref_o).abs().max().item() <= 3 * u * v.float().abs().max().item()
    # float32 scores of 64 products each: a few units in the last place of the largest on top.
    assert (m.double() - ref_m).abs().max().item() <= 2 * u / 0.69 + 4e-7 * ref_m.abs().max().item()
    got = _backward(q, k, v, o, m, do, causal, scale)
    want, flips = emulated_backward(q, k, v, o, m, do, causal, scale)
    for name, a, b, f in zip(("dq", "dk", "dv"), got, want, flips):
        assert ((a.float() - b).abs() <= f + u * b.abs() + 1e-5 * (1 + b.abs().max())).all(), name
