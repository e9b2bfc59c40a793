"""The float32 kernels on split operands (the library's float32 picks) against float64 and against the
block kernels on the float32 matrix instruction, at row counts around tiles, blocks and steps of every
launch shape, in layouts, at scales and magnitudes, and with infinities."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu
BLOCKS = {"fwd": {"id": 0}, "bwd": {"dkdv": 0, "dq": 0}}


def _rand(shape, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(shape, device="cuda", generator=g)


def _exact(q, k, v, do, causal, scale):
    q, k, v, do = (t.double() for t in (q, k, v, do))
    s = torch.matmul(q, k.transpose(-1, -2).contiguous()) * scale
    if causal:
        s = s.masked_fill(torch.ones(s.shape[-2:], dtype=torch.bool, device=s.device).triu(1), -math.inf)
    p = torch.softmax(s, -1)
    o = torch.matmul(p, v)
    ds = (torch.matmul(do, v.transpose(-1, -2).contiguous()) - (do * o).sum(-1, keepdim=True)) * p * scale
    return o, torch.matmul(ds, k), torch.matmul(ds.transpose(-1, -2).contiguous(), q), \
        torch.matmul(p.transpose(-1, -2).contiguous(), do)


def _run(q, k, v, do, causal, scale, blocks):
    from tattn.api import _backward, _forward

    o, m = _forward(q, k, v, causal, scale, config=BLOCKS["fwd"] if blocks else None)
    return (o, *_backward(q, k, v, o, m, do, causal, scale, config=BLOCKS["bwd"] if blocks else None)), m


def _compare(q, k, v, do, causal, scale):
    """No further from float64 than the block kernels, up to a quarter and 2^-24 (both are a few
    roundings of 2^-24 per sum; the order differs)."""
    ref = _exact(q, k, v, do, causal, scale)
    got, m = _run(q, k, v, do, causal, scale, False)
    old, mb = _run(q, k, v, do, causal, scale, True)
    for name, a, b, r in zip(("o", "dq", "dk", "dv"), got, old, ref):
        size = r.norm().item()
        ea, eb = (a.double() - r).norm().item(), (b.double() - r).norm().item()
        assert ea <= 1.25 * eb + 2.0 ** -24 * size, (name, ea / size, eb / size)
    # |scores| and their float32 sums: a few units in the last place of the largest, in log2.
    assert (m - mb).abs().max().item() <= 1e-6 * (1 + mb.abs().max().item())
    again, _ = _run(q, k, v, do, causal, scale, False)
    assert all(torch.equal(a, b) for a, b in zip(got, again))


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [16, 32, 64, 128])
@pytest.mark.parametrize("z,h,n", [(2, 3, 2), (40, 16, 31), (40, 16, 33), (2, 3, 64), (40, 16, 65), (5, 7, 127),
                                   (32, 8, 129), (1, 5, 257), (16, 16, 260), (1, 16, 513), (3, 8, 1000)])
def test_split_kernels_against_float64(z, h, n, d, causal):
    _compare(*(_rand((z, h, n, d), n + s) for s in range(4)), causal, d ** -0.5)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [16, 32, 64, 128])
@pytest.mark.parametrize("z,h,n", [(65, 8, 4), (65, 8, 24), (33, 8, 33), (2, 3, 41), (100, 1, 146), (47, 1, 400), (16, 1, 1100)])
def test_split_kernels_at_the_edges_of_their_picks(z, h, n, d, causal):
    """Two slices per CU and short rows; around one workgroup per CU at head dim 128."""
    from tattn import _lib

    for kernel in (_lib.K_FWD, _lib.K_BWD_DKDV, _lib.K_BWD_DQ):
        assert (_lib.picked(kernel, (z, h, n, d), _lib.F32, causal) == _lib.PICK_PLANES) == (d < 128 or n > 96)
    _compare(*(_rand((z, h, n, d), n + s) for s in range(4)), causal, d ** -0.5)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("scale", [-0.125, 0.0, 0.5])
def test_scales(scale, causal):
    _compare(*(_rand((2, 8, 300, 64), 50 + s) for s in range(4)), causal, scale)


@pytest.mark.parametrize("causal", [False, True])
def test_layouts(causal):
    """Token-major, interleaved, and broadcast key / value views."""
    _compare(*(_rand((2, 200, 8, 64), 70 + s).transpose(1, 2) for s in range(4)), causal, 0.125)
    _compare(*(t.transpose(1, 2) for t in _rand((2, 200, 4, 8, 64), 80).unbind(2)), causal, 0.125)
    q, do = (_rand((2, 8, 200, 64), 90 + s) for s in range(2))
    k, v = (_rand((1, 1, 200, 64), 95 + s).expand(2, 8, 200, 64) for s in range(2))
    _compare(q, k, v, do, causal, 0.125)


@pytest.mark.parametrize("mag", [(1e-18, 1e18, 1.0, 1.0), (1.0, 1.0, 1e-37, 1.0), (1.0, 1.0, 1.0, 1e-36),
                                 (1e-3, 1e3, 1e30, 1e-30), (1.0, 1.0, 1e36, 1e-20)])
def test_magnitudes(mag):
    """Values near both ends of the exponent range: no precision is lost to the planes' own range."""
    _compare(*(_rand((2, 4, 150, 64), 100 + s) * x for s, x in enumerate(mag)), False, 0.125)


@pytest.mark.parametrize("n", [40, 200, 600])
@pytest.mark.parametrize("causal", [False, True])
def test_infinities_and_nans_go_where_the_block_kernels_take_them(causal, n):
    _infinities_and_nans(2, n, causal)


@pytest.mark.parametrize("n", [31, 60])
@pytest.mark.parametrize("causal", [False, True])
def test_infinities_and_nans_in_short_rows(causal, n):
    _infinities_and_nans(65, n, causal)


def _infinities_and_nans(z, n, causal):
    q, k, v, do = (_rand((z, 8, n, 64), 30 + s) for s in range(4))
    q[0, 1, 17, 5] = float("nan")
    k[0, 2, 3, 7] = float("-inf")  # hides key 3 from queries whose component is positive
    v[0, 3, 9, 11] = float("inf")
    v[1, 1, 6, 0] = float("nan")
    do[1, 2, 8, 1] = float("inf")
    v[1, 3, 1, 2] = 3e35
    got, m = _run(q, k, v, do, causal, 0.125, False)
    old, mb = _run(q, k, v, do, causal, 0.125, True)
    for a, b in zip((*got, m), (*old, mb)):
        assert torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(torch.isinf(a), torch.isinf(b))
        ok = torch.isfinite(b)
        assert torch.equal(torch.sign(a[~ok & ~torch.isnan(b)]), torch.sign(b[~ok & ~torch.isnan(b)]))
    assert torch.isfinite(got[0][0, 2][q[0, 2, :, 7] > 0]).all()


def test_overlapping_rows_take_the_block_kernels():
    """Keys that all share one row (row stride 0) are the block kernels' case: same bits."""
    from tattn.api import _forward

    q = _rand((2, 4, 100, 64), 1)
    k, v = (_rand((2, 4, 1, 64), 2 + s).expand(2, 4, 100, 64) for s in range(2))
    got, want = _forward(q, k, v, False, 0.125), _forward(q, k, v, False, 0.125, config={"id": 0})
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def _hidden_keys(shape, causal, scale, hide, low, q0):
    """q, k, v whose keys in `hide` score q0 * low on top; the forward's O and M against float64: scores of
    visible keys are sums of D products and rows sums of up to N, each a rounding of 2^-24, in the norm."""
    from tattn.api import _forward

    z, h, n, d = shape
    q, k, v = (_rand(shape, 200 + s) for s in range(3))
    q[..., 0] = q0
    k[..., 0] = 0.0
    k[:, :, hide, 0] = low
    s = torch.matmul(q.double(), k.double().transpose(-1, -2).contiguous()) * scale
    if low == -math.inf:
        s[..., hide] = -math.inf
    s = torch.where(s < -1e37, torch.full_like(s, -math.inf), s)  # below float32's range (or hidden by far)
    if causal:
        s = s.masked_fill(torch.ones(n, n, dtype=torch.bool, device="cuda").triu(1), -math.inf)
    seen = (s > -1e6).any(-1)  # rows with a visible key
    assert seen.float().mean() > 0.4
    want = torch.matmul(torch.softmax(s, -1), v.double())
    o, m = _forward(q, k, v, causal, scale)
    assert torch.isfinite(o[seen]).all() and torch.isfinite(m[seen]).all()
    bound = 4 * math.sqrt(n + d) * 2.0 ** -24
    assert (o.double() - want)[seen].norm().item() <= bound * want[seen].norm().item()
    assert (m.double() - torch.logsumexp(s, -1) / math.log(2))[seen].abs().max().item() <= 1e-6 * (1 + m[seen].abs().max().item())


# Waves per row tile and tiles per step: {2, 4}, {4, 2}, {4, 1}, {1, 1}; head dim 128 {2, 2}, {4, 1}.
SHAPES = [(2, 4, 128, 64), (4, 16, 512, 64), (40, 16, 512, 64), (65, 8, 30, 32), (1, 8, 600, 128), (16, 16, 600, 128)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("low", [-1e10, -1e20, -1e30, -3.4028234663852886e38, -math.inf])
@pytest.mark.parametrize("side", ["right", "left", "middle"])
def test_keys_hidden_by_very_low_scores(shape, causal, low, side):
    """Padding written into one component of k: whole tiles, so that a wave sees hidden keys first, last or only."""
    n = shape[2]
    edge = min(32, n // 2)
    hide = {"right": slice(edge, n), "left": slice(0, n // 2), "middle": slice(edge, n - edge // 2)}[side]
    _hidden_keys(shape, causal, 0.125, hide, low, 1.0)


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("causal", [False, True])
def test_infinitely_low_scores_of_some_rows_leave_the_others(shape, causal):
    """Even rows overflow to -inf on the hidden keys, odd rows (q = 2^-126 there) score a few below zero."""
    n = shape[2]
    q0 = torch.tensor([16.0, 2.0 ** -126], device="cuda").repeat((n + 1) // 2)[:n]
    for hide in (slice(0, n // 2), slice(min(32, n // 2), n)):
        _hidden_keys(shape, causal, 0.125, hide, -3e38, q0)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [16, 32, 64])
@pytest.mark.parametrize("n", [2, 3, 5, 40])
def test_short_sums_are_no_further_from_float64_than_the_block_kernels(n, d, causal):
    """Where few products are summed, what a product loses shows. 512 slices: the norm of 16,000 errors or
    more has a spread of about 0.6%, so 3% covers the difference of two of them."""
    q, k, v, do = (_rand((64, 8, n, d), 300 + s) for s in range(4))
    ref = _exact(q, k, v, do, causal, d ** -0.5)
    got, _ = _run(q, k, v, do, causal, d ** -0.5, False)
    old, _ = _run(q, k, v, do, causal, d ** -0.5, True)
    for name, a, b, r in zip(("o", "dq", "dk", "dv"), got, old, ref):
        ea, eb = (a.double() - r).norm().item(), (b.double() - r).norm().item()
        assert ea <= 1.03 * eb, (name, ea / eb)


@pytest.mark.parametrize("which", range(4))
def test_numbers_beyond_the_largest_bf16(which):
    """3.4e38 is finite in float32 and rounds to infinity in bf16."""
    t = [_rand((2, 4, 150, 64), 400 + s) * 1e-3 for s in range(4)]
    t[which] = t[which].clone()
    t[which][0, 1, 40:44, 3] = 3.4e38
    t[(1, 0, 3, 2)[which]][..., 3] = 0.0  # its partner in the products: everything stays finite
    q, k, v, do = t
    ref = _exact(q, k, v, do, False, 0.125)
    got, _ = _run(q, k, v, do, False, 0.125, False)
    old, _ = _run(q, k, v, do, False, 0.125, True)
    for name, a, b, r in zip(("o", "dq", "dk", "dv"), got, old, ref):
        assert torch.equal(torch.isfinite(a), torch.isfinite(b)), name
        ok = torch.isfinite(b) & (r.abs() < 3e38)
        ea, eb, size = ((a.double() - r)[ok].norm().item(), (b.double() - r)[ok].norm().item(), r[ok].norm().item())
        assert ea <= 1.25 * eb + 2.0 ** -24 * size, (name, ea / size, eb / size)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("mag", [(1.0, 1.0, 1.0, 1e-13), (1.0, 1.0, 1.0, 1e-25), (1.0, 1.0, 1e-14, 1e-14), (1.0, 1.0, 1e-17, 1e-18),
                                 (1e-20, 1e20, 1e-28, 1.0), (1.0, 1.0, 1e-15, 3e-21)])
def test_small_magnitudes(mag, d, causal):
    """Loss gradients of ordinary and of very small size (dS down to 1e-38, where planes lose bits)."""
    _compare(*(_rand((2, 4, 150, d), 500 + s) * x for s, x in enumerate(mag)), causal, d ** -0.5)


def test_tiny_rows_beside_ordinary_ones():
    """Every fourth row of dO at 2^e of the others: the others keep what the block kernels give. The dS of a tiny
    row are about 2^e * 8 / 150 (dP of 64 products, P of 150 keys), or 2^(e - 4.2), and held to 2^-134: its dQ has a
    relative error of at most 2^(-129 - e), or that of float32 sums (2^-21)."""
    q, k, v, do = (_rand((2, 4, 150, 64), 600 + s) for s in range(4))
    ordinary = torch.arange(150, device="cuda") % 4 != 0
    for e in (-95, -105, -115, -125):
        rel = max(2.0 ** -21, 2.0 ** (-129 - e))
        w = torch.where(ordinary, 1.0, 2.0 ** e)[:, None]
        t = (q, k, v, do * w)
        ref = _exact(*t, False, 0.125)
        got, _ = _run(*t, False, 0.125, False)
        old, _ = _run(*t, False, 0.125, True)
        for name, a, b, r in zip(("o", "dq", "dk", "dv"), got, old, ref):
            ea, eb = ((x.double() - r)[:, :, ordinary].norm().item() for x in (a, b))
            assert ea <= 1.25 * eb + 2.0 ** -24 * r.norm().item(), (e, name)
        tiny = ref[1][:, :, ~ordinary]
        assert (got[1].double()[:, :, ~ordinary] - tiny).norm().item() <= rel * tiny.norm().item(), e


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("layout", ["one row", "rows 16 MiB apart", "tokens"])
def test_both_directions_run_kernels_with_the_same_scores(layout, causal):
    """Keys and values that the forward leaves to the block kernels while the backward's contiguous copies
    would pass for the split ones, at scores of thousands, where M has to match the scores to their last bit:
    attention's gradients are those of the block kernels given O and M."""
    from tattn import _lib, attention
    from tattn.api import _backward, _forward

    n = 16 if layout == "rows 16 MiB apart" else 200
    q, do = _rand((1, 4, n, 64), 1) * 30, _rand((1, 4, n, 64), 2)
    if layout == "one row":
        k, v = ((_rand((1, 4, 1, 64), 3 + s) * (30, 1)[s]).expand(1, 4, n, 64) for s in range(2))
    elif layout == "tokens":
        k, v = (_rand((1, n, 4, 64), 3 + s).transpose(1, 2) for s in range(2))
    else:
        k, v = (torch.empty_strided((1, 4, n, 64), (0, 64, 1 << 22, 1), device="cuda").copy_(_rand((1, 4, n, 64), 3 + s)) for s in range(2))
    blocks = _lib.picked(_lib.K_FWD, (1, 4, n, 64), _lib.F32, causal, strides=k.stride(), v_strides=v.stride()) == 0
    assert blocks == (layout != "tokens")
    t = [x.detach().requires_grad_() for x in (q, k, v)]
    got = torch.autograd.grad(attention(*t, causal=causal), t, do)
    o, m = _forward(q, k, v, causal, 0.125)
    want = _backward(q, k, v, o, m, do, causal, 0.125, config={"dkdv": 0, "dq": 0} if blocks else None)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
