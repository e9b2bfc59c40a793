"""Launches with few rows: the kernels whose waves split the summed dimension (the library's pick
there), against the block kernels of the tile tables on the same inputs: row counts around tiles and
steps, every head dim, layouts, scales, both masks."""

import pytest
import torch

pytestmark = pytest.mark.gpu
U = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


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


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [16, 32, 64, 128])
@pytest.mark.parametrize("z,h,n", [(4, 8, 129), (3, 11, 160), (2, 16, 255), (1, 16, 257), (2, 5, 513), (1, 7, 1000), (1, 3, 2049)])
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
