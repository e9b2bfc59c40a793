"""Short rows (N <= 128, 16-bit): the kernels that hold whole slices in LDS, at the edges of their
tiles (32 rows, 64, 128) and of a workgroup's slices, against the block kernels and float32."""

import pytest
import torch

from oracle.reference import naive_attention

pytestmark = pytest.mark.gpu
NS = [1, 24, 31, 32, 33, 63, 64, 65, 96, 97, 127, 128]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [16, 32, 64, 128])
@pytest.mark.parametrize("n", NS)
def test_short_rows_match_the_block_kernels(n, d, causal, dtype):
    """Gradients are those of the pipelined entries bit for bit (same chains and orders, from the
    same O and M); O and M agree to a rounding of P (the row max may differ) and O with float32."""
    from tattn.api import _backward, _forward

    g = torch.Generator(device="cuda").manual_seed(1000 * d + n)
    z, h = (1, 3) if n > 32 else (1, 5)  # spare waves in the last workgroup
    q, k, v, do = (torch.randn((z, h, n, d), device="cuda", dtype=dtype, generator=g) for _ in range(4))
    scale = d ** -0.5
    o, m = _forward(q, k, v, causal, scale)
    ob, mb = _forward(q, k, v, causal, scale, config={"id": 0})
    # One rounding of each P (half an ulp, relative) and of O itself, on values up to |v|'s maximum.
    u = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    bound = 3 * u * v.float().abs().max().item()
    assert (o.float() - ob.float()).abs().max().item() <= bound
    assert (m - mb).abs().max().item() <= 2 * u / 0.69
    ref = naive_attention(q.float(), k.float(), v.float(), causal=causal)
    assert (o.float() - ref).abs().max().item() <= bound
    got = _backward(q, k, v, o, m, do, causal, scale)
    want = _backward(q, k, v, o, m, do, causal, scale, config={"dkdv": 0, "dq": 0})
    for name, a, b in zip(("dq", "dk", "dv"), got, want):
        assert torch.equal(a, b), name


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [16, 32, 64, 128])
@pytest.mark.parametrize("n", NS)
def test_short_forward_gives_the_bits_of_the_block_kernels(n, d, causal, dtype):
    """Scores of ordinary size (N(0, 1) scaled by 1/sqrt(d)): the same max in the exponent, the same rounded
    P and the same order of sums as the block kernels, so O and M are theirs exactly."""
    from tattn.api import _forward

    g = torch.Generator(device="cuda").manual_seed(2000 * d + n)
    q, k, v = (torch.randn((2, 3, n, d), device="cuda", dtype=dtype, generator=g) for _ in range(3))
    o, m = _forward(q, k, v, causal, d ** -0.5)
    ob, mb = _forward(q, k, v, causal, d ** -0.5, config={"id": 0})
    assert torch.equal(o, ob) and torch.equal(m, mb)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("low", [-8.0, -40.0, -3000.0, float("-inf")])
def test_short_rows_whose_first_tile_scores_far_below_the_rest(low, causal, dtype):
    """Keys 0-31 hidden by one component of k (left padding; its product with q is 8 low, exact in both types):
    rows that see later keys take their max from those. O against float64: one rounding of each P and of
    O (u relative each, |v| bounds the values)."""
    from tattn.api import _forward

    n, scale = 100, 0.125
    g = torch.Generator(device="cuda").manual_seed(7)
    q, k, v = (torch.randn((2, 3, n, 64), device="cuda", dtype=dtype, generator=g) for _ in range(3))
    q[..., 0] = 8.0
    k[..., 0] = 0.0
    k[:, :, :32, 0] = low
    o, m = _forward(q, k, v, causal, scale)
    s = torch.matmul(q.double(), k.double().transpose(-1, -2).contiguous()) * scale
    if causal:
        s = s.masked_fill(torch.ones(n, n, dtype=torch.bool, device="cuda").triu(1), float("-inf"))
    want = torch.matmul(torch.softmax(s, -1), v.double())
    rows = slice(32 if causal else 0, n)  # causal: earlier rows see hidden keys only
    u = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    assert (o.double() - want)[:, :, rows].abs().max().item() <= 3 * u * v.float().abs().max().item()
    assert (m.double() - torch.logsumexp(s, -1) / 0.6931471805599453)[:, :, rows].abs().max().item() <= 2 * u / 0.69


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [16, 32, 64, 128])
@pytest.mark.parametrize("n", [24, 70, 128])
def test_whole_short_backward_matches_three_launches(n, d, causal, dtype):
    """tattn_bwd in one launch against preprocess, dK/dV and dQ with the library's picks: same bits, delta included."""
    from tattn import _lib
    from tattn.api import _DTYPES, _forward

    z, h, scale = 2, 5, d ** -0.5
    g = torch.Generator(device="cuda").manual_seed(3000 * d + n)
    q, k, v, do = (torch.randn((z, h, n, d), device="cuda", dtype=dtype, generator=g) for _ in range(4))
    o, m = _forward(q, k, v, causal, scale)
    lib, code, st = _lib.load(), _DTYPES[dtype], _lib.strides4(q)
    stream = torch.cuda.current_stream().cuda_stream
    args = (st, z, h, n, d, code, int(causal), scale, -1, stream)
    one, three = ([torch.empty_like(q) for _ in range(3)] + [torch.empty_like(m)] for _ in range(2))
    p = [t.data_ptr() for t in (q, k, v, o, do, m)]
    _lib.check(lib.tattn_bwd(*p[:5], *(t.data_ptr() for t in one[:3]), p[5], one[3].data_ptr(), *args), "tattn_bwd")
    dq, dk, dv, delta = (t.data_ptr() for t in three)
    _lib.check(lib.tattn_bwd_preprocess(p[3], p[4], delta, st, z, h, n, d, code, stream), "tattn_bwd_preprocess")
    _lib.check(lib.tattn_bwd_dkdv(p[0], p[1], p[2], p[4], dk, dv, p[5], delta, *args), "tattn_bwd_dkdv")
    _lib.check(lib.tattn_bwd_dq(p[0], p[1], p[2], p[4], dq, p[5], delta, *args), "tattn_bwd_dq")
    for name, a, b in zip(("dq", "dk", "dv", "delta"), one, three):
        assert torch.equal(a, b), name
