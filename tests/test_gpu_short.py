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
