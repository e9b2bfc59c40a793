"""The backward on inputs read where they lie: which layouts take that route (CPU), and that it
gives the bits of contiguous copies (GPU)."""

import pytest
import torch

from tattn.api import _one_layout


def _tok(z, h, n, d, dtype=torch.float16, device="cpu"):
    return torch.empty(z, n, h, d, dtype=dtype, device=device).transpose(1, 2)


def test_one_layout_rule():
    a, b = _tok(2, 3, 20, 32), _tok(2, 3, 20, 32)
    assert _one_layout(a, b) and _one_layout(a.contiguous(), b.contiguous())
    assert not _one_layout(a, b.contiguous())  # two layouts
    packed = torch.empty(2, 20, 3, 3, 32, dtype=torch.float16)  # q, k, v interleaved per token
    q, k, v = (t.transpose(1, 2) for t in packed.unbind(2))
    assert _one_layout(q, k, v) and not _one_layout(q, a)
    assert not _one_layout(*(torch.empty(2, 3, 32, 20, dtype=torch.float16).transpose(2, 3) for _ in range(2)))  # d stride
    odd = torch.empty(2, 3, 20, 36, dtype=torch.float16)[..., :32]  # rows 72 bytes apart
    assert not _one_layout(odd, odd)
    off = torch.empty(2 * 3 * 20 * 32 + 1, dtype=torch.float16)[1:].view(2, 3, 20, 32)  # base off by 2 bytes
    assert not _one_layout(a.contiguous(), off)
    wide = torch.empty_strided((1, 1, 1024, 64), (0, 0, 1 << 20, 1), dtype=torch.float16, device="meta")  # 2 GiB slices
    assert not _one_layout(wide, wide)
    row = torch.empty(2, 3, 1, 32, dtype=torch.float16).expand(2, 3, 20, 32)  # one row, 20 times
    assert not _one_layout(row, row)
    window = torch.empty(2, 3, 20 * 16 + 16, dtype=torch.float16).unfold(2, 32, 16)  # rows that share halves
    assert window.stride(2) == 16 and not _one_layout(window, window)


@pytest.mark.gpu
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", [(2, 3, 33, 16), (2, 3, 161, 32), (2, 4, 512, 64), (1, 3, 700, 64), (1, 2, 257, 128)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("packed", [False, True])
def test_backward_in_place_gives_the_bits_of_copies(shape, dtype, causal, packed):
    """Token-major views, and views of one buffer that holds all five tensors side by side (rows
    that are 5 h d apart), against contiguous inputs: rows past the end of the sequence, ragged
    and whole blocks, every kernel family."""
    from tattn.api import _backward, _forward

    z, h, n, d = shape
    g = torch.Generator(device="cuda").manual_seed(n + d)
    q, k, v, do = (torch.randn(shape, device="cuda", dtype=dtype, generator=g) for _ in range(4))
    scale = d ** -0.5
    o, m = _forward(q, k, v, causal, scale)
    want = _backward(q, k, v, o, m, do, causal, scale)
    buf = torch.full((z, n, 5 if packed else 1, h, d), float("nan"), device="cuda", dtype=dtype)
    views = []
    for i, t in enumerate((q, k, v, o, do)):
        dst = buf[:, :, i] if packed else torch.empty((z, n, h, d), device="cuda", dtype=dtype)
        dst.copy_(t.transpose(1, 2))
        views.append(dst.transpose(1, 2))
    qv, kv, vv, ov, dov = views
    assert _one_layout(*views) and not qv.is_contiguous()
    got = _backward(qv, kv, vv, ov, m, dov, causal, scale)
    for name, a, b in zip(("dq", "dk", "dv"), got, want):
        assert a.is_contiguous() and torch.equal(a, b), name


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("stride", [0, 16])
@pytest.mark.parametrize("n,d", [(1, 64), (20, 32), (100, 64), (300, 64), (513, 32), (200, 128)])
def test_overlapping_rows(n, d, stride, dtype):
    """All five inputs as rows that overlap (one row n times; rows 16 elements apart): rows past the end
    of the sequence hold data there. `_backward` copies them; the library call runs its generic kernels
    (4 waves, 32 rows per step) on them as they are. Each gives the bits of contiguous copies."""
    from tattn import _lib
    from tattn.api import _DTYPES, _backward, _forward

    z, h, scale = 2, 3, 0.125
    g = torch.Generator(device="cuda").manual_seed(n + d + stride)
    span = (n - 1) * stride + d
    views = [torch.randn(z * h * span, device="cuda", generator=g).to(dtype).as_strided((z, h, n, d), (h * span, span, stride, 1))
             for _ in range(5)]
    copies = [t.contiguous().clone() for t in views]
    _, m = _forward(copies[0], copies[1], copies[2], False, scale)
    # float32: the forward leaves such keys to the block kernels, and the backward follows it there.
    blocks = {"dkdv": 0, "dq": 0} if dtype == torch.float32 else None
    want = _backward(copies[0], copies[1], copies[2], copies[3], m, copies[4], False, scale, config=blocks)
    got = _backward(views[0], views[1], views[2], views[3], m, views[4], False, scale)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    grads = [torch.empty_like(copies[0]) for _ in range(3)]
    delta = torch.empty_like(m)
    rc = _lib.load().tattn_bwd_layouts(*(t.data_ptr() for t in (*views, *grads, m, delta)), _lib.strides4(views[0]),
                                       _lib.strides4(copies[0]), z, h, n, d, _DTYPES[dtype], 0, scale, -1,
                                       torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    generic = {"dkdv": {"kind": 0, "block_n": 128, "block_m": 32}, "dq": {"kind": 0, "block_m": 128, "block_n": 32}}
    want = _backward(copies[0], copies[1], copies[2], copies[3], m, copies[4], False, scale, config=generic)
    for name, a, b in zip(("dq", "dk", "dv"), grads, want):
        assert torch.equal(a, b), name
