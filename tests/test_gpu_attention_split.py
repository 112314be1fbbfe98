"""Attention whose last round of few workgroups is split over the keys (selas_attention_split): against
softmax(q k^T / sqrt(128)) v in 64 bits (bf16 probabilities and output: max abs 1e-2 of the largest value, relative L2
4e-3, as without a split), with the items of the full rounds bit-equal to selas_attention_v, at ranges that end inside
a key tile, in strided outputs, with a range whose scores are all -inf, and in a captured graph.
"""

from __future__ import annotations

import ctypes

import pytest
import torch

from selas_amd import _lib
from selas_amd.attention import attention

from .conftest import seeded

pytestmark = pytest.mark.gpu


def inputs(b, h, l, seed):
    g = seeded(seed)
    return tuple(torch.randn(b, h, l, 128, generator=g).to(torch.bfloat16).cuda() for _ in range(3))


def workspace(b, h, l):
    n = ctypes.c_int64()
    _lib.call("selas_attention_workspace_bytes", b, h, l, ctypes.byref(n))
    return n.value


def unsplit(q, k, v):
    b, h, l, d = q.shape
    y = torch.empty(b, l, h * d, dtype=q.dtype, device="cuda")
    _lib.call("selas_attention_v", q.data_ptr(), k.data_ptr(), v.data_ptr(), b, h, l, d, y.data_ptr(), h * d, _lib.BF16,
              _lib.stream(q.device))
    return y


def check(y, q, k, v, i, j):
    s = torch.softmax(q[i, j].double() @ k[i, j].double().t() / 128 ** 0.5, -1) @ v[i, j].double()
    d = y[i, :, j * 128:(j + 1) * 128].double() - s
    assert d.abs().max() <= 1e-2 * s.abs().max() and d.norm() <= 4e-3 * s.norm()


# 264 and 528 items of 256 queries (8 and 16 split, partial last key tiles), 257 (the fewest: one, of 20 queries).
@pytest.mark.parametrize("b,h,l", [(1, 24, 2816), (1, 24, 2700), (2, 24, 2785), (1, 257, 256), (1, 1, 65556)])
def test_against_64_bits_and_the_unsplit_call(b, h, l):
    cu = torch.cuda.get_device_properties(0).multi_processor_count
    q, k, v = inputs(b, h, l, b + h + l)
    wide = torch.zeros(b, l, h * 128 + 64, dtype=torch.bfloat16, device="cuda")
    y = attention(q, k, v, out=wide[..., :h * 128])
    u = unsplit(q, k, v)
    assert torch.count_nonzero(wide[..., h * 128:]) == 0
    if cu == 256 and l > 256:
        assert workspace(b, h, l) > 0
    if not workspace(b, h, l):
        assert torch.equal(y, u)
    items = -(-l // 256)
    whole = b * h * items // cu * cu if workspace(b, h, l) else b * h * items
    i, j, t = whole // items // h, whole // items % h, whole % items  # the first split item
    if whole < b * h * items:
        assert torch.equal(y[i, :256 * t, j * 128:(j + 1) * 128], u[i, :256 * t, j * 128:(j + 1) * 128])
    if l < 4096:
        check(y, q, k, v, b - 1, h - 1)
        check(y, q, k, v, min(i, b - 1), j if i < b else h - 1)
    d = (y.double() - u.double())[:, -min(l, 512):, -128:]  # the last head's end: split
    assert d.norm() <= 4e-3 * u.double()[:, -min(l, 512):, -128:].norm()


# Lengths that are cut (2816, 3000, 5400 tokens), and one that fills no round alone but one and an eighth in pairs.
@pytest.mark.parametrize("b,h,l", [(2, 24, 1536), (3, 24, 2816), (4, 24, 3000), (2, 24, 5400), (3, 32, 2561), (2, 1, 65556)])
def test_an_image_has_the_same_bits_in_every_batch(b, h, l):
    q, k, v = inputs(b, h, l, 11)
    y = attention(q, k, v)
    for i in range(b):
        assert torch.equal(y[i:i + 1], attention(q[i:i + 1], k[i:i + 1], v[i:i + 1])), i
    if l < 4096:
        check(y, q, k, v, b - 1, h - 1)
        check(y, q, k, v, 0, h - 1)


def test_a_range_without_weight():
    q, k, v = inputs(1, 24, 2816, 3)
    q[..., 0] = 1.0
    k[:, :, 256:1024, 0] = float("-inf")
    y = attention(q, k, v)
    assert torch.isfinite(y).all()
    check(y, q, k, v, 0, 23)
    v[0, 23, 2000, 5] = float("nan")
    y = attention(q, k, v)
    assert torch.isnan(y[0, :, 23 * 128 + 5]).all() and torch.isfinite(y[0, :, 23 * 128 + 6]).all()


def test_workspace_is_checked_and_a_graph_replays():
    q, k, v = inputs(1, 24, 2816, 4)
    if not workspace(1, 24, 2816):
        pytest.skip("this GPU's CU count does not split the shape")
    y = torch.zeros(1, 2816, 24 * 128, dtype=torch.bfloat16, device="cuda")
    args = (q.data_ptr(), k.data_ptr(), v.data_ptr(), 1, 24, 2816, 128, y.data_ptr(), 24 * 128, _lib.BF16)
    small = torch.empty(1024, dtype=torch.uint8, device="cuda")
    for ws, n in ((None, 0), (small.data_ptr(), 1024)):
        with pytest.raises(ValueError):
            _lib.call("selas_attention_split", *args, ws, n, _lib.stream(q.device))
    assert torch.count_nonzero(y) == 0
    want = attention(q, k, v)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = attention(q, k, v)
    for _ in range(3):
        got.zero_()
        graph.replay()
        assert torch.equal(attention(q, k, v), want)
        torch.cuda.synchronize()
        assert torch.equal(got, want)
