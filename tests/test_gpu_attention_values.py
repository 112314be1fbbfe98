"""selas_attention_v (values read as they are, transposed by the LDS reads) against selas_attention on the values laid
out by transpose_heads: the same products in the same order, so the same bits, at the edges of the 64-key and 128- and
256-query tiles and in both workgroup sizes; and against softmax(q k^T / sqrt(128)) v in 64 bits (bf16 probabilities
and output: max abs 1e-2 of the largest value, relative L2 4e-3).
"""

from __future__ import annotations

import pytest
import torch

from selas_amd import _lib
from selas_amd.attention import attention, transpose_heads

from .conftest import seeded

pytestmark = pytest.mark.gpu


# 48 heads of 1536 or 1537 tokens fill more than one round of workgroups, the rest a part of one.
@pytest.mark.parametrize("b,h,l", [(1, 2, 1), (1, 3, 63), (2, 2, 64), (1, 2, 65), (1, 2, 127), (1, 1, 129), (1, 2, 192),
                                   (1, 2, 257), (1, 24, 768), (1, 24, 1536), (1, 22, 1500), (2, 24, 1537)])
def test_same_bits_as_the_transposed_values(b, h, l):
    g = seeded(b + h + l)
    q, k, v = (torch.randn(b, h, l, 128, generator=g).to(torch.bfloat16).cuda() for _ in range(3))
    wide = torch.zeros(b, l, h * 128 + 64, dtype=torch.bfloat16, device="cuda")
    y = attention(q, k, v, out=wide[..., :h * 128])
    ref, vt = torch.empty(b, l, h * 128, dtype=torch.bfloat16, device="cuda"), transpose_heads(v)
    _lib.call("selas_attention", q.data_ptr(), k.data_ptr(), vt.data_ptr(), b, h, l, 128, ref.data_ptr(), h * 128,
              _lib.BF16, _lib.stream(q.device))
    assert torch.equal(y, ref) and torch.count_nonzero(wide[..., h * 128:]) == 0
    # v as a strided view ([B, L, H, 128] in memory): copied, same bits
    assert torch.equal(attention(q, k, v.transpose(1, 2).contiguous().transpose(1, 2)), ref)
    i, j = b - 1, h - 1
    s = torch.softmax(q[i, j].double() @ k[i, j].double().t() / 128 ** 0.5, -1) @ v[i, j].double()
    d = y[i, :, j * 128:(j + 1) * 128].double() - s
    assert d.abs().max() <= 1e-2 * s.abs().max() and d.norm() <= 4e-3 * s.norm()


def test_values_off_alignment_are_refused():
    q, k, v = (torch.randn(1, 1, 65, 128, generator=seeded(1)).to(torch.bfloat16).cuda() for _ in range(3))
    odd = torch.empty(65 * 128 + 1, dtype=torch.bfloat16, device="cuda")[1:].view(1, 1, 65, 128)
    with pytest.raises(_lib.Unsupported):
        attention(q, k, odd.copy_(v))


@pytest.mark.parametrize("l", [65, 768, 3000])
def test_out_may_overlap_the_values(l):
    q, k, v = (torch.randn(1, 1, l, 128, generator=seeded(l + i)).to(torch.bfloat16).cuda() for i in range(3))
    want = attention(q, k, v)
    buf = torch.zeros(l + 8, 128, dtype=torch.bfloat16, device="cuda")
    for vo, oo in ((0, 0), (0, 8), (8, 0)):  # the same rows; 8 rows later, 8 earlier
        buf[vo:vo + l] = v[0, 0]
        got = attention(q, k, buf[vo:vo + l].view(1, 1, l, 128), out=buf[oo:oo + l].unsqueeze(0))
        assert got.data_ptr() == buf[oo].data_ptr() and torch.equal(got, want)
