"""The few-row GEMV (NF4, M <= 2, K = 1024, 2048, 3072) and the streaming one that follows it at M = 3: at row counts
around a workgroup's and a round's, alone and in a group with the same bits, and with x of any magnitude.

The kernel multiplies x, exact in scaled fp16, by code * absmax with the code in fp16 and fp32 sums, so the reference
is the oracle's fp32 decode, in 64 bits. An output is off by at most 2^-9 of itself (its bf16 rounding) and by the code
roundings, 2^-12 of a product at most, which over K >= 1024 products of random sign stay below 1e-4 of the row's
products in quadrature: max abs 1e-2 of the largest output and relative L2 4e-3 hold for rows of 4 outputs. (The bf16
decode of the weight is itself 1.1e-3 of that quadrature sum away, too far for rows of 4 small outputs.)
"""

from __future__ import annotations

import pytest
import torch

from oracle import nf4 as onf4
from selas_amd import codecs
from selas_amd.linear import nf4_linear, nf4_linear_grouped

from .conftest import seeded

pytestmark = pytest.mark.gpu


def weight(n, k, seed):
    w = torch.randn(n, k, generator=seeded(seed)) * 0.02
    p, a = onf4.encode(w.numpy())
    ref = torch.from_numpy(onf4.decode(p, a, 64, out=onf4.F32).copy()).view(n, k).double()
    b = (torch.randn(n, generator=seeded(seed + 1)) * 0.02).to(torch.bfloat16)
    return (torch.from_numpy(p).cuda(), torch.from_numpy(a).cuda(), 64, codecs.NF4_CODE, (n, k), b.cuda()), ref, b.double()


def check(y, x, ref, b, slack=0.0):
    want = x.double().cpu() @ ref.t() + b
    for r in range(x.shape[0]):  # row by row: each relative to its own size
        d = (y[r].double().cpu() - want[r]).abs().sub(slack).clamp(min=0)
        assert d.max() <= 1e-2 * want[r].abs().max() and d.norm() <= 4e-3 * want[r].norm()


@pytest.mark.parametrize("k", [1024, 2048, 3072])
@pytest.mark.parametrize("m", [1, 2, 3, 4])
def test_alone_and_in_a_group(m, k):
    ws = [weight(n, k, 7 * i + k) for i, n in enumerate((4, 12, 16, 20, 4100, 300))]
    wide = torch.randn(m, k + 64, generator=seeded(m + k)).to(torch.bfloat16).cuda()
    x = wide[:, 32:32 + k]
    ys = nf4_linear_grouped(x, [w for w, _, _ in ws])
    for (w, ref, b), y in zip(ws, ys):
        check(y, x, ref, b)
        assert torch.equal(y, nf4_linear(x.contiguous(), *w))
    no_bias = ws[3][0][:5] + (None,)
    check(nf4_linear(x, *no_bias), x, ws[3][1], 0.0)


@pytest.mark.parametrize("k", [1024, 3072])
def test_a_row_has_the_same_bits_on_either_side_of_the_third(k):
    # Rows do not see each other: M = 1 gives a row the bits of M = 2, and M = 3 those of M = 32. Between the two kernels
    # only the order of the fp32 sums and the granularity of x's scale differ, about 1e-6 of a sum: an output differs
    # where that crosses a bf16 rounding, by 2^-8 of itself, so with 1 % of such outputs by 4e-4 in the 2-norm.
    w, _, _ = weight(1500, k, 21)
    x = torch.randn(32, k, generator=seeded(k)).to(torch.bfloat16).cuda()
    one, two, three, all32 = (nf4_linear(x[:m], *w) for m in (1, 2, 3, 32))
    assert torch.equal(one, two[:1]) and torch.equal(nf4_linear(x[1:2], *w), two[1:])
    assert torch.equal(three, all32[:3]) and torch.equal(nf4_linear(x[29:], *w), all32[29:])
    d = (two.double() - three[:2].double()).norm()
    assert d <= 4e-4 * three[:2].double().norm()


def test_one_round_and_a_part():
    w, ref, b = weight(18432, 3072, 3)
    x = torch.nn.functional.silu(torch.randn(1, 3072, generator=seeded(5))).to(torch.bfloat16).cuda()
    check(nf4_linear(x, *w), x, ref, b)


def test_rows_of_any_magnitude():
    w, ref, b = weight(256, 3072, 11)
    b = b * 0
    w = w[:5] + (None,)
    x = torch.randn(4, 3072, generator=seeded(6))
    x[0] *= 2.0 ** -60
    x[1] *= 2.0 ** 60
    x[2, 17] = 3.0e38
    x[3] = x[3].abs() + 1.0
    x = x.to(torch.bfloat16).cuda()
    check(nf4_linear(x, *w), x, ref, b)
    z = torch.zeros(2, 3072, dtype=torch.bfloat16, device="cuda")
    z[1, 5] = float("nan")
    y = nf4_linear(z, *w)
    assert torch.count_nonzero(y[0]) == 0 and torch.isnan(y[1]).all()


@pytest.mark.parametrize("m", [1, 2, 4, 32])
@pytest.mark.parametrize("exponent", [-111, -112, -113, -119, -125, -129])
def test_rows_of_the_smallest_magnitudes(m, exponent):
    # Below 2^-112 the scale that would bring x to 2^14 has no normal inverse; at 2^-129 x is subnormal. The outputs'
    # own bf16 rounding is 2^-134 where they are subnormal.
    w, ref, _ = weight(256, 3072, 12)
    x = (torch.randn(m, 3072, generator=seeded(m)) * 2.0 ** exponent).to(torch.bfloat16)
    if m > 1:
        x[m - 1, 100:] = 0.0  # lanes and slices of zeros beside tiny ones
    x = x.cuda()
    check(nf4_linear(x, *w[:5], None), x, ref, 0.0, slack=2.0 ** -134)
