"""Narrow tiles of the tiled GEMM (256, 192 and 128 rows x 128 columns), taken where 256-column tiles leave CUs idle.

Every tile sums K in the same order, so a launch's rows have the bits of the same rows in a launch of any other
size; and every launch meets the GEMM's bound against the oracle (max abs 1e-2 of the largest value, relative
L2 4e-3: bf16 operands and output, fp32 sums).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import int8_row as oi8
from oracle import nf4 as onf4
from selas_amd import _lib, codecs
from selas_amd.kernels import Kernels
from selas_amd.linear import int8_row_linear, int8_row_linear_gelu, nf4_linear, nf4_linear_gelu

from .conftest import seeded
from .test_capi import tile_query

pytestmark = pytest.mark.gpu


def weight(codec, n, k, dev):
    w = torch.randn(n, k, generator=seeded(n + k)) * 0.02
    enc = codecs.encode_nf4 if codec == "nf4" else codecs.encode_int8_row
    e = enc("w", w.to(dev))
    if codec == "nf4":
        ref = onf4.decode(e.parts["packed"].cpu().numpy(), e.parts["absmax"].cpu().numpy(), 64, out=onf4.BF16)
        args = (e.parts["packed"], e.parts["absmax"], 64, codecs.NF4_CODE, e.shape)
    else:
        ref = oi8.decode(e.parts["q"].cpu().numpy(), e.parts["scale"].cpu().numpy(), oi8.BF16)
        args = (e.parts["q"], e.parts["scale"], e.shape)
    return args, torch.from_numpy(onf4.bf16_to_f32(np.asarray(ref))).view(n, k).double()


# The tile each size runs in on 256 CUs: 128 rows x 128 columns at the smallest, with one row past a tile and partial
# columns (100 rows; 257 x 1000; K of one, two and four blocks: every remainder of the three-block loop); 192 rows in
# whole tiles (8 x 24 of them), one row past and one short; 256 rows, one row short of a tile and one past; and the wide
# tile that follows it at 769 x 9216.
@pytest.mark.parametrize("m,n,k,tile", [
    (33, 64, 64, (128, 128)), (100, 260, 128, (128, 128)), (257, 1000, 256, (128, 128)), (385, 3072, 3072, (128, 128)),
    (1536, 3072, 192, (192, 128)), (1345, 3072, 320, (192, 128)), (575, 9216, 128, (192, 128)),
    (767, 9216, 128, (256, 128)), (2049, 3072, 320, (256, 128)), (769, 9216, 320, (192, 256))])
@pytest.mark.parametrize("codec", ["nf4", "int8_row"])
def test_narrow_tiles(codec, m, n, k, tile):
    dev = torch.device("cuda")
    if torch.cuda.get_device_properties(dev).multi_processor_count == 256:
        assert tile_query(m, n, k, _lib.CODEC_NF4 if codec == "nf4" else _lib.CODEC_INT8_ROW) == tile
    args, w_ref = weight(codec, n, k, dev)
    lin = nf4_linear if codec == "nf4" else int8_row_linear
    x = torch.randn(m, k, generator=seeded(m)).to(torch.bfloat16).to(dev)
    b = (torch.randn(n, generator=seeded(n)) * 0.02).to(torch.bfloat16).to(dev)
    y = lin(x, *args, b)
    rows = torch.unique(torch.cat([torch.arange(0, m, max(1, m // 40)), torch.tensor([m - 1])]))
    ref = x[rows].double().cpu() @ w_ref.t() + b.double().cpu()
    d = y[rows].double().cpu() - ref
    assert d.abs().max() <= 1e-2 * ref.abs().max() and d.norm() <= 4e-3 * ref.norm()
    big = torch.randn(5000, k, generator=seeded(m + 1)).to(torch.bfloat16).to(dev)  # elsewhere in a larger launch, most in wider tiles
    big[1111:1111 + m] = x
    assert torch.equal(lin(big, *args, b)[1111:1111 + m], y)
    if n % 256 == 0:  # the GELU columns in the epilogue: the bits of the linear and the GELU segment
        gelu = nf4_linear_gelu if codec == "nf4" else int8_row_linear_gelu
        ((plain, g),) = gelu([(x, *args, b, 256, None)])
        assert torch.equal(plain, y[:, :n - 256]) and torch.equal(g, Kernels().gelu(y[:, n - 256:]))


@pytest.mark.parametrize("quant", ["nf4", "int8"])
@pytest.mark.parametrize("rows", [1, 5, 33])
def test_modulations_side_by_side(quant, rows):
    # The grouped launch writes a double block's image and text vectors into one buffer: the bits of the linears one by
    # one and their concatenation; 33 rows are past the grouped kernel.
    from selas_amd import flux as F

    cfg = F.FluxConfig(hidden=1024, heads=8, mlp_hidden=512)
    m = F.RandomFlux(cfg, "cuda", seed=3, n_double=2, n_single=3, quant=quant)
    sv = torch.randn(rows, 1, cfg.hidden, generator=seeded(rows)).to(torch.bfloat16).cuda()
    one, got = m.modulations(sv, grouped=False), m.modulations(sv)
    assert len(got) == 5 and all(a.shape == b.shape and torch.equal(a, b) for a, b in zip(one, got))
