"""The encoders' fast paths (reciprocal and table search, exact redo near a boundary) byte-exact against the oracle,
for fp32, bf16 and fp16 input: elements within a few ulp of every midpoint or half, blocks and rows without a safe
reciprocal (zero, subnormal, huge, Inf, NaN), sizes around a workgroup, and the forms that take the general path.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import int8_row as oi8
from oracle import nf4 as onf4
from selas_amd import _lib, codecs

from .conftest import seeded
from .test_capi import codebook_with_midpoint, edge_midpoints

pytestmark = pytest.mark.gpu
DTYPES = [torch.float32, torch.bfloat16, torch.float16]


def check_nf4(t, **kw):
    e = codecs.encode_nf4("w", t.cuda(), **kw)
    with np.errstate(all="ignore"):
        p, a = onf4.encode(t.float().numpy(), kw.get("blocksize", 64))
    assert np.array_equal(e.parts["absmax"].cpu().numpy(), a, equal_nan=True)
    assert (e.parts["packed"].cpu().numpy() == p).all()


def check_int8(t):
    e = codecs.encode_int8_row("w", t.cuda())
    with np.errstate(all="ignore"):
        q, s = oi8.encode(t.float().numpy())
    assert np.array_equal(e.parts["scale"].cpu().numpy(), s, equal_nan=True)
    ok = np.isfinite(t.float().numpy())  # Inf / Inf is NaN, whose cast to int8 is not defined
    assert (e.parts["q"].cpu().numpy() == q)[ok].all()


def near(values, dtype, ulps=6):
    """Each value and its neighbours, up to ``ulps`` floats to either side, rounded to dtype."""
    v = torch.as_tensor(np.asarray(values, dtype=np.float32))
    out = [v]
    lo, hi = v.numpy(), v.numpy()
    for _ in range(ulps):
        lo, hi = np.nextafter(lo, np.float32(-np.inf)), np.nextafter(hi, np.float32(np.inf))
        out += [torch.from_numpy(lo.copy()), torch.from_numpy(hi.copy())]
    return torch.cat(out).to(dtype)


@pytest.mark.parametrize("dtype", DTYPES)
def test_nf4_near_every_midpoint(dtype):
    mids = onf4.midpoints()
    blocks = []
    for a in (1.0, 0.0371, 3.0, 0.9999, 1.7e-3, 117.25):
        a = torch.tensor(a).to(dtype).float().item()
        v = near(mids.astype(np.float64) * a, dtype, 20)  # entries of the table are 16 ulp off at most
        v = torch.cat([v, v.new_zeros(-v.numel() % 63)]).view(-1, 63)
        blocks.append(torch.cat([v, torch.full((v.shape[0], 1), a).to(dtype)], 1))
    check_nf4(torch.cat(blocks))


@pytest.mark.parametrize("dtype", DTYPES)
def test_int8_near_every_half(dtype):
    rows = []
    for a in (127.0, 1.0, 0.0731, 2.9e-3, 300.0):
        a = torch.tensor(a).to(dtype).float().item()
        v = near((np.arange(-127, 127) + 0.5) * (a / 127), dtype)
        rows.append(torch.cat([v, torch.full((3520 - v.numel(),), a).to(dtype)]))
    check_int8(torch.stack(rows))


@pytest.mark.parametrize("dtype", DTYPES)
def test_specials(dtype):
    t = torch.randn(12, 128, generator=seeded(1))
    t[1] = 0.0
    t[2] *= 1e-42  # subnormal in fp32 and bf16, zero in fp16
    t[3] *= 1e-32
    t[4] *= 1e33
    t[5, 7], t[6, 9], t[7, 70] = float("inf"), float("-inf"), float("nan")
    t[8] = -0.0
    t[9, :64] = 1.0
    t[10] = torch.finfo(dtype).max
    check_nf4(t.to(dtype))
    check_int8(t.to(dtype))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("blocks", [1, 31, 32, 33, 127, 129, 1000])
def test_sizes_around_a_workgroup(dtype, blocks):
    check_nf4((torch.randn(blocks, 64, generator=seeded(blocks)) * 0.02).to(dtype))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("shape", [(3, 8), (5, 2040), (4, 4096), (4, 4104), (2, 8200), (3, 16384), (2, 16392), (7, 100),
                                   (3, 4, 16)])
def test_int8_row_lengths(dtype, shape):
    # every register count of the row kernel, its longest row, and rows past it or not a multiple of 8 (general kernel)
    check_int8((torch.randn(*shape, generator=seeded(shape[-1])) * 0.02).to(dtype))


@pytest.mark.parametrize("dtype", DTYPES)
def test_unaligned_strided_and_other_blocksizes(dtype):
    buf = (torch.randn(64 * 40 + 1, generator=seeded(2)) * 0.02).to(dtype)
    odd = buf.cuda()[1:].view(40, 64)  # off 16-byte alignment
    e, p = codecs.encode_nf4("w", odd), onf4.encode(buf[1:].float().numpy())
    assert (e.parts["packed"].cpu().numpy() == p[0]).all() and (e.parts["absmax"].cpu().numpy() == p[1]).all()
    e, q = codecs.encode_int8_row("w", odd), oi8.encode(buf[1:].view(40, 64).float().numpy())
    assert (e.parts["q"].cpu().numpy() == q[0]).all() and (e.parts["scale"].cpu().numpy() == q[1]).all()
    w = (torch.randn(64, 96, generator=seeded(3)) * 0.02).to(dtype)
    check_nf4(w, blocksize=32)
    e, p = codecs.encode_nf4("w", w.cuda().t()), onf4.encode(w.t().contiguous().float().numpy())
    assert e.shape == (96, 64) and (e.parts["packed"].cpu().numpy() == p[0]).all()


def test_codebook_without_a_search_table():
    # midpoints closer than a bucket: the general kernel, also for 16-bit input (through fp32)
    code = tuple(float(c) for c in np.linspace(-0.1, 0.1, 15, dtype=np.float32)) + (1.0,)
    w = torch.randn(32, 64, generator=seeded(4)).bfloat16()
    e = codecs.encode_nf4("w", w.cuda(), code=code)
    a = w.float().abs().amax(1, keepdim=True)
    c = torch.tensor(code)
    idx = torch.bucketize(w.float() / a, (c[1:] + c[:-1]) / 2).view(-1, 2)
    assert torch.equal(e.parts["packed"].cpu(), ((idx[:, 0] << 4) | idx[:, 1]).to(torch.uint8))


def takes_table(code):
    w = torch.zeros(64, dtype=torch.bfloat16, device="cuda")
    p, a = torch.zeros(32, dtype=torch.uint8, device="cuda"), torch.zeros(1, device="cuda")
    try:
        _lib.call("selas_nf4_encode_typed", w.data_ptr(), _lib.BF16, 64, 64, _lib.code_array(code), p.data_ptr(),
                  a.data_ptr(), _lib.stream(w.device))
    except _lib.Unsupported:
        return False
    return True


@pytest.mark.parametrize("dtype", DTYPES)
def test_codebooks_with_midpoints_at_and_near_bucket_edges(dtype):
    # The elements within 2 ulp of every midpoint of blocks of 400 magnitudes: byte-exact whether the codebook takes
    # the table (midpoints 1e-5 inside an edge, a midpoint of 0, the spread codes) or not (midpoints at an edge).
    bad, good = edge_midpoints()
    a = (torch.rand(400, generator=seeded(9)) + 0.1).to(dtype).float().numpy()
    spread = [tuple(float(c) for c in np.linspace(-0.97, 0.99, 16)), codebook_with_midpoint(0.0)]
    for code, table in [(codebook_with_midpoint(m), False) for m in bad] + \
            [(codebook_with_midpoint(m), True) for m in good] + [(c, True) for c in spread]:
        assert takes_table(code) == table
        v = near(a[:, None] * onf4.midpoints(code)[None, :], dtype, 2).view(5, 400, 15).permute(1, 0, 2).reshape(400, 75)
        w = torch.cat([v[:, :63], torch.from_numpy(a)[:, None].to(dtype), v[:, 12:], torch.from_numpy(a)[:, None].to(dtype)],
                      1)
        e = codecs.encode_nf4("w", w.cuda(), code=code)
        p, absmax = onf4.encode(w.float().numpy(), 64, code)
        assert np.array_equal(e.parts["absmax"].cpu().numpy(), absmax)
        assert (e.parts["packed"].cpu().numpy() == p).all(), code
