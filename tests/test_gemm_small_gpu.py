"""GPU parity of relation_linear on the shapes with few or narrow output tiles, against a
float64 product of the same operands.

  split_kernel           fp32 A, few tiles: the eight waves split K (fewer than eight
                         32-wide chunks, one more than a round, ragged M and N), 16x16
                         tiles (up to 256 of them) and 32x32
  dma_tile_kernel        64x64 tiles: 16-bit operands under one 128x128 tile per CU (the
                         bits of the 128x128 tiles), and fp32 operands
  smallk_stream_kernel   K <= 128, whole 128-column tiles: one and several row tiles per
                         workgroup, a partial last one, every K; the bits of smallk_kernel

Each kernel's sums are fp32 sums of exact products, so an output is within 1e-5 of
sum |a w| (K <= 2304 terms, eight partial sums: 2304 x 2^-24 is 1.4e-4 at worst for one
chain, its usual size sqrt(K) x 2^-24 = 3e-6), plus half an ulp of a 16-bit output.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from relation_lm import _native  # noqa: F401  (registers torch.ops.relation_lm)

pytestmark = pytest.mark.gpu
ops = torch.ops.relation_lm


def run(device, m, n, k, adt, wdt, odt, bias, pad=0, seed=0):
    g = torch.Generator().manual_seed(m * 7 + n * 3 + k + seed)
    base = torch.randn(m, k + pad, generator=g).to(adt)
    w = (torch.randn(n, k, generator=g) / np.sqrt(k)).to(wdt)
    b = (0.5 * torch.randn(n, generator=g)).to(wdt) if bias else None
    a = base[:, :k]
    got = ops.relation_linear(base.to(device)[:, :k], w.to(device),
                              None if b is None else b.to(device), odt)
    torch.cuda.synchronize()
    assert got.shape == (m, n) and got.dtype == odt
    # A 16-bit weight sees A rounded to its type.
    a64, w64 = a.to(wdt).double(), w.double()
    want, mag = a64 @ w64.T, a64.abs() @ w64.abs().T
    if b is not None:
        want, mag = want + b.double(), mag + b.double().abs()
    tol = 1e-5 * mag + 1e-6
    if odt != torch.float32:
        bits = 8 if odt == torch.bfloat16 else 11
        tol = tol + torch.exp2(torch.floor(torch.log2(want.abs().clamp(min=1e-30))) - bits)
    off = (got.double().cpu() - want).abs()
    assert bool((off <= tol).all()), (m, n, k, float(off.max()))
    return got


BF, HF, FL = torch.bfloat16, torch.float16, torch.float32


@pytest.mark.parametrize("m,n,k", [(65, 16, 160), (97, 33, 224), (192, 576, 2304), (1000, 130, 288),
                                   (70, 100, 1024), (1, 8, 1024), (17, 70, 1312), (64, 1024, 1024),
                                   (64, 1040, 1056)])
@pytest.mark.parametrize("wdt,odt", [(BF, FL), (HF, BF), (FL, FL), (FL, BF)])
def test_waves_split_k(device, m, n, k, wdt, odt):
    run(device, m, n, k, FL, wdt, odt, True)
    run(device, m, n, k, FL, wdt, odt, False, pad=8)


@pytest.mark.parametrize("m,n,k", [(1, 4608, 128), (33, 72, 64), (64, 576, 2304), (3, 7, 32),
                                   (5, 512, 576), (40, 20, 36)])
def test_fp32_few_rows(device, m, n, k):
    run(device, m, n, k, FL, FL, FL, True)


@pytest.mark.parametrize("m,n,k,pad", [(3000, 516, 64, 0), (2049, 512, 96, 4), (1100, 1000, 32, 0),
                                       (4200, 300, 1024, 0), (600, 2000, 100, 0)])
def test_fp32_tiles(device, m, n, k, pad):
    run(device, m, n, k, FL, FL, FL, True, pad=pad)


@pytest.mark.parametrize("m,n,k,odt", [(65, 8, 192, FL), (300, 512, 576, BF), (3585, 520, 576, BF),
                                       (100, 72, 64 * 5, HF)])
def test_16_bit_small_tiles(device, m, n, k, odt):
    run(device, m, n, k, BF, BF, odt, True)
    run(device, m, n, k, BF, BF, odt, False, pad=16)


def test_16_bit_tile_sizes_agree(device):
    """The same rows in a problem of 64x64 tiles and in one of 128x128 tiles: same bits."""
    g = torch.Generator().manual_seed(4)
    a = torch.randn(8192, 576, generator=g).to(BF).to(device)
    w = (torch.randn(512, 576, generator=g) / 24).to(BF).to(device)
    whole = ops.relation_linear(a, w, None, FL)
    part = ops.relation_linear(a[:700], w, None, FL)
    torch.cuda.synchronize()
    assert torch.equal(whole[:700], part)


@pytest.mark.parametrize("m", [65, 640, 4100])
@pytest.mark.parametrize("n,k", [(128, 32), (1024, 64), (4608, 96), (6144, 128)])
@pytest.mark.parametrize("odt", [BF, FL])
def test_small_k_streamed(device, m, n, k, odt):
    got = run(device, m, n, k, BF, BF, odt, True)
    # N - 8 columns end in a partial tile and take smallk_kernel: same bits.
    g = torch.Generator().manual_seed(m * 7 + n * 3 + k)
    a = torch.randn(m, k, generator=g).to(BF).to(device)
    w = (torch.randn(n, k, generator=g) / np.sqrt(k)).to(BF).to(device)
    b = (0.5 * torch.randn(n, generator=g)).to(BF).to(device)
    ragged = ops.relation_linear(a, w[:n - 8].contiguous(), b[:n - 8].contiguous(), odt)
    torch.cuda.synchronize()
    assert torch.equal(got[:, :n - 8], ragged)


def test_small_k_strided_rows(device):
    run(device, 300, 256, 128, HF, HF, HF, True, pad=24)
    out = torch.zeros(200, 512, dtype=BF, device=device)
    a = torch.randn(200, 64, generator=torch.Generator().manual_seed(1)).to(BF).to(device)
    w = torch.randn(256, 64, generator=torch.Generator().manual_seed(2)).to(BF).to(device)
    ops.relation_linear_out(a, w, None, out[:, 256:])
    torch.cuda.synchronize()
    assert torch.equal(out[:, 256:], ops.relation_linear(a, w, None, BF))
    assert bool((out[:, :256] == 0).all())


@pytest.mark.parametrize("m,k", [(1, 1024), (24, 1056), (64, 2304), (24, 992)])
@pytest.mark.parametrize("wdt", [BF, HF])
def test_long_rows_reach_the_caches(device, m, k, wdt):
    """fp32 rows against a 16-bit weight, at lengths where the product alone is split: the
    cache-row scatter still writes the caches."""
    g = torch.Generator().manual_seed(m + k)
    a = torch.randn(m, k, generator=g).to(device)
    w = (torch.randn(96, k, generator=g) / np.sqrt(k)).to(wdt).to(device)
    caches = [torch.zeros(m, 8, n, device=device) for n in (16, 16, 32, 32)]
    out = ops.packed_projection_to_caches(a, w, *caches, torch.tensor(5, device=device), False)
    torch.cuda.synchronize()
    lo = 0
    for c in caches:
        n = c.size(2)
        assert torch.equal(c[:, 5], out[:, lo:lo + n]) and bool(c[:, 5].any())
        assert not bool(c[:, [0, 1, 2, 3, 4, 6, 7]].any())
        lo += n
    a64, w64 = a.to(wdt).double(), w.double()
    assert bool(((out.double() - a64 @ w64.T).abs() <= 1e-5 * (a64.abs() @ w64.abs().T) + 1e-6).all())


@pytest.mark.parametrize("adt,wdt,odt", [(BF, BF, BF), (HF, HF, FL), (FL, BF, FL), (FL, FL, FL)])
@pytest.mark.parametrize("m,n", [(5, 128), (100, 256), (4100, 1024), (130, 72)])
def test_empty_reduction_is_the_bias(device, m, n, adt, wdt, odt):
    """K = 0 reads neither operand (their pointers are null here): every output row is the bias."""
    x = torch.empty(m, 8, dtype=adt, device=device)[:, :0]
    w = torch.empty(n, 0, dtype=wdt, device=device).as_strided((n, 0), (0, 1))
    b = torch.randn(n, generator=torch.Generator().manual_seed(n)).to(wdt).to(device)
    out = torch.full((m, n), float("nan"), dtype=odt, device=device)
    ops.relation_linear_out(x, w, b, out)
    torch.cuda.synchronize()
    assert torch.equal(out, b.to(odt).expand(m, n))
