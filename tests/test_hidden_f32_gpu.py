"""The relation hidden of fp32 / fp16 caches (hidden_f32_kernel: 32 x 32 tiles where few
64 x 64 ones exist, 64 x 64 tiles, the update form) against the expression in float64.

The products op[a] * op[p] are rounded to fp32 once and R of them are summed in fp32: an
error of (R + 3) x 2^-24 times the sum of the magnitudes at worst; the GELU's slope is at
most 1.13, its own approximation 2e-7, and an fp16 cache holds exact inputs.
"""
import pytest
import torch

import relation_lm  # noqa: F401
from relation_lm.kernels.relation_reduce import (relation_hidden_cache_update,
                                                 relation_hidden_cached,
                                                 relation_hidden_cached_seq)

pytestmark = pytest.mark.gpu


def inputs(device, b, q, k, h, r, t, dtype):
    g = torch.Generator().manual_seed(b + q + h + r)
    rnd = lambda *s, scale=1.0: (torch.randn(*s, generator=g) * scale).to(dtype)
    a = torch.randint(0, t, (b, q), generator=g)
    p = torch.randint(0, t, (b, q, k), generator=g)
    p.view(-1)[0] = t + 3                                      # out of range: gathers zeros
    args = rnd(b, t, 2 * h), rnd(b, t, r), a, p, rnd(h, r, scale=r ** -0.5)
    return args, [x.to(device) for x in args]


def check(got, expanded, operand, a, p, wm):
    h, r, t = wm.shape[0], wm.shape[1], operand.shape[1]
    b = torch.arange(a.shape[0])
    ok = p < t
    pc = p.clamp(max=t - 1)
    x_a = expanded.double()[b[:, None], a][..., :h]
    x_p = expanded.double()[b[:, None, None], pc][..., h:] * ok[..., None]
    prod = operand.double()[b[:, None], a][:, :, None] * operand.double()[b[:, None, None], pc]
    prod = prod * ok[..., None]
    want = torch.nn.functional.gelu(prod @ wm.double().T + x_a[:, :, None] + x_p)
    mag = prod.abs() @ wm.double().abs().T + x_a[:, :, None].abs() + x_p.abs()
    assert got.shape == want.shape
    tol = 1.13 * (r + 3) * 2.0 ** -24 * mag + 2e-6
    assert bool(((got.double().cpu() - want).abs() <= tol).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("b,q,k,h,r", [
    (1, 1, 1, 1, 8), (4, 1, 6, 2304, 128), (2, 5, 7, 100, 40), (1, 11, 3, 33, 136),
    (1, 33, 1, 64, 256), (2, 64, 8, 1024, 128), (1, 340, 5, 700, 72)])
def test_hidden(device, dtype, b, q, k, h, r):
    args, dev = inputs(device, b, q, k, h, r, 50, dtype)
    if q == 1:
        got = relation_hidden_cached(dev[0], dev[1], dev[2][:, 0].contiguous(),
                                     dev[3][:, 0].contiguous(), dev[4])[:, None]
    else:
        got = relation_hidden_cached_seq(*dev)
    torch.cuda.synchronize()
    check(got, *args)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("b,k,h,r", [(1, 3, 64, 128), (9, 8, 100, 40), (3, 5, 200, 264)])
def test_update_form_reads_the_row_it_writes(device, dtype, b, k, h, r):
    args, dev = inputs(device, b, 1, k, h, r, 50, dtype)
    g = torch.Generator().manual_seed(7)
    rnd = lambda *s: (torch.randn(*s, generator=g) * r ** -0.5).to(dtype)
    wa, wp, b1 = rnd(h, r), rnd(h, r), rnd(h)
    dev[2][:, 0] = 20
    dev[3][:, 0, -1] = 20
    args[2][:, 0] = 20
    args[3][:, 0, -1] = 20
    got = relation_hidden_cache_update(
        dev[0], dev[1], dev[2][:, 0].contiguous(), dev[3][:, 0].contiguous(), wa.to(device),
        wp.to(device), dev[4], b1.to(device), torch.tensor(20, device=device))
    torch.cuda.synchronize()
    row = args[1][:, 20].double()
    fresh = torch.cat([row @ wa.double().T + b1.double(), row @ wp.double().T], -1)
    ulp = 2.0 ** (-11 if dtype == torch.float16 else -22)
    assert bool(((dev[0][:, 20].double().cpu() - fresh).abs() <= ulp * fresh.abs().clamp(min=1)
                 + r * 2.0 ** -22).all())
    expanded = args[0].double()
    expanded[:, 20] = fresh
    check(got[:, None], expanded, *args[1:])
