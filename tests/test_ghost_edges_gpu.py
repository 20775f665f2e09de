"""Ghost products whose last tile ends inside a wave's 64 x 64 block, at its edge, or leaves whole blocks
without rows, against float64."""

import pytest
import torch

from dattri_llm_amd import kernels

pytestmark = pytest.mark.gpu

# 16-bit inputs are exact and every dtype's products are summed in fp32: two sums of up to 160 products and one of
# up to 257 * 129 terms of random sign, each step within 2^-24.
TOL = 1e-5


def _factors(gen, b, t, k, d, dtype):
    return (torch.randn(b, t, k, generator=gen).to(dtype).cuda(), torch.randn(b, t, d, generator=gen).to(dtype).cuda())


@pytest.mark.parametrize("t1", [1, 64, 65, 128, 129, 192, 193, 256, 257])
@pytest.mark.parametrize("t2", [1, 64, 65, 128, 129])
@pytest.mark.parametrize("dtype,bias", [(torch.bfloat16, False), (torch.float16, True), (torch.float32, True)])
def test_edges(t1, t2, dtype, bias):
    gen = torch.Generator().manual_seed(1000 * t1 + t2)
    print(f"{t1} x {t2} {dtype}", flush=True)
    a1, g1 = _factors(gen, 2, t1, 96, 160, dtype)
    a2, g2 = _factors(gen, 3, t2, 96, 160, dtype)
    x, y = a1.double().flatten(0, 1), g1.double().flatten(0, 1)
    p = (x @ a2.double().flatten(0, 1).t() + float(bias)) * (y @ g2.double().flatten(0, 1).t())
    p = p.view(2, t1, 3, t2)
    got = kernels.ghost_gram(a1, g1, a2, g2, bias=bias)
    assert (got.double() - p.sum((1, 3))).abs().max() <= TOL * p.sum((1, 3)).abs().max()
    got = kernels.ghost_gram_per_token(a1, g1, a2, g2, bias=bias)
    assert (got.double() - p.sum(3)).abs().max() <= TOL * p.sum(3).abs().max()
