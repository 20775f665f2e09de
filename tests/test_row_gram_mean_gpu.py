"""``row_gram(divisor=...)``: the division as the tiles are written equals a
division of the undivided product (whole tiles, ragged widths, padded columns,
token splits, one row), and the covariances of ``kfac_factors`` through it
match float64 over the gradient-carrying rows."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,p", [(1, 8), (300, 40), (777, 261), (3000, 520), (4096, 1024), (2048, 5888)])
def test_divided_product(device, dtype, n, p):
    from dattri_llm_amd import kernels

    x = torch.randn(n, p, generator=torch.Generator(device=device).manual_seed(n), device=device).to(dtype)
    whole = kernels.row_gram(x)
    got = kernels.row_gram(x, divisor=n)
    assert torch.equal(got, whole * (1.0 / torch.tensor(float(n), device=device)))
    for i in range(256, p, 256):  # tiles below the diagonal are the ones above it
        assert torch.equal(got[i:i + 256, :i], got[:i, i:i + 256].t())
    with pytest.raises(ValueError):
        kernels.row_gram(x, divisor=0)
    with pytest.raises(ValueError):
        kernels.row_gram(x, out=whole, accumulate=True, divisor=n)


@pytest.mark.parametrize("padded", [False, True])
def test_covariances(device, padded):
    from dattri_llm_amd.gradient import ops

    gen = torch.Generator(device=device).manual_seed(1)
    a = torch.randn(3, 150, 320, generator=gen, device=device).bfloat16()
    g = torch.randn(3, 150, 264, generator=gen, device=device).bfloat16()
    if padded:
        g[1, 100:] = 0
    live = (g != 0).any(-1)
    a64, g64 = a[live].double(), g[live].double()
    for bias in (False, True):
        if bias:
            a64 = torch.cat([a64, torch.ones_like(a64[:, :1])], 1)
        got_a, got_g = ops.kfac_factors(a, g, "nn.Linear", {"has_bias": bias})
        for got, x in ((got_a, a64), (got_g, g64)):
            want = x.t() @ x / x.shape[0]
            # 450 bf16 products summed in fp32: within 450 * 2^-24 of the diagonal's scale
            assert float((got.double() - want).abs().max()) <= 3e-5 * float(want.abs().max())
