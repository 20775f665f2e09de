"""The 256 x 256 dW kernel on rows that end off a 16-byte boundary (a bias
column) and on fp32 rows split into three bf16 parts, against float64: widths
that end inside a tile, a chunk and a pair of elements, one token, token counts
around a stage, k-blocked outputs, and values the parts cannot hold.

TOL bounds fp32 sums of up to 600 normal products (each within 2^-24 of its
partial sum's magnitude); a 16-bit result adds half a unit in its last place."""

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = 1e-5
HALF_ULP = {torch.float32: 0.0, torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11}


def _factors(device, dtype, b, t, k, d, seed=0):
    gen = torch.Generator(device=device).manual_seed(seed)
    return (torch.randn(b, t, k, generator=gen, device=device).to(dtype),
            torch.randn(b, t, d, generator=gen, device=device).to(dtype))


def _check(a, g, bias, out, out_dtype):
    want = torch.stack([y.double().t() @ x.double() for x, y in zip(a, g)])
    if bias:
        want = torch.cat([want, g.double().sum(1).unsqueeze(-1)], -1)
    want = want.flatten(1)
    off = (out.reshape(out.shape[0], -1).double() - want).abs()
    assert out.dtype == out_dtype
    assert bool((off <= TOL * want.abs().max() + HALF_ULP[out_dtype] * want.abs()).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("out_dtype", [None, torch.float32])
@pytest.mark.parametrize("shape", [(2, 70, 256, 256), (3, 31, 264, 520), (1, 600, 1032, 264), (17, 1, 512, 768)])
def test_rows_off_alignment(device, dtype, out_dtype, shape):
    from dattri_llm_amd import kernels

    a, g = _factors(device, dtype, *shape)
    print(f"materialize bias {shape} {dtype} -> {out_dtype}", flush=True)
    _check(a, g, True, kernels.materialize_linear(a, g, bias=True, out_dtype=out_dtype), out_dtype or dtype)


@pytest.mark.parametrize("tokens", [64, 130])
@pytest.mark.parametrize("k,d", [(512, 1024), (1024, 1024), (768, 2048), (2048, 2048)])
def test_tile_orders(device, tokens, k, d):
    """8, 16, 24 and 64 tiles per sample around the line between whole samples
    and eighths of each sample per XCD: every tile is taken once."""
    from dattri_llm_amd import kernels

    a, g = _factors(device, torch.bfloat16, 5, tokens, k, d)
    _check(a, g, False, kernels.materialize_linear(a, g, out_dtype=torch.float32), torch.float32)


def _split(b, t, k, d):
    from dattri_llm_amd import _native as nat

    need = ctypes.c_size_t()
    nat.check(nat.load().da_materialize_linear_workspace(nat.DA_F32, b, t, k, d, ctypes.byref(need)), "query")
    return need.value > 0


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("blocked", [False, True])
@pytest.mark.parametrize("shape", [(16, 400, 1024, 1024), (8, 351, 1020, 2044), (6, 600, 2048, 1280),
                                   (64, 16, 1024, 1024), (33, 30, 2044, 2052)])
def test_split_rows(device, shape, bias, blocked):
    from dattri_llm_amd import kernels

    b, t, k, d = shape
    assert _split(b, t, k, d)
    a, g = _factors(device, torch.float32, *shape)
    print(f"materialize split {shape} bias={bias} blocked={blocked}", flush=True)
    out = kernels.materialize_linear(a, g, bias=bias, blocked=blocked)
    _check(a, g, bias, out, torch.float32)
    wide = torch.zeros(t, b, k + 60, device=device)  # sequence-first rows inside wider ones
    wide[..., 60:] = a.transpose(0, 1)
    again = kernels.materialize_linear(wide.transpose(0, 1)[..., 60:], g, bias=bias, blocked=blocked)
    assert torch.equal(out, again)
    _check(a, g, bias, kernels.materialize_linear(a, g, bias=bias, out_dtype=torch.bfloat16), torch.bfloat16)


@pytest.mark.parametrize("value", [float("inf"), float("nan"), -3.4e38, 1e-38])
def test_values_the_parts_cannot_hold(device, value):
    from dattri_llm_amd import kernels

    shape = (16, 400, 1024, 1024)
    assert _split(*shape)
    a, g = _factors(device, torch.float32, *shape)
    g[:, :, 7] = g[:, :, 7].abs() + 0.1  # one column without sign changes, so infinities keep theirs
    a[3, 11, 5] = value
    got = kernels.materialize_linear(a, g).cpu()
    want = torch.stack([y.t() @ x for x, y in zip(a.cpu(), g.cpu())]).flatten(1)
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(torch.isinf(got), torch.isinf(want))
    ok = torch.isfinite(want) & (want.abs() < 1e30)
    assert float((got[ok] - want[ok]).abs().max()) <= 4 * TOL * float(want[ok].abs().max())


@pytest.mark.parametrize("log_a,log_g", [(70, 69), (-122, 45)])
def test_one_product_at_the_ends_of_the_range(device, log_a, log_g):
    """Every entry one product: infinite where fp32 is, nowhere NaN, and as exact
    relative to itself where the parts are too small to hold it."""
    from dattri_llm_amd import kernels

    b, t, k, d = 16, 400, 1024, 1024
    assert _split(b, t, k, d)
    a, g = _factors(device, torch.float32, b, t, k, d, seed=3)
    a[:, 1:] = 0
    a[:, 0] = (a[:, 0].abs().clamp(max=1.0) + 1.0) * 2.0**log_a
    g *= 2.0**log_g
    got = kernels.materialize_linear(a, g)
    want = (g[:, 0, :, None] * a[:, 0, None, :]).flatten(1)
    exact = (g[:, 0, :, None].double() * a[:, 0, None, :].double()).flatten(1).abs()
    assert not bool(got.isnan().any())
    assert torch.equal(got.isinf(), want.isinf()) and torch.equal(got.sign(), want.sign())
    assert bool(((got.double().abs() - exact).abs() <= 2.0**-22 * exact)[want.isfinite()].all())
