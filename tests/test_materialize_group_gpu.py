"""Several small layers' per-sample weight gradients in one launch
(``materialize_linear_group``), against float64 products of the same inputs:
tiles that end inside 64 outputs, token counts that end inside a stage, bias
columns, both output layouts, strided factors, more layers than one launch
takes, and the large layers that keep their own launches.

A sum of T fp32 products is off by at most T * 2^-24 of the sum of their
magnitudes; TOL covers T <= 700 normal factors, and a 16-bit result adds half
a unit in its last place."""

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = 1e-5
HALF_ULP = {torch.float32: 0.0, torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11}


def _ref(a, g, bias):
    m = torch.einsum("bto,btk->bok", g.double(), a.double())
    if bias:
        m = torch.cat([m, g.double().sum(1).unsqueeze(-1)], -1)
    return m.flatten(1)


def _layers(device, dtype, shapes, seed=0):
    gen = torch.Generator(device=device).manual_seed(seed)
    out = []
    for i, (b, t, k, d, bias) in enumerate(shapes):
        a = torch.randn(b, t, k + 8, generator=gen, device=device).to(dtype)[..., :k]
        g = torch.randn(t, b, d, generator=gen, device=device).to(dtype).transpose(0, 1)  # sequence-first capture
        out.append((a.contiguous() if i % 2 else a, g, bias))
    return out


def _check(layers, outs, out_dtype):
    for (a, g, bias), got in zip(layers, outs):
        want = _ref(a, g, bias)
        assert got.dtype == out_dtype
        off = (got.reshape(got.shape[0], -1).double() - want).abs()
        assert bool((off <= TOL * want.abs().max() + HALF_ULP[out_dtype] * want.abs()).all())


SHAPES = [(3, 1, 64, 64, False), (5, 63, 128, 72, True), (2, 64, 8, 200, True), (1, 65, 200, 136, False),
          (4, 129, 72, 8, True), (7, 33, 192, 64, False), (32, 64, 128, 512, True), (2, 700, 64, 128, True)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("out_dtype", [None, torch.float32])
def test_group_matches_float64(device, dtype, out_dtype):
    from dattri_llm_amd import kernels

    layers = _layers(device, dtype, SHAPES)
    assert all(kernels._groupable(a, g) for a, g, _ in layers)
    outs = kernels.materialize_linear_group(layers, out_dtype=out_dtype)
    _check(layers, outs, out_dtype or dtype)
    for (a, _g, bias), m in zip(layers, outs):
        assert kernels.is_blocked(m) == (not bias and a.shape[-1] % 64 == 0)


def test_more_layers_than_one_launch_and_mixed_sizes(device):
    from dattri_llm_amd import kernels

    shapes = [(2, 20 + i, 64 + 8 * (i % 5), 72, i % 3 == 0) for i in range(55)]
    shapes.insert(7, (2, 40, 2048, 2048, False))  # its own launch
    shapes.insert(30, (2, 40, 61, 30, True))      # widths padded: its own launch
    layers = _layers(device, torch.bfloat16, shapes, seed=1)
    assert sum(kernels._groupable(a, g) for a, g, _ in layers) == 55
    _check(layers, kernels.materialize_linear_group(layers), torch.bfloat16)
    assert kernels.materialize_linear_group([]) == []


@pytest.mark.parametrize("dense_test", [False, True])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_block_of_small_layers(device, dtype, dense_test):
    """The grouped path inside layerwise_cross_dot: materialized-route linear
    layers, norms and a dense layer of one block, every layer's sum kept."""
    from dattri_llm_amd.gradient import Factorized, Gradient, ops

    gen = torch.Generator(device=device).manual_seed(5)

    def rnd(*shape):
        return torch.randn(*shape, generator=gen, device=device).to(dtype)

    def side(b, t):
        data = {f"lin{i}": Factorized(rnd(b, t, 128), rnd(b, t, 64 * (1 + i % 3)) / 16, {"has_bias": i % 2 == 0})
                for i in range(5)}
        data["norm"] = Factorized(rnd(b, t, 128), rnd(b, t, 128) / 16,
                                  {"has_bias": True, "eps": 1e-5, "normalized_shape": (128,)})
        data["dense"] = rnd(b, 1000)
        types = {n: "nn.LayerNorm" if n == "norm" else "nn.Linear" for n in data}
        form = {n: "materialized" if n == "dense" else "factorized" for n in data}
        return Gradient(form, data, types, {n: "batch" if n == "dense" else "batch_token" for n in data})

    train, test = side(9, 40), side(4, 48)
    per_layer = ops.layerwise_cross_dot(train, test, reduce="none", mode="materialized")
    if dense_test:
        data = {n: ops.materialize_blocked(v, test.layer_types[n]) for n, v in test.data.items()}
        test = Gradient(dict.fromkeys(data, "materialized"), data, test.layer_types, dict.fromkeys(data, "batch"))
    got = ops.layerwise_cross_dot(train, test, mode="materialized").double()
    want = sum(v.double() for v in per_layer.values())
    # per-layer results are rounded to the compute dtype one by one, the block's once
    tol = 1e-5 if dtype == torch.float32 else 8 * 2.0**-8
    assert float((got - want).abs().max()) <= tol * float(want.abs().max())


def test_narrow_layers_with_many_rows_stay_alone(device):
    """16-bit adapter layers on both sides of the line, beside a wide one, in one
    call: those with many rows per tile keep their own launch."""
    from dattri_llm_amd import kernels

    shapes = [(4, 1600, 64, 2048, False), (2, 1600, 1024, 16, False), (1, 3000, 256, 64, True), (2, 700, 128, 200, False),
              (32, 800, 64, 1024, True)]
    layers = _layers(device, torch.bfloat16, shapes)
    assert [kernels._groupable(a, g) for a, g, _ in layers] == [True, True, True, True, False]
    assert all(kernels._groupable(a.float(), g.float()) for a, g, _ in layers)
    outs = kernels.materialize_linear_group(layers, out_dtype=torch.float32)
    for (a, g, bias), got in zip(layers, outs):
        want = _ref(a, g, bias)
        # sums of up to 3000 products: 2^-24 sqrt(3000 / 2) of their size, the largest of 10^5 five times that
        assert float((got.reshape(got.shape[0], -1).double() - want).abs().max()) <= 2 * TOL * float(want.abs().max())
