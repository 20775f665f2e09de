"""Norm layers sharing one launch, against float64: both sides of the group's
limits (256 tokens, 2048 sums), odd widths, one token, strided and
sequence-first rows, all three kinds, with and without a bias.

Bounds: x_hat is a rounding or two of 2^-24 per operation and the token sum of
n terms is within n * 2^-24 of the sum of the terms' magnitudes; with random
signs 1e-5 of the largest result holds to 512 tokens."""

import ctypes

import pytest
import torch

TOL = 1e-5


def _want(x, g, kind, eps, bias):
    x, g = x.double(), g.double()
    if kind == 1:
        x = x - x.mean(-1, keepdim=True)
    if kind != 2:
        x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)
    out = (x * g).sum(1)
    return torch.cat([out, g.sum(1)], -1) if bias else out


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bias", [False, True])
def test_group_matches_float64(device, dtype, bias):
    from dattri_llm_amd import kernels

    gen = torch.Generator(device=device).manual_seed(3)

    def rnd(*s):
        return torch.randn(*s, generator=gen, device=device).to(dtype)

    layers = []
    for n, (b, t, d) in enumerate([(3, 64, 128), (1, 1, 4), (5, 7, 100), (2, 17, 1023), (2, 256, 1024), (2, 257, 64),
                                   (3, 9, 2048), (2, 5, 4100), (40, 2, 8)]):
        layers.append((rnd(b, t, d) + 0.5, rnd(b, t, d), n % 3, 1e-5, bias))
    x, g = rnd(64, 3, 128), rnd(64, 3, 256)
    layers.append((x.transpose(0, 1), g.transpose(0, 1)[..., 128:], 1, 0.0, bias))  # sequence-first, half a row
    layers.append((rnd(1, 6, 64).expand(4, 6, 64), rnd(4, 6, 64), 0, 1e-6, bias))
    print(f"norm group {dtype} bias={bias}", flush=True)
    got = kernels.norm_weight_grad_group(layers)
    for (x, g, kind, eps, hb), out in zip(layers, got):
        want = _want(x, g, kind, eps, hb)
        assert out.dtype == torch.float32 and out.shape == want.shape
        assert float((out.double() - want).abs().max()) <= TOL * float(want.abs().max()), (tuple(x.shape), kind)
    alone = kernels.norm_weight_grad_group(layers[:1])[0]
    want = _want(*layers[0])
    assert float((alone.double() - want).abs().max()) <= TOL * float(want.abs().max())


@pytest.mark.gpu
def test_group_many_layers(device):
    """More layers than one launch takes."""
    from dattri_llm_amd import kernels

    gen = torch.Generator(device=device).manual_seed(4)
    layers = [(torch.randn(2, 5, 8 + i, generator=gen, device=device),
               torch.randn(2, 5, 8 + i, generator=gen, device=device), 1, 1e-5, True) for i in range(70)]
    for (x, g, kind, eps, bias), out in zip(layers, kernels.norm_weight_grad_group(layers)):
        want = _want(x, g, kind, eps, bias)
        assert float((out.double() - want).abs().max()) <= TOL * float(want.abs().max())


@pytest.mark.gpu
@pytest.mark.parametrize("layer_type", ["nn.LayerNorm", "nn.RMSNorm", "nn.GroupNorm"])
def test_final_factors_with_a_group_axis(device, layer_type):
    """4-D final factors of a norm layer beside an ordinary one: scored layer by
    layer and summed over layers alike."""
    from dattri_llm_amd.gradient import Factorized, Gradient, ops

    gen = torch.Generator(device=device).manual_seed(6)

    def side(b):
        data = {n: Factorized(*(torch.randn(b, *shape, generator=gen, device=device) for _ in range(2)),
                              module_kwargs=None) for n, shape in (("grouped", (4, 5, 16)), ("plain", (6, 16)))}
        return Gradient(dict.fromkeys(data, "factorized"), data, dict.fromkeys(data, layer_type),
                        dict.fromkeys(data, "batch_token"))

    one, two = side(3), side(2)
    each = ops.layerwise_cross_dot(one, two, reduce="none")
    want = sum(each.values())
    assert float((ops.layerwise_cross_dot(one, two) - want).abs().max()) <= TOL * float(want.abs().max())


def test_group_rejects_what_one_layer_does():
    from dattri_llm_amd import _native as nat

    lib = nat.load()

    def call(**kw):
        rec = nat.NormLayer(x=0x10000, g=0x20000, out=0x30000, batch=1, tokens=4, d=64, x_bstride=256, x_tstride=64,
                            g_bstride=256, g_tstride=64, kind=0, has_bias=0, eps=1e-5)
        dtype = kw.pop("dtype", nat.DA_F32)
        for k, v in kw.items():
            setattr(rec, k, v)
        return lib.da_norm_weight_grad_group(ctypes.byref(rec), 1, dtype, None)

    for bad in ({"dtype": 9}, {"kind": 3}, {"d": 0}, {"d": 2052, "x_tstride": 2052, "g_tstride": 2052}, {"tokens": 0},
                {"batch": -1}, {"x": 0x10008}, {"g_tstride": 66}, {"out": None}, {"d": 1028, "has_bias": 1}):
        assert call(**bad) == nat.DA_ERR_INVALID, bad
    assert lib.da_norm_weight_grad_group(None, 1, nat.DA_F32, None) == nat.DA_ERR_INVALID
    assert lib.da_norm_weight_grad_group(None, 0, nat.DA_F32, None) == 0
