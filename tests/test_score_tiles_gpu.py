"""Score GEMM at the edges of its output tiles: the row groups of the narrow
ring (8, 16, 32 and 64 query rows, 8 and 16 train rows), layers that end
inside a unit, k-blocked layers beside row-major ones, transposed launches.

Against float64 products of the same inputs.  A sum of n fp32 products in any
order is off by at most n * 2^-24 of the sum of the products' magnitudes; the
partial tiles keep n small, and 1e-5 of the largest score is what the other
score GEMM tests hold it to."""

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = 1e-5
WIDTHS = (64, 1000, 1024, 4168)  # under one unit, a ragged tail, whole units, several units and a tail


def _layers(gen, device, dtype, b1, b2):
    pairs = []
    for i, w in enumerate(WIDTHS):
        m1, m2 = (torch.randn(b, w, generator=gen, device=device).to(dtype) for b in (b1, b2))
        if w % 64 == 0 and dtype != torch.float32 and i % 2 == 0:  # one side k-blocked
            m2 = m2.view(b2, w // 64, 64).permute(1, 0, 2).contiguous().permute(1, 0, 2)
        pairs.append((m1, m2))
    return pairs


def _check(pairs, dtype, b1, b2):
    from dattri_llm_amd import kernels

    print(f"score_gemm {b1}x{b2} {dtype}", flush=True)
    want = sum(x.reshape(b1, -1).double() @ y.reshape(b2, -1).double().t() for x, y in pairs)
    got = kernels.score_gemm(pairs)
    assert float((got.double() - want).abs().max()) <= TOL * float(want.abs().max())
    swapped = kernels.score_gemm([(y, x) for x, y in pairs])  # the taller side first: a transposed launch
    assert float((swapped.double() - want.t()).abs().max()) <= TOL * float(want.abs().max())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("b1", [1, 8, 9, 16])
def test_narrow_ring_row_groups(device, dtype, b1):
    gen = torch.Generator(device=device).manual_seed(b1)
    for b2 in (1, 7, 8, 9, 16, 17, 32, 33, 64, 65, 130):
        _check(_layers(gen, device, dtype, b1, b2), dtype, b1, b2)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("b1", [64, 65, 127, 128, 129, 257])
def test_large_tile_edges(device, dtype, b1):
    """Both sides of the line where the 128 x 256 tile takes over, and its edges."""
    gen = torch.Generator(device=device).manual_seed(b1)
    for b2 in (128, 129, 255, 256, 257, 600):
        _check(_layers(gen, device, dtype, b1, b2), dtype, b1, b2)


def test_large_tile_accumulates_and_splits(device):
    """One share and several shares of the width per tile, into an existing
    output in both orientations; strided operands."""
    from dattri_llm_amd import kernels

    gen = torch.Generator(device=device).manual_seed(3)
    for b1, b2, w in ((130, 300, 128), (130, 300, 65536 + 72), (2100, 1030, 264)):
        m1 = torch.randn(b1, w + 8, generator=gen, device=device).bfloat16()[:, :w]
        m2 = torch.randn(b2, w + 16, generator=gen, device=device).bfloat16()[:, :w]
        first = torch.randn(b1, b2, generator=gen, device=device)
        want = first.double() + m1.double() @ m2.double().t()
        print(f"score_gemm accumulate {b1}x{b2} w={w}", flush=True)
        for x, y, out in ((m1, m2, first.clone()), (m2, m1, first.t().contiguous())):
            got = kernels.score_gemm([(x, y)], out=out, accumulate=True)
            ref = want if out.shape == want.shape else want.t()
            assert float((got.double() - ref).abs().max()) <= TOL * float(want.abs().max())


@pytest.mark.parametrize("b1,b2", [(8, 32), (16, 60), (40, 50)])
def test_fp32_chains_are_short(device, b1, b2):
    """Many fp32 layers in one launch: random-sign products, so a chain of n
    roundings of 2^-24 leaves about 2^-24 sqrt(n / 2) of the scores.  Chains of 8
    steps (4 products each), one 64-bit sum over them, then at most 256 + 4
    partial sums by a tree of at most 32 in a row: sqrt(4 + 16) * 2^-24 = 2.7e-7,
    against 4.5e-7 and more for one chain over a range of 450 products."""
    from dattri_llm_amd import kernels

    gen = torch.Generator(device=device).manual_seed(b1)
    layers = [(torch.randn(b1, w, generator=gen, device=device), torch.randn(b2, w, generator=gen, device=device))
              for w in [16384] * 10 + [65536] * 3 + [131072]]
    want = sum(x.double() @ y.double().t() for x, y in layers)
    got = kernels.score_gemm(layers).double()
    assert float((got - want).norm() / want.norm()) <= 2.7e-7


@pytest.mark.parametrize("b1,b2,apart", [(3, 70, False), (64, 64, True), (130, 20, True)])
def test_fp32_layouts_in_one_call(device, monkeypatch, b1, b2, apart):
    """Row-major and k-blocked fp32 layers of one call, together and in a launch
    each: the row-major ones keep the streaming kernel where that pays."""
    from dattri_llm_amd import kernels

    gen = torch.Generator(device=device).manual_seed(b2)
    pairs = []
    for w, blocked in ((131072, False), (4096, True), (65536 + 4, False), (64, True)):
        m1, m2 = (torch.randn(b, w, generator=gen, device=device) for b in (b1, b2))
        pairs.append((kernels.blocked_storage(b1, w, torch.float32, m1.device).copy_(m1.view(b1, -1, 64))
                      if blocked else m1, m2))
    launches = []
    run = kernels._run
    monkeypatch.setattr(kernels, "_run", lambda dev, name, *a: (launches.append(name), run(dev, name, *a)))
    first = torch.randn(b1, b2, generator=gen, device=device)
    want = sum(x.reshape(b1, -1).double() @ y.double().t() for x, y in pairs)
    for order in (pairs, pairs[::-1]):
        launches.clear()
        got = kernels.score_gemm(order)
        assert len(launches) == 1 + apart
        assert float((got.double() - want).abs().max()) <= TOL * float(want.abs().max())
        got = kernels.score_gemm(order, out=first.clone(), accumulate=True)
        assert float((got.double() - want - first).abs().max()) <= TOL * float(want.abs().max())


@pytest.mark.parametrize("b1,b2,widths,bound", [
    (65, 129, [16384] * 10 + [65536] * 3 + [131072], 5.7e-7),
    (200, 512, [65536] * 4, 5.7e-7),
    (4096, 2048, [32768], 6.9e-7),
    (256, 256, [2048], 3.8e-7),
])
def test_fp32_chains_of_large_tiles(device, b1, b2, widths, bound):
    """The same on the 128 x 256 tile: chains of 128 steps, a second chain over
    at most 128 of them per share, and at most 32 + 8 partial planes in a row:
    2^-24 sqrt(64 + 4 + 20) = 5.6e-7, and with one share 2^-24 sqrt(64 + 64) =
    6.8e-7, against 1.3e-6 and 5.4e-6 for one chain per share.  A share of up to 8
    stages is one chain: 2^-24 sqrt(20 + 20) = 3.8e-7 for 40 steps."""
    from dattri_llm_amd import kernels

    gen = torch.Generator(device=device).manual_seed(b1)
    layers = [(torch.randn(b1, w, generator=gen, device=device), torch.randn(b2, w, generator=gen, device=device))
              for w in widths]
    print(f"score_gemm chains {b1}x{b2} of {sum(widths)}", flush=True)
    want = sum(x.double() @ y.double().t() for x, y in layers)
    got = kernels.score_gemm(layers).double()
    assert float((got - want).norm() / want.norm()) <= bound
