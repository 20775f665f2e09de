"""Router top-k where the order is unique, where ties fall inside or at the edge of the k largest, and rows of
both in one wave, against torch on the CPU."""

import pytest
import torch

from dattri_llm_amd import kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("e,k", [(1, 1), (2, 2), (7, 3), (8, 8), (9, 1), (64, 8), (128, 16), (129, 5), (256, 16)])
@pytest.mark.parametrize("n", [1, 31, 65, 400])
def test_topk(e, k, n):
    gen = torch.Generator().manual_seed(e * 31 + k * 7 + n)
    # whole steps of 1/32 apart: far more than a rounding of the probabilities, so ties are the planted ones
    x = torch.rand(n, e, generator=gen).argsort(-1).float() / 32
    order = x.argsort(-1, descending=True)
    for row in range(0, n, 3):  # a tie between places j and j + 1, the last of them the edge (k - 1, k) where there is one
        j = int(torch.randint(0, min(k, e - 1), (1,), generator=gen)) if e > 1 else None
        if j is not None:
            x[row, order[row, j + 1]] = x[row, order[row, j]]
    print(f"topk {n} x {e}, k = {k}", flush=True)
    w, idx = kernels.moe_topk(x.cuda(), k)
    tv, ti = torch.topk(torch.softmax(x, -1), k, dim=-1)
    assert torch.equal(idx.cpu(), ti)
    torch.testing.assert_close(w.cpu(), tv / tv.sum(-1, keepdim=True), rtol=1e-5, atol=1e-7)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("e,k", [(12, 12), (13, 13), (64, 12), (64, 13), (128, 16), (129, 13), (256, 16)])
def test_topk_16_bit(e, k, dtype):
    """16-bit logits with the ties that rounding gives them, both sides of the
    lines where the passes are skipped."""
    gen = torch.Generator().manual_seed(e + k)
    # multiples of 2^-5 below 4: exact in both types, so equal logits are the only equal probabilities
    x = (torch.randint(-127, 128, (333, e), generator=gen) / 32).to(dtype)
    print(f"topk {dtype} {e} experts, k = {k}", flush=True)
    w, idx = kernels.moe_topk(x.cuda(), k)
    tv, ti = torch.topk(torch.softmax(x.float(), -1), k, dim=-1)
    assert torch.equal(idx.cpu(), ti)
    torch.testing.assert_close(w.cpu(), tv / tv.sum(-1, keepdim=True), rtol=1e-5, atol=1e-7)
