"""Expert routing around its limits, bit for bit against torch on the CPU."""

import pytest
import torch

from dattri_llm_amd import kernels

pytestmark = pytest.mark.gpu


# Steps are 8192 entries of up to 8192 (slot, sample) blocks; more blocks (k > experts)
# take the by-expert sort and one wave per expert.
@pytest.mark.parametrize("batch,tokens,experts,k", [(1, 1, 1, 1), (1, 63, 3, 2), (1, 8191, 2, 1), (1, 8193, 2, 1),
                                                    (3, 4097, 5, 2), (7, 1, 8, 8), (2048, 2, 4, 4), (2730, 3, 3, 3),
                                                    (2730, 3, 3, 4), (8192, 1, 1, 2), (512, 5, 2, 16), (513, 5, 2, 16)])
def test_route(batch, tokens, experts, k):
    n = batch * tokens
    gen = torch.Generator().manual_seed(n + k)
    idx = torch.randint(-1, experts + 1, (n, k), generator=gen)  # out-of-range entries are dropped
    print(f"route {batch} x {tokens}, {experts} experts, k = {k}", flush=True)
    offsets, entries, seg, rows = (x.cpu() for x in kernels.moe_route(idx.cuda(), experts, batch, tokens))
    keys, start = idx.t().flatten(), 0
    for e in range(experts):
        p = (keys == e).nonzero().flatten()
        sample = p % n // tokens
        assert offsets[e] == start
        assert torch.equal(entries[start:start + p.numel()].long(), p)
        assert torch.equal(rows[start:start + p.numel()].long(), sample.sort(stable=True).indices)
        want = torch.nn.functional.pad(torch.bincount(sample, minlength=batch).cumsum(0), (1, 0))
        assert torch.equal(seg[e].long(), want)
        start += p.numel()
    assert offsets[experts] == start
