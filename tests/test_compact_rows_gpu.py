"""Row compaction against torch's nonzero: whole numbers, bit for bit."""

import pytest
import torch

from dattri_llm_amd import kernels

pytestmark = pytest.mark.gpu


# A step is 1024 threads of 16 rows: around one row, one thread, one wave, one and
# several steps; samples of one row, shorter than a thread's run and across steps.
@pytest.mark.parametrize("batch,tokens", [(1, 1), (3, 5), (1, 16), (17, 1), (2, 512), (64, 16), (1, 1024), (16383, 1),
                                          (1, 16384), (5, 3277), (1, 16385), (7, 7001), (3, 32768), (4, 0), (0, 4)])
@pytest.mark.parametrize("share", [0.0, 0.1, 0.85, 1.0])
@pytest.mark.parametrize("shift", [0, 1])  # off a 16-byte boundary: byte loads
def test_compact_rows(batch, tokens, share, shift):
    gen = torch.Generator().manual_seed(batch * 131 + tokens)
    n = batch * tokens
    mask = torch.rand(n + shift, generator=gen)[shift:] < share
    store = torch.zeros(n + shift, dtype=torch.bool, device="cuda")
    store[shift:] = mask.cuda()
    seg, rows = kernels.compact_rows(store[shift:], batch, tokens)
    want = mask.nonzero().flatten()
    counts = mask.view(batch, tokens).sum(1) if n else torch.zeros(batch, dtype=torch.int64)
    assert seg.cpu().tolist() == [0, *counts.cumsum(0).tolist()]
    assert torch.equal(rows[: want.numel()].cpu().long(), want)
