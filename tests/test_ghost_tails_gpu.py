"""Grouped ghost products whose last tiles run in pieces, against float64: few
and many tiles, groups of unlike lengths, ragged ends, empty samples, samples
of one row, offsets that start past row 0, both engines of fp32, and a
workspace without room for pieces.

Bounds: the products of the 16-bit factors are exact in fp32 and an fp32 sum of
n terms in any order is within n * 2^-24 of the sum of its magnitudes; with
random signs the error against the largest result stays under 1e-5 for the
sizes here, all dtypes."""

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = 1e-5


def _seg(gen, b, rows, start=0):
    cuts = torch.randint(start, rows + 1, (b - 1,), generator=gen).sort().values
    return torch.cat([torch.tensor([start]), cuts, torch.tensor([rows])]).to(torch.int32)


def _group(gen, device, dtype, rows, k, d, seg, index=False):
    phys = rows + 7 if index else rows
    a = torch.randn(phys, k, generator=gen) * 0.5
    g = torch.randn(phys, d, generator=gen) * 0.05
    idx = torch.randperm(phys, generator=gen)[:rows].to(torch.int32) if index else None
    return (a.to(device, dtype), g.to(device, dtype), seg.to(device), None if idx is None else idx.to(device))


def _packed(x, idx):
    return x.double() if idx is None else x.double()[idx.long()]


def _want(groups1, groups2, bias):
    out = 0
    for (a1, g1, s1, i1), (a2, g2, s2, i2) in zip(groups1, groups2):
        p = (_packed(a1, i1) @ _packed(a2, i2).t() + float(bias)) * (_packed(g1, i1) @ _packed(g2, i2).t())

        def ranges(s, n):
            m = torch.zeros(s.numel() - 1, n, dtype=torch.float64, device=p.device)
            for b, (x, y) in enumerate(zip(s[:-1].tolist(), s[1:].tolist())):
                m[b, x:y] = 1
            return m

        out = out + ranges(s1, p.shape[0]) @ p @ ranges(s2, p.shape[1]).t()
    return out


def _close(got, want):
    assert float((got.double() - want).abs().max()) <= TOL * float(want.abs().max())


CASES = {  # b1, b2, [(rows1, rows2, k, d), ...], first row
    "one tile": (3, 2, [(200, 100, 1024, 2048)], 0),
    "ragged": (7, 5, [(1054, 391, 4096, 1000)], 0),
    "single rows": (300, 130, [(300, 130, 2048, 2048)], 0),
    "past the first row": (5, 4, [(700, 300, 1536, 1536)], 77),
    "unlike groups": (6, 3, [(500, 260, 8192, 512), (129, 513, 640, 3200), (64, 1, 4096, 64), (30, 400, 72, 72)], 0),
    "a round and a bit": (9, 8, [(4100, 2100, 512, 520)], 0),
    "two rounds and a bit": (9, 8, [(4100, 2100, 512, 520), (4100, 2100, 520, 512), (260, 130, 4096, 4096)], 0),
}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("name", CASES)
def test_tails_match_float64(device, name, dtype):
    from dattri_llm_amd import kernels

    print(f"tails {name} {dtype}", flush=True)
    b1, b2, groups, start = CASES[name]
    gen = torch.Generator().manual_seed(7)
    index = name in ("ragged", "unlike groups")
    g_1, g_2 = [], []
    for r1, r2, k, d in groups:
        one = name == "single rows"
        s1 = torch.arange(r1 + 1, dtype=torch.int32) if one else _seg(gen, b1, r1, start)
        s2 = torch.arange(r2 + 1, dtype=torch.int32) if one else _seg(gen, b2, r2, start)
        g_1.append(_group(gen, device, dtype, r1, k, d, s1, index))
        g_2.append(_group(gen, device, dtype, r2, k, d, s2, index))
    want = _want(g_1, g_2, True)
    got = kernels.ghost_gram_grouped(g_1, g_2, bias=True)
    _close(got, want)
    assert torch.equal(got, kernels.ghost_gram_grouped(g_1, g_2, bias=True))
    _close(kernels.ghost_gram_grouped(g_1, g_2, bias=True, out=got, accumulate=True), 2 * want)


def test_tails_behind_values_that_cannot_be_split(device):
    """Scores decided by fp32 values below the split range, whose smaller parts a
    bf16 cannot hold: the fp32 launch takes every tile whole, each score as exact
    relative to itself."""
    from dattri_llm_amd import kernels

    gen = torch.Generator().manual_seed(3)
    g_1 = [_group(gen, device, torch.float32, 700, 1024, 2048, _seg(gen, 5, 700))]
    g_2 = [_group(gen, device, torch.float32, 300, 1024, 2048, _seg(gen, 4, 300))]
    for (a, g, seg, _idx), scale in ((g_1[0], 2.0**-122), (g_2[0], 2.0**45)):
        value = (a[:, 7].abs().clamp(max=1.0) + 1.0) * scale
        a.zero_()
        first = seg[:-1][seg[1:] > seg[:-1]].long()  # one row a sample
        a[first, 7] = value[first]
        g.abs_()
    want = _want(g_1, g_2, False)
    got = kernels.ghost_gram_grouped(g_1, g_2)
    assert bool((want > 0).any()) and bool((got[want == 0] == 0).all())
    assert float(((got.double() - want).abs() / want)[want > 0].max()) <= TOL


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_tails_without_room_run_whole(device, dtype):
    """A workspace below what the query asks for pieces: the same sums, tile by tile."""
    from dattri_llm_amd import _native as nat, kernels

    gen = torch.Generator().manual_seed(5)
    r1, r2, k, d, b1, b2 = 700, 300, 1024, 2048, 5, 4
    g_1 = [_group(gen, device, dtype, r1, k, d, _seg(gen, b1, r1))]
    g_2 = [_group(gen, device, dtype, r2, k, d, _seg(gen, b2, r2))]
    want = _want(g_1, g_2, False)
    lib, code, keep = nat.load(), nat.dtype_code(dtype), []
    es = nat.ELEM_BYTES[dtype]
    sides = [kernels._grouped_sides(g, nb, [k], [d], [0], 0, dtype, 16 // es, es, keep)
             for g, nb in ((g_1, b1), (g_2, b2))]
    ks, ds, need = (ctypes.c_int64 * 1)(k), (ctypes.c_int64 * 1)(d), ctypes.c_size_t()
    nat.check(lib.da_ghost_gram_grouped_workspace(sides[0], sides[1], 1, ks, ds, code, ctypes.byref(need)), "query")
    assert need.value > 256 * 128 * 4  # pieces planned
    ws = torch.empty(need.value, dtype=torch.uint8, device=device)
    for size in (need.value, need.value - 1, 65536):
        out = torch.empty(b1, b2, device=device)
        nat.check(lib.da_ghost_gram_grouped(sides[0], sides[1], 1, ks, ds, code, out.data_ptr(), b2, 0,
                                            ws.data_ptr(), size, nat.stream_ptr(out.device)), "grouped")
        _close(out, want)
    assert lib.da_ghost_gram_grouped(sides[0], sides[1], 1, ks, ds, code, out.data_ptr(), b2, 0, ws.data_ptr(), 16,
                                     nat.stream_ptr(out.device)) != 0
