"""fp32 products on the 16-bit matrix pipe (three-part split rows): the ghost,
diagonal, grouped and per-token forms against float64, at widths that end
inside a stage, and the values the parts cannot hold (infinities, NaN, the
ends of the exponent range), which the fp32 kernels must take over whole.

Bounds: an fp32 dot product of n terms summed in any order is within n * 2^-24
of the sum of its magnitudes; with random signs the error against the largest
result stays under 1e-5 for the sizes here (the bound the fp32 kernels are held
to).  Results with infinities are compared entry by entry with torch's fp32
result on the CPU: the same entries are infinite or NaN."""

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = 1e-5
SHAPES = [  # b1, t1, b2, t2, k, d
    (6, 256, 4, 128, 1024, 1028),
    (5, 300, 3, 270, 772, 2048),
    (9, 257, 2, 129, 2052, 516),
]


def _factors(device, b1, t1, b2, t2, k, d, seed=0):
    gen = torch.Generator(device=device).manual_seed(seed)

    def rnd(*s):
        return torch.randn(*s, generator=gen, device=device)

    return rnd(b1, t1, k), rnd(b1, t1, d) * 0.03, rnd(b2, t2, k), rnd(b2, t2, d) * 0.03


def _per_token_ref(a1, g1, a2, g2, bias, dtype=torch.float64):
    out = []
    for j in range(a2.shape[0]):
        ka = a1.to(dtype) @ a2[j].to(dtype).t() + float(bias)
        out.append((ka * (g1.to(dtype) @ g2[j].to(dtype).t())).sum(-1))
    return torch.stack(out, -1)  # (B1, T1, B2)


def _is_split(a1, a2, k, d, diag=False):
    """The workspace query asks for the split copies."""
    from dattri_llm_amd import _native as nat, kernels

    need = ctypes.c_size_t()
    s1, s2 = kernels._side(a1, a1, False), kernels._side(a2, a2, False)
    query = nat.load().da_ghost_gram_diag_workspace if diag else nat.load().da_ghost_gram_workspace
    nat.check(query(s1, s2, k, d, nat.DA_F32, ctypes.byref(need)), "query")
    return need.value > 6 * (a1.shape[0] * a1.shape[1] + a2.shape[0] * a2.shape[1]) * (k + d)


def _close(got, want):
    assert float((got.double() - want).abs().max()) <= TOL * float(want.abs().max())


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("shape", SHAPES)
def test_split_forms_match_float64(device, shape, bias):
    from dattri_llm_amd import kernels

    b1, t1, b2, t2, k, d = shape
    a1, g1, a2, g2 = _factors(device, *shape)
    print(f"split {shape} bias={bias}", flush=True)
    assert _is_split(a1, a2, k, d)
    per_token = _per_token_ref(a1, g1, a2, g2, bias)
    _close(kernels.ghost_gram(a1, g1, a2, g2, bias=bias), per_token.sum(1))
    _close(kernels.ghost_gram_per_token(a1, g1, a2, g2, bias=bias), per_token)
    n = min(b1, b2)
    own = torch.stack([_per_token_ref(a1[i:i + 1], g1[i:i + 1], a1[i:i + 1], g1[i:i + 1], bias).sum()
                       for i in range(n)])
    _close(kernels.ghost_gram_diag(a1[:n], g1[:n], a1[:n], g1[:n], bias=bias), own)


def test_split_strided_and_sequence_first_sides(device):
    from dattri_llm_amd import kernels

    a1, g1, a2, g2 = _factors(device, 6, 256, 4, 128, 1024, 1024, seed=2)
    want = _per_token_ref(a1, g1, a2, g2, False).sum(1)
    wide = torch.zeros(6, 256, 1536, device=device)
    wide[..., 256:1280] = a1
    seq = g2.transpose(0, 1).contiguous().transpose(0, 1)
    _close(kernels.ghost_gram(wide[..., 256:1280], g1, a2, seq), want)


@pytest.mark.parametrize("indexed", [False, True])
def test_split_grouped_rows(device, indexed):
    """Groups of different widths, ragged and empty samples, rows through an
    index, fewer live rows than the factors hold; more matrices than one
    pre-pass takes."""
    from dattri_llm_amd import kernels

    gen = torch.Generator(device=device).manual_seed(4)
    widths = [(1024, 520), (516, 1028)] * 7
    counts = [((300, 0, 41), (130, 60)), ((5, 250, 9), (200, 3))] * 7
    groups1, groups2 = [], []
    want = torch.zeros(3, 2, dtype=torch.float64, device=device)
    for (k, d), (n1, n2) in zip(widths, counts):
        sides = []
        for n in (n1, n2):
            live = sum(n)
            rows = live + 17  # rows past the last segment, never part of a sample
            a, g = (torch.randn(rows, w, generator=gen, device=device) for w in (k, d))
            seg = torch.tensor([0, *torch.tensor(n).cumsum(0).tolist()], dtype=torch.int32, device=device)
            order = torch.randperm(rows, generator=gen, device=device) if indexed else torch.arange(rows, device=device)
            sides.append((a, g, seg, order.to(torch.int32) if indexed else None, order, n))
        (a1, g1, s1, i1, o1, c1), (a2, g2, s2, i2, o2, c2) = sides
        x1, y1, x2, y2 = a1[o1].double(), g1[o1].double(), a2[o2].double(), g2[o2].double()
        prod = (x1[:sum(c1)] @ x2[:sum(c2)].t() + 1.0) * (y1[:sum(c1)] @ y2[:sum(c2)].t())
        want += torch.stack([torch.stack([q.sum() for q in p.split(list(c2), 1)]) for p in prod.split(list(c1), 0)])
        groups1.append((a1, g1, s1, i1))
        groups2.append((a2, g2, s2, i2))
    print(f"split grouped indexed={indexed}", flush=True)
    _close(kernels.ghost_gram_grouped(groups1, groups2, bias=True), want)


def test_index_past_the_packed_rows(device):
    """The C entry told only the packed row count, its index naming rows of a
    larger capture: the split route reads the rows the index names."""
    from dattri_llm_amd import _native as nat, kernels

    b, t, k, d, rows = 24, 64, 1024, 1028, 9001
    gen = torch.Generator(device=device).manual_seed(8)
    a, g = (torch.randn(rows, w, generator=gen, device=device) for w in (k, d))
    index = torch.randperm(rows, generator=gen, device=device)[:b * t].to(torch.int32)
    seg = torch.arange(0, b * t + 1, t, dtype=torch.int32, device=device)
    x, y = (m[index.long()].double().view(b, t, -1) for m in (a, g))
    want = _per_token_ref(x, y, x, y, False).sum(1)
    lib, need = nat.load(), ctypes.c_size_t()
    side = (nat.FactorSide * 1)(kernels._side(a, g, False, seg, index, b * t))  # b * t packed rows, not 9001
    ks, ds = (ctypes.c_int64 * 1)(k), (ctypes.c_int64 * 1)(d)
    nat.check(lib.da_ghost_gram_grouped_workspace(side, side, 1, ks, ds, nat.DA_F32, ctypes.byref(need)), "query")
    assert need.value > 6 * b * t * (k + d)  # the split copies are in it
    ws, out = torch.empty(need.value, dtype=torch.uint8, device=device), torch.empty(b, b, device=device)
    nat.check(lib.da_ghost_gram_grouped(side, side, 1, ks, ds, nat.DA_F32, out.data_ptr(), b, 0, ws.data_ptr(),
                                        need.value, nat.stream_ptr(out.device)), "grouped")
    _close(out, want)


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 3.4e38, 1e-38, 1e-44])
@pytest.mark.parametrize("place", ["a1", "g2"])
def test_values_the_parts_cannot_hold(device, value, place):
    from dattri_llm_amd import kernels

    shape = (6, 256, 4, 128, 512, 512)
    f = dict(zip(("a1", "g1", "a2", "g2"), _factors(device, *shape, seed=3)))
    assert _is_split(f["a1"], f["a2"], 512, 512)
    f[place][2, 17, 40] = value
    f[place][1, 3] = 0.0
    args = (f["a1"], f["g1"], f["a2"], f["g2"])
    got = kernels.ghost_gram(*args).cpu()
    tok = kernels.ghost_gram_per_token(*args).cpu()
    want = _per_token_ref(*(x.cpu() for x in args), False, dtype=torch.float32)
    for g, w in ((tok, want), (got, want.sum(1))):
        assert torch.equal(torch.isnan(g), torch.isnan(w))
        assert torch.equal(torch.isposinf(g), torch.isposinf(w)) and torch.equal(torch.isneginf(g), torch.isneginf(w))
        ok = torch.isfinite(w)
        assert float((g[ok] - w[ok]).abs().max()) <= 4 * TOL * float(w[ok].abs().max())


def test_split_rows_of_every_scale(device):
    """Samples scaled from 2^-45 to 2^45 per factor: every pair's score is as
    exact, relative to itself, as at scale one."""
    from dattri_llm_amd import kernels

    a1, g1, a2, g2 = _factors(device, 7, 256, 5, 128, 512, 512, seed=6)
    s = (2.0 ** torch.arange(-45, 46, 15, device=device, dtype=torch.float32)).view(-1, 1, 1)
    assert _is_split(a1, a2, 512, 512)
    want = _per_token_ref(a1, g1, a2, g2, False).sum(1)
    got = kernels.ghost_gram(a1 * s, g1, a2, g2).double() / s.view(-1, 1)
    assert float(((got - want).abs().amax(1) / want.abs().amax(1)).max()) <= TOL


def _forms(a1, g1, a2, g2):
    """The ghost, per-token, diagonal and grouped products of one layer."""
    from dattri_llm_amd import kernels

    def packed(a, g):
        b, t = a.shape[:2]
        seg = torch.arange(0, b * t + 1, t, dtype=torch.int32, device=a.device)
        return a.reshape(b * t, -1), g.reshape(b * t, -1), seg, None

    n = min(a1.shape[0], a2.shape[0])
    assert _is_split(a1, a2, a1.shape[-1], g1.shape[-1]) and _is_split(a1[:n], a2[:n], a1.shape[-1], g1.shape[-1], True)
    return {"ghost": kernels.ghost_gram(a1, g1, a2, g2),
            "per token": kernels.ghost_gram_per_token(a1, g1, a2, g2).sum(1),
            "grouped": kernels.ghost_gram_grouped([packed(a1, g1)], [packed(a2, g2)]),
            "diagonal": kernels.ghost_gram_diag(a1[:n], g1[:n], a2[:n], g2[:n])}


def _of_form(want, name):
    return want.diagonal()[:min(want.shape)] if name == "diagonal" else want


@pytest.mark.parametrize("log1,log2", [(70, 69), (100, 100), (64, 62.5), (62, 60)])
def test_products_past_the_range(device, log1, log2):
    """Every entry in range, one product a pair that leaves the fp32 range, ends
    just inside it or is near it: infinities where fp32 has them, nowhere NaN."""
    shape = (33, 256, 24, 128, 512, 512)
    a1, g1, a2, g2 = _factors(device, *shape, seed=11)
    x, y = (torch.rand(a.shape[0], generator=torch.Generator().manual_seed(n)) + 0.5 for a, n in ((a1, 1), (a2, 2)))
    x, y = x * 2.0**log1, y * 2.0**log2
    for a, v in ((a1, x), (a2, y)):
        a.zero_()
        a[:, 5, 9] = v.to(device)
    kg = (g1[:, 5].double() @ g2[:, 5].double().t()).cpu()
    ka = x[:, None] * y  # fp32, one rounding as in any kernel
    want = ka * kg.float()
    near = (ka.double() * kg).abs().sub(2.0**128).abs() < 2.0**115  # kg may round past the end either way
    bound = TOL * float((x[:, None].double() * y).max() * kg.abs().max())
    for name, got in _forms(a1, g1, a2, g2).items():
        got, w, skip = got.cpu(), _of_form(want, name), _of_form(near, name)
        assert not bool(got.isnan().any()) and torch.equal(got.sign(), w.sign()), name
        assert torch.equal(got.isinf() | skip, w.isinf() | skip), name
        ok = w.isfinite() & got.isfinite()
        assert bool(((got.double() - w.double()).abs()[ok] <= bound).all()), name


def test_tiny_values_decide(device):
    """One product a pair, of an entry near 2^-122 whose smaller parts a bf16
    cannot hold: each score as exact, relative to itself, as at scale one."""
    a1, g1, a2, g2 = (x.abs() + 0.1 for x in _factors(device, 33, 256, 24, 128, 512, 512, seed=12))
    for a, scale in ((a1, 2.0**-122), (a2, 2.0**45)):
        v = (a[:, 5, 9].clamp(max=1.0) + 1.0) * scale
        a.zero_()
        a[:, 5, 9] = v
    want = _per_token_ref(a1, g1, a2, g2, False).sum(1)
    for name, got in _forms(a1, g1, a2, g2).items():
        w = _of_form(want, name)
        assert float(((got.double() - w).abs() / w).max()) <= TOL, name


def test_without_room_for_the_copies(device, monkeypatch):
    """Where the GPU has no room for the split copies the calls run the fp32
    kernels in the workspace those need; without that they fail as before."""
    from dattri_llm_amd import _native as nat, kernels

    a1, g1, a2, g2 = _factors(device, 33, 256, 24, 128, 512, 512, seed=13)
    wide = [torch.randn(16, 400, 1024, device=device, generator=torch.Generator(device=device).manual_seed(n))
            for n in (1, 2)]
    whole = _forms(a1, g1, a2, g2)
    dense = kernels.materialize_linear(*wide)
    refused, allowed, take = [], [1 << 20], nat.workspace

    def scarce(nbytes, dev):
        if nbytes > allowed[0]:
            refused.append(nbytes)
            raise torch.OutOfMemoryError("no room")
        return take(nbytes, dev)

    monkeypatch.setattr(nat, "workspace", scarce)
    per_token = _per_token_ref(a1, g1, a2, g2, False)
    for name, got in _forms(a1, g1, a2, g2).items():
        _close(got, _of_form(per_token.sum(1), name))
        assert not torch.equal(got, whole[name]), name  # other kernels
    want = torch.stack([y.double().t() @ x.double() for x, y in zip(*wide)]).flatten(1)
    _close(kernels.materialize_linear(*wide), want)
    _close(dense, want)
    assert len(refused) == 5 and min(refused) > 6 * (33 * 256 + 24 * 128) * 512
    allowed[0] = 8
    with pytest.raises(torch.OutOfMemoryError):
        kernels.ghost_gram(a1, g1, a2, g2)
