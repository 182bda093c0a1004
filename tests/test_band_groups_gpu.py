"""The one-pass attention of long segments with one and with two groups of waves to a workgroup (csrc/mixers/band_attn.hip)
against 64 bits: no, one, an odd and an even number of key tiles, tiles without keys of theirs, a scale below zero."""
import pytest
import torch

from fasttalk_llm_microservice_amd.ops import mixers as M
from test_band_attention_gpu import DEV, cases, reference, segments

pytestmark = pytest.mark.gpu
LOW = torch.finfo(torch.float32).min


@pytest.mark.parametrize("name,sizes,opt,lens,pos0", [c for c in cases() if c[0] in (
    "causal, cap, sink 0", "window, kept, table", "sigmoid, distance", "two maps", "blocks")] + [
    ("one tile", dict(heads=4, kv_heads=1, dk=128, dv=128, window=0), {}, [64, 1], [0, 0]),
    ("three tiles, a sink each", dict(heads=4, kv_heads=4, dk=64, dv=128, window=0), dict(sinks=True), [33, 129], [159, 0]),
    ("below zero", dict(heads=2, kv_heads=2, dk=64, dv=64, window=0), dict(scale=-0.125), [140], [70])],
    ids=lambda v: v if isinstance(v, str) else "")
def test_groups(name, sizes, opt, lens, pos0, monkeypatch):
    g = torch.Generator().manual_seed(len(name))
    rnd = lambda *s: torch.randn(*s, generator=g)   # noqa: E731
    opt, hq = dict(opt), sizes["heads"] * opt.get("maps", 1)
    table, terms, sinks = opt.pop("table", 0), opt.pop("terms", False), opt.pop("sinks", False)
    if table:
        opt["dist_bias"] = (0.5 * rnd(table, hq)).to(DEV)
    if terms:
        opt.update({k: torch.rand(hq, generator=g).to(DEV) for k in ("r1", "r2", "pb")})
    if sinks:
        opt["sink"] = rnd(hq).to(DEV)
    sp = M.WindowSpec(**{"scale": sizes["dk"] ** -0.5, **sizes, **opt})
    seg, blocks = segments(lens, pos0, 16, g)
    kc = rnd(blocks, 16, sp.kv_heads * sp.maps * sp.dk).to(DEV, torch.bfloat16)
    vc = rnd(blocks, 16, sp.kv_heads * sp.dv).to(DEV, torch.bfloat16)
    q = (2.0 * rnd(sum(lens), hq * sp.dk)).to(DEV)
    want = reference(q, kc, vc, seg, sp, 32)
    # what a page holds past the last key counts for nothing
    for s in range(seg.num):
        kv = seg.host[2][s]
        if kv % 16:
            page = int(seg.block_tables[s, kv // 16])
            kc[page, kv % 16:] = float("nan")
            vc[page, kv % 16:] = float("nan")
    rows = torch.cat([torch.full((n,), n >= 32) for n in lens]).to(DEV)
    norm = float(want[rows].norm())
    monkeypatch.setattr(M, "_band_pays", lambda *a: True)
    for groups in (1, 2):
        monkeypatch.setattr(M, "_band_groups", lambda *a: groups)
        got = M.window_attention_products(torch.full((q.shape[0], hq, sp.dv), 7.0, device=DEV), q, kc, vc, seg, sp, 32)
        assert bool((got[~rows] == 7.0).all())
        # fp32 sums of a few hundred terms: about 2^-22
        assert float((got.double() - want)[rows].norm()) / norm < 1e-6


@pytest.mark.parametrize("rows,count,pos,window,groups", [(300, 1, 0, 0, 1), (777, 1, 0, 0, 2), (2048, 1, 0, 0, 2),
                                                          (8192, 1, 0, 0, 1), (64, 1, 8000, 0, 2), (100, 16, 0, 0, 1),
                                                          (2048, 1, 0, 512, 1)])
def test_rule(rows, count, pos, window, groups):
    start = [i * rows for i in range(count + 1)]
    seg = M.Segments(None, None, None, None, None, count, rows, pos + rows, host=(start, [pos] * count, [pos + rows] * count))
    assert M._band_groups(seg, M.WindowSpec(heads=16, kv_heads=4, dk=128, dv=128, window=window, scale=1.0), 32) == groups


@pytest.mark.parametrize("groups", [1, 2])
@pytest.mark.parametrize("opt", [{}, dict(softcap=5.0), dict(sink=LOW), dict(terms=True)], ids=str)
def test_lowest_biases(groups, opt, monkeypatch):
    """A distance table that masks with the type's lowest value: rows that see masked keys only weigh them all alike, others
    not at all."""
    opt = dict(opt)
    g = torch.Generator().manual_seed(2)
    if opt.pop("terms", False):
        opt.update({k: torch.rand(4, generator=g).to(DEV) for k in ("r1", "r2")})
    table = torch.full((300, 4), LOW, device=DEV)
    table[:, 1] = 0.25                        # a head that sees all
    table[3:, 2] = 0.5                        # one that does from a distance of 3 on: the first three rows see masked keys only
    table[:3, 3] = -0.5                       # one that sees no further: its first tiles are masked
    sp = M.WindowSpec(heads=4, kv_heads=2, dk=64, dv=64, window=0, scale=0.125, dist_bias=table, **opt)
    seg, blocks = segments([150, 70], [0, 0], 16, g)
    kc, vc = (torch.randn(blocks, 16, 128, generator=g).to(DEV, torch.bfloat16) for _ in range(2))
    q = torch.randn(220, 4, 64, generator=g).to(DEV)
    want = reference(q.view(220, 256), kc, vc, seg, sp, 32)
    alike = torch.zeros(220, 4, dtype=torch.bool, device=DEV)          # (64 bits tell such scores apart: their mean instead)
    alike[:, 0] = True
    alike[:3, 2] = alike[150:153, 2] = True
    for s, (a, b) in enumerate(((0, 150), (150, 220))):
        v = vc[seg.block_tables[s].long()].reshape(-1, 2, 64).double()
        mean = v.cumsum(0)[:b - a] / torch.arange(1, b - a + 1, device=DEV)[:, None, None]
        mean = mean.repeat_interleave(2, 1)
        want[a:b][alike[a:b]] = mean[alike[a:b]]
    if "sink" in opt:                        # the sink is as low: one more that weighs the same
        n = torch.cat([torch.arange(1, 151), torch.arange(1, 71)]).to(DEV)[:, None, None].double()
        want = torch.where(alike[:, :, None], want * n / (n + 1), want)
    monkeypatch.setattr(M, "_band_pays", lambda *a: True)
    monkeypatch.setattr(M, "_band_groups", lambda *a: groups)
    got = M.window_attention_products(torch.zeros(220, 4, 64, device=DEV), q.view(220, 256), kc, vc, seg, sp, 32)
    # fp32 sums of a few hundred terms: about 2^-22
    assert float((got.double() - want).norm() / want.norm()) < 1e-6


@pytest.mark.parametrize("lens,pos0", [([300], [0]), ([64], [3000])])
@pytest.mark.parametrize("groups", [1, 2])
def test_distance_terms_are_as_exact_as_the_products(lens, pos0, groups, monkeypatch):
    """Scores that are mostly logarithms of the distance: no further from 64 bits than the fp32 products with the library's."""
    g = torch.Generator().manual_seed(5)
    r1, r2 = (0.5 + torch.rand(4, generator=g)).to(DEV), (0.5 + torch.rand(4, generator=g)).to(DEV)
    sp = M.WindowSpec(heads=4, kv_heads=1, dk=128, dv=128, window=0, scale=128 ** -0.5, r1=r1, r2=r2)
    seg, blocks = segments(lens, pos0, 16, g)
    kc, vc = (torch.randn(blocks, 16, 128, generator=g).to(DEV, torch.bfloat16) for _ in range(2))
    q = (0.05 * torch.randn(sum(lens), 512, generator=g)).to(DEV)
    want = reference(q, kc, vc, seg, sp, 1)
    monkeypatch.setattr(M, "_band_pays", lambda *a: True)
    monkeypatch.setattr(M, "_band_groups", lambda *a: groups)
    new, old = (M.window_attention_products(torch.zeros(sum(lens), 4, 128, device=DEV), q, k, v, seg, sp, 1)
                for k, v in ((kc, vc), (kc.float(), vc.float())))
    e_new, e_old = (float((x.double() - want).norm() / want.norm()) for x in (new, old))
    assert e_new < 1.05 * e_old, (e_new, e_old)


@pytest.mark.parametrize("groups", [1, 2])
@pytest.mark.parametrize("opt", [{}, dict(softcap=5.0), dict(table=True)], ids=str)
@pytest.mark.parametrize("sink", [float("inf"), torch.finfo(torch.float32).max, LOW, -float("inf")])
def test_extreme_sinks(groups, opt, sink, monkeypatch):
    """A sink far above all scores takes all of the weight, one far below none."""
    g = torch.Generator().manual_seed(6)
    extra = dict(dist_bias=torch.randn(40, 4, generator=g).to(DEV)) if opt.get("table") else opt
    sp = M.WindowSpec(heads=4, kv_heads=2, dk=64, dv=64, window=0, scale=0.125, sink=sink, **extra)
    seg, blocks = segments([150, 70], [0, 9], 16, g)
    kc, vc = (torch.randn(blocks, 16, 128, generator=g).to(DEV, torch.bfloat16) for _ in range(2))
    q = torch.randn(220, 256, generator=g).to(DEV)
    monkeypatch.setattr(M, "_band_pays", lambda *a: True)
    monkeypatch.setattr(M, "_band_groups", lambda *a: groups)
    got = M.window_attention_products(torch.full((220, 4, 64), 7.0, device=DEV), q, kc, vc, seg, sp, 32)
    if sink > 0:
        assert bool((got == 0).all())
    else:
        want = reference(q, kc, vc, seg, M.WindowSpec(heads=4, kv_heads=2, dk=64, dv=64, window=0, scale=0.125, **extra), 32)
        assert float((got.double() - want).norm() / want.norm()) < 1e-6       # fp32 sums of a few hundred terms: about 2^-22
