"""The one-pass attention of long segments (csrc/mixers/band_attn.hip) against the same attention in
64 bits: every mask and score term, at the edges of its tiles (64 keys, 16 pairs a wave, 64 and 128 a
workgroup), several segments with short ones among them.  Its error may not exceed that of the
banded fp32 products it stands for."""
import math

import pytest
import torch

from fasttalk_llm_microservice_amd.ops import mixers as M

pytestmark = pytest.mark.gpu
DEV = "cuda"


def segments(lens, pos0, bs, g):
    start = [0]
    for n in lens:
        start.append(start[-1] + n)
    kv = [p + n for p, n in zip(pos0, lens)]
    nb = [-(-k // bs) for k in kv]
    perm = torch.randperm(sum(nb), generator=g).int()
    bt = torch.zeros(len(lens), max(nb), dtype=torch.int32)
    at = 0
    for i, k in enumerate(nb):
        bt[i, :k] = perm[at:at + k]
        at += k
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)   # noqa: E731
    return M.Segments(i32(start), i32(pos0), i32([0] * len(lens)), i32(kv), bt.to(DEV), len(lens), max(lens), max(kv),
                      host=(start, list(pos0), kv)), sum(nb)


def reference(q, kc, vc, seg, sp, min_rows):
    out = torch.zeros(q.shape[0], sp.heads * sp.maps, sp.dv, dtype=torch.float64, device=DEV)
    bs, rep, d64 = kc.shape[1], sp.heads // sp.kv_heads, torch.float64
    par = lambda t: None if t is None else t.to(d64)   # noqa: E731
    for s in range(seg.num):
        a, b = seg.host[0][s], seg.host[0][s + 1]
        if b - a < min_rows:
            continue
        p0, kv = seg.host[1][s], seg.host[2][s]
        pages = seg.block_tables[s, :-(-kv // bs)].long()
        k = kc[pages].reshape(-1, sp.kv_heads * sp.maps, sp.dk)[:kv].to(d64)
        v = vc[pages].reshape(-1, sp.kv_heads, sp.dv)[:kv].to(d64)
        i = torch.arange(p0, p0 + b - a, device=DEV)[:, None]
        j = torch.arange(kv, device=DEV)[None]
        seen = j <= i
        if sp.window > 0:
            near = (i // sp.window == j // sp.window) if sp.blocks else (i - j < sp.window)
            seen = seen & (near | (j < sp.keep_first))
        d = (i - j).clamp_min(0)
        for h in range(sp.heads):
            for m in range(sp.maps):
                x = h * sp.maps + m
                z = q[a:b].view(b - a, -1, sp.dk)[:, x].to(d64) @ k[:, h // rep * sp.maps + m].T * sp.scale
                if sp.softcap:
                    z = sp.softcap * torch.tanh(z / sp.softcap)
                if sp.r1 is not None:
                    z = z - par(sp.r1)[x] * torch.log1p(par(sp.r2)[x] * d)
                if sp.dist_bias is not None:
                    z = z + par(sp.dist_bias)[d.clamp_max(sp.dist_bias.shape[0] - 1), x]
                if sp.sigmoid:
                    w = torch.sigmoid(z + (par(sp.pb)[x] if sp.pb is not None else 0.0)) * seen
                else:
                    z = z.masked_fill(~seen, -math.inf)
                    if sp.sink is not None:
                        sk = par(sp.sink)[x] if isinstance(sp.sink, torch.Tensor) else torch.tensor(sp.sink, dtype=d64, device=DEV)
                        z = torch.cat([z, sk.expand(b - a, 1)], 1)
                    w = torch.softmax(z, -1)[:, :kv]
                out[a:b, x] = w @ v[:, h // rep]
    return out


def cases():
    f = lambda *s: dict(zip(("heads", "kv_heads", "dk", "dv", "window"), s))   # noqa: E731
    yield "causal", f(4, 1, 128, 128, 0), {}, [64], [0]
    yield "causal, cap, sink 0", f(4, 2, 128, 128, 0), dict(softcap=30.0, sink=0.0), [200, 5, 33], [0, 7, 100]
    yield "window", f(3, 1, 64, 128, 100), {}, [65, 130], [0, 301]
    yield "window, kept, table", f(4, 2, 128, 128, 70), dict(keep_first=9, table=90), [300, 32], [0, 511]
    yield "window, kept beyond a tile", f(2, 2, 64, 64, 40), dict(keep_first=130), [257], [64]
    yield "blocks", f(4, 1, 128, 64, 96), dict(blocks=True), [191, 97], [95, 0]
    yield "two maps", f(4, 2, 64, 128, 128), dict(maps=2), [129, 63], [0, 1000]
    yield "sigmoid, distance", f(2, 1, 128, 128, 150), dict(sigmoid=True, terms=True), [260], [31]
    yield "sink per head, one key head each", f(2, 2, 128, 128, 33), dict(sinks=True), [32, 70], [0, 640]
    yield "many pairs (eight waves)", f(16, 4, 128, 128, 0), dict(softcap=20.0), [1024], [0]
    yield "three heads a group, many pairs", f(48, 16, 64, 64, 256), {}, [700, 400], [0, 90]


@pytest.mark.parametrize("name,sizes,opt,lens,pos0", list(cases()), ids=[c[0] for c in cases()])
@pytest.mark.parametrize("bs", [4, 16])
def test_against_64_bits(name, sizes, opt, lens, pos0, bs, monkeypatch):
    g = torch.Generator().manual_seed(len(name) * 10 + bs)
    rnd = lambda *s: torch.randn(*s, generator=g)   # noqa: E731
    opt = dict(opt)
    hq = sizes["heads"] * opt.get("maps", 1)
    table, terms, sinks = opt.pop("table", 0), opt.pop("terms", False), opt.pop("sinks", False)
    extra = {}
    if table:
        extra["dist_bias"] = (0.5 * rnd(table, hq)).to(DEV)
    if terms:
        extra.update({k: torch.rand(hq, generator=g).to(DEV) for k in ("r1", "r2", "pb")})
    if sinks:
        extra["sink"] = rnd(hq).to(DEV)
    sp = M.WindowSpec(scale=sizes["dk"] ** -0.5, **sizes, **opt, **extra)
    seg, blocks = segments(lens, pos0, bs, g)
    kc = rnd(blocks, bs, sp.kv_heads * sp.maps * sp.dk).to(DEV, torch.bfloat16)
    vc = rnd(blocks, bs, sp.kv_heads * sp.dv).to(DEV, torch.bfloat16)
    q = (2.0 * rnd(sum(lens), hq * sp.dk)).to(DEV)
    want = reference(q, kc, vc, seg, sp, 32)
    out = torch.full((q.shape[0], hq, sp.dv), 7.0, device=DEV)
    assert M.band_attention_ok(out, q, kc, vc, seg, sp) and M._band_pays(seg, sp, 32)
    got = M.window_attention_products(out, q, kc, vc, seg, sp, 32)
    rows = torch.cat([torch.full((n,), n >= 32) for n in lens]).to(DEV)
    assert bool((got[~rows] == 7.0).all())                     # short segments are not this path's
    # the same attention as fp32 products on widened caches (another path of the same function)
    old = M.window_attention_products(torch.zeros_like(out), q, kc.float(), vc.float(), seg, sp, 32)
    norm = float(want[rows].norm())
    e_new, e_old = (float((x.double() - want)[rows].norm()) / norm for x in (got, old))
    # fp32 sums of a few hundred terms: about 2^-22; no further from 64 bits than the products
    assert e_new < 1e-6 and e_new < 1.5 * e_old + 1e-7, (e_new, e_old)
    again = M.window_attention_products(torch.zeros_like(out), q, kc, vc, seg, sp, 32)
    assert torch.equal(again[rows], got[rows])
    half = M.window_attention_products(torch.zeros_like(out, dtype=torch.bfloat16), q, kc, vc, seg, sp, 32)
    assert torch.equal(half[rows], got[rows].bfloat16())       # rounded once, on the way out


def off_by_one(x):
    """x at an address two or four bytes past a 16-byte boundary"""
    flat = torch.empty(x.numel() + 1, dtype=x.dtype, device=x.device)[1:]
    return flat.copy_(x.flatten()).view(x.shape)


@pytest.mark.parametrize("form", ["q columns", "q off", "q heads apart", "k off", "v off", "k pages apart", "out rows apart",
                                  "out off", "wide tables", "table columns", "start apart"])
def test_operands_of_other_layouts(form):
    """Operands that are not dense or not aligned: the banded products take them."""
    g = torch.Generator().manual_seed(3)
    sp = M.WindowSpec(heads=4, kv_heads=2, dk=64, dv=64, window=0, scale=0.125)
    seg, blocks = segments([40, 3, 65], [9, 0, 30], 4, g)
    kc, vc = (torch.randn(blocks, 4, 128, generator=g).to(DEV, torch.bfloat16) for _ in range(2))
    q = torch.randn(108, 256, generator=g).to(DEV)
    out = torch.full((108, 4, 64), 7.0, device=DEV)
    want = M.window_attention_products(out.clone(), q, kc, vc, seg, sp, 32)
    if form == "q columns":
        q = torch.cat([q, q], 1)[:, 256:]
    elif form == "q off":
        q = off_by_one(q)
    elif form == "q heads apart":
        q = q.view(108, 4, 64)
    elif form == "k off":
        kc = off_by_one(kc)
    elif form == "v off":
        vc = off_by_one(vc)
    elif form == "k pages apart":
        kc = torch.cat([kc, kc], 1)[:, 4:]
    elif form == "out rows apart":
        out = torch.full((108, 8, 64), 7.0, device=DEV)[:, 4:]
    elif form == "out off":
        out = off_by_one(out)
    elif form == "wide tables":
        seg.block_tables = seg.block_tables.long()
    elif form == "table columns":
        seg.block_tables = torch.cat([seg.block_tables, seg.block_tables], 1)[:, :seg.block_tables.shape[1]]
    else:
        seg.start = torch.stack([seg.start, seg.start], 1)[:, 0]
    got = M.window_attention_products(out, q, kc, vc, seg, sp, 32)
    # both forms are within 1e-6 of the sums in 64 bits (test_against_64_bits)
    torch.testing.assert_close(got, want, rtol=0, atol=2e-6 * float(want.abs().max()))


@pytest.mark.parametrize("kind", ["cap", "sigmoid", "two maps, cap"])
@pytest.mark.parametrize("n", [40, 3], ids=["long", "decode"])
def test_infinite_queries(kind, n):
    """Queries of +-inf, or that only bf16 rounds to it: scores of +-inf, which a cap and a sigmoid map to finite ones."""
    g = torch.Generator().manual_seed(8)
    opt = {"cap": dict(softcap=5.0, blocks=True), "sigmoid": dict(sigmoid=True), "two maps, cap": dict(softcap=5.0, maps=2)}[kind]
    sp = M.WindowSpec(heads=4, kv_heads=2, dk=64, dv=64, window=100, scale=0.125, **opt)
    seg, blocks = segments([n, n], [9, 130], 8, g)
    kc = torch.randn(blocks, 8, 128 * sp.maps, generator=g).to(DEV, torch.bfloat16)
    vc = torch.randn(blocks, 8, 128, generator=g).to(DEV, torch.bfloat16)
    q = torch.randn(2 * n, 4 * sp.maps * 64, generator=g).to(DEV)
    q[0, 5], q[1, 70], q[n + 1, 64 * 4 * sp.maps - 1] = float("inf"), -float("inf"), 3.4e38
    assert bool((kc != 0).all())
    out = torch.full((2 * n, 4 * sp.maps, 64), 7.0, device=DEV)
    want = reference(q, kc, vc, seg, sp, 1)
    got = M.window_attention_products(out, q, kc, vc, seg, sp, 32) if n >= 32 else M.window_attention(q, kc, vc, seg, sp, out=out)
    assert bool(want.isfinite().all())
    assert float((got.double() - want).norm() / want.norm()) < 1e-6       # fp32 sums, as test_against_64_bits


@pytest.mark.parametrize("opt", [{}, dict(sink=0.5), dict(window=40, keep_first=3), dict(sigmoid=True)])
def test_segments_without_keys(opt):
    """A long segment whose context is empty (the first, so that nothing lies before its pages' ids): zeros."""
    g = torch.Generator().manual_seed(4)
    sp = M.WindowSpec(**{**dict(heads=4, kv_heads=2, dk=64, dv=64, window=0, scale=0.125), **opt})
    seg, blocks = segments([33, 40, 3], [0, 9, 5], 4, g)
    seg.host[2][0] = 0
    seg.kv_len[0] = 0
    kc, vc = (torch.randn(blocks, 4, 128, generator=g).to(DEV, torch.bfloat16) for _ in range(2))
    q = torch.randn(76, 256, generator=g).to(DEV)
    out = torch.full((76, 4, 64), 7.0, device=DEV)
    assert M.band_attention_ok(out, q, kc, vc, seg, sp) and M._band_pays(seg, sp, 32)
    got = M.window_attention_products(out, q, kc, vc, seg, sp, 32)
    want = reference(q, kc, vc, seg, sp, 40)
    assert bool((got[:33] == 0).all()) and bool((got[73:] == 7.0).all())
    # fp32 sums of a few dozen terms
    assert float((got[33:73].double() - want[33:73]).norm()) < 1e-6 * float(want.norm())
