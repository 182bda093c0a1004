"""Windowed attention of decode rows on the matrix units (csrc/mixers/window_decode.hip) against the same
attention in 64 bits and against the general kernel: every mask and score term, at the edges of its tiles (32 keys
a wave, 256 a workgroup), short segments and long ones (left alone)."""
import pytest
import torch

from fasttalk_llm_microservice_amd.ops import mixers as M
from test_band_attention_gpu import DEV, reference, segments

pytestmark = pytest.mark.gpu


def cases():
    f = lambda *s: dict(zip(("heads", "kv_heads", "dk", "dv", "window"), s))   # noqa: E731
    yield "causal", f(4, 1, 128, 128, 0), {}, [1, 1, 1, 1], [0, 31, 32, 600]
    yield "causal, cap, sink 0", f(16, 1, 128, 128, 0), dict(softcap=30.0, sink=0.0), [1, 5, 33, 31], [255, 256, 0, 7]
    yield "window", f(3, 1, 64, 128, 100), {}, [1, 1], [50, 301]
    yield "window, kept, table", f(4, 2, 128, 128, 70), dict(keep_first=9, table=90), [1, 3], [511, 71]
    yield "window, kept beyond a tile", f(2, 2, 64, 64, 40), dict(keep_first=130), [1, 2], [64, 300]
    yield "blocks", f(4, 1, 128, 64, 96), dict(blocks=True), [1, 1, 2], [95, 96, 200]
    yield "two maps", f(4, 2, 64, 128, 128), dict(maps=2), [1, 9], [1000, 0]
    yield "sigmoid, distance", f(2, 1, 128, 128, 150), dict(sigmoid=True, terms=True), [1, 1], [31, 400]
    yield "sink per head, one key head each", f(2, 2, 128, 128, 33), dict(sinks=True), [1, 7], [640, 0]
    yield "sixteen heads, cap, sink per head", f(32, 2, 128, 128, 200), dict(softcap=8.0, sinks=True, keep_first=3), [1, 2], [450, 31]
    many = lambda n: [(37 * i) % 290 + (i == 5) for i in range(n)]   # noqa: E731
    yield "many groups (four waves)", f(16, 8, 128, 128, 0), dict(sinks=True, softcap=20.0), [1] * 33, many(33)
    yield "many groups (two waves)", f(8, 8, 64, 128, 0), dict(table=40), [1] * 60 + [3, 2], many(62)
    yield "seventeen heads a group (general kernel)", f(17, 1, 64, 64, 0), {}, [1], [300]


@pytest.mark.parametrize("name,sizes,opt,lens,pos0", list(cases()), ids=[c[0] for c in cases()])
@pytest.mark.parametrize("bs", [3, 16])
@pytest.mark.parametrize("tiles", [False, True], ids=["", "tiles"])
def test_against_64_bits(name, sizes, opt, lens, pos0, bs, tiles, monkeypatch):
    # attention without score terms goes to the tile kernel of the head-mixing attention, unless it is told not to
    if not tiles:
        monkeypatch.setattr(M, "_plain_tiles", lambda *a: False)
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
    if tiles and not M._plain_tiles(sp, kc):
        pytest.skip("the same kernels as without")
    fits = tiles or M.native_mixers().window_decode_fits(q, kc, vc, sp.heads, sp.maps, sp.kv_heads, sp.dk, sp.dv)
    assert tiles or fits == ("general kernel" not in name)
    want = reference(q, kc, vc, seg, sp, 1)
    out = torch.full((q.shape[0], hq, sp.dv), 7.0, device=DEV)
    got = M.window_attention(q, kc, vc, seg, sp, skip_from=32, out=out.clone())
    rows = torch.cat([torch.full((n,), n < 32) for n in lens]).to(DEV)
    assert bool((got[~rows] == 7.0).all())                     # long segments are not this call's
    old = M.window_attention(q, kc.float(), vc.float(), seg, sp)      # the general kernel, on widened caches
    norm = float(want[rows].norm())
    e_new, e_old = (float((x.double() - want)[rows].norm()) / norm for x in (got, old))
    # fp32 sums of a few hundred terms: about 2^-22; no further from 64 bits than the general kernel
    assert e_new < 1e-6 and e_new < 1.5 * e_old + 1e-7, (e_new, e_old)
    # rows in bf16 are the fp32 ones, rounded once
    assert (M.window_out_dtype(q, kc, vc, sp, torch.bfloat16, False) == torch.bfloat16) == fits
    if fits:
        got16 = M.window_attention(q, kc, vc, seg, sp, skip_from=32, out=out.bfloat16())
        assert torch.equal(got16[rows], got[rows].bfloat16())
