"""Latent attention of long segments in one kernel (csrc/mixers/latent_prefill.hip) against 64 bits."""
import pytest
import torch

from fasttalk_llm_microservice_amd.ops import mixers as M
from test_mixer_kernels_gpu import DEV, make_seg, to_dev

pytestmark = pytest.mark.gpu
RANK, DR = 512, 64


def reference(qa, qr, cache, seg, lens, pos0, scale, sink):
    """fp64 on the kernel's operands (queries rounded to bf16); also sum_j p_j |c_j|."""
    heads, t, _ = qa.shape
    qa, qr = qa.bfloat16().double(), qr.bfloat16().double()
    out, size, a = torch.zeros(heads, t, RANK, dtype=torch.float64, device=DEV), None, 0
    size = torch.zeros_like(out)
    for s, n in enumerate(lens):
        b, kv = a + n, pos0[s] + n
        bs = cache.shape[1]
        k = cache[seg.block_tables[s, :(kv + bs - 1) // bs].long()].reshape(-1, RANK + DR)[:kv].double()
        sc = (qa[:, a:b] @ k[:, :RANK].t() + (qr[a:b] @ k[:, RANK:].t()).transpose(0, 1)) * scale
        see = torch.arange(kv, device=DEV)[None] <= (pos0[s] + torch.arange(n, device=DEV))[:, None]
        sc = sc.masked_fill(~see, float("-inf"))
        top = sc.max(-1, keepdim=True).values
        if sink is not None:
            top = torch.maximum(top, sink.double()[:, None, None])
        p = (sc - top).exp()
        den = p.sum(-1, keepdim=True)
        if sink is not None:
            den = den + (sink.double()[:, None, None] - top).exp()
        out[:, a:b] = p / den @ k[:, :RANK]
        size[:, a:b] = p / den @ k[:, :RANK].abs()
        a = b
    return out, size


@pytest.mark.parametrize("sink", [False, True])
@pytest.mark.parametrize("lens,pos0,heads,page", [
    ([32], [0], 1, 8),                              # one tile of keys, a quarter of a workgroup's pairs
    ([128, 40, 3, 64], [31, 0, 5, 2], 1, 16),       # whole workgroups; a short segment, left alone
    ([33, 100, 65], [7, 0, 130], 3, 8),             # heads that do not divide 128
    ([43], [1], 16, 64),
    ([70], [900], 5, 8),                           # more than 64 pages
])
@pytest.mark.parametrize("rise", [0.0, 0.05])       # scores that grow with the key: the reference moves often
def test_latent_prefill(lens, pos0, heads, page, sink, rise):
    g = torch.Generator(device=DEV).manual_seed(sum(lens) + heads)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)      # noqa: E731
    seg, _ = make_seg(lens, pos0, list(range(len(lens))), block_size=page)
    seg = to_dev(seg)
    seg.host = (seg.start.tolist(), seg.pos0.tolist(), seg.kv_len.tolist())
    t = sum(lens)
    cache = rnd(int(seg.block_tables.max()) + 1, page, RANK + DR)
    qa, qr, scale = rnd(heads, t, RANK), rnd(t, heads, DR), 0.07
    if rise:
        for s in range(len(lens)):
            kv = pos0[s] + lens[s]
            rows = cache[seg.block_tables[s, :(kv + page - 1) // page].long()]
            rows.view(-1, RANK + DR)[:, -1] = rise * torch.arange(rows.shape[0] * page, device=DEV)
            cache[seg.block_tables[s, :rows.shape[0]].long()] = rows
        qr[:, :, -1] = 20.0
    cache = cache.bfloat16()
    sinks = rnd(heads) * 3 if sink else None
    assert M.latent_prefill_ok(qa, cache, RANK, torch.bfloat16) and M._latent_prefill_pays(seg, heads, 32)
    out = torch.full((heads, t, RANK), 7.0, device=DEV)
    M.latent_attention_products(out, qa, qr, cache, seg, scale, RANK, 32, torch.bfloat16, sinks)
    want, size = reference(qa, qr, cache, seg, lens, pos0, scale, sinks)
    a = 0
    for n in lens:
        got, w, z = out[:, a:a + n].double(), want[:, a:a + n], size[:, a:a + n]
        if n < 32:
            assert bool((got == 7.0).all())
        else:
            # weights rounded to bf16 (half a unit: 2^-8); scores of up to 2^8 and their sums in fp32 (2^-12)
            assert bool(((got - w).abs() <= (2 ** -8 + 2 ** -12) * z + 1e-6).all())
        a += n


@pytest.mark.parametrize("form", ["queries across", "queries off", "rotated across", "cache off", "pages apart", "out across",
                                  "wide tables", "bf16 queries"])
def test_operands_of_other_layouts(form):
    """Operands that are not dense, aligned or fp32: the two products take them."""
    g = torch.Generator(device=DEV).manual_seed(5)
    heads, lens, pos0 = 2, [70, 5, 33], [3, 0, 20]
    t = sum(lens)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)      # noqa: E731
    off = lambda x: torch.empty(x.numel() + 1, dtype=x.dtype, device=DEV)[1:].copy_(x.flatten()).view(x.shape)   # noqa: E731
    seg, blocks = make_seg(lens, pos0, [0, 1, 2], block_size=8)
    seg = to_dev(seg)
    seg.host = (seg.start.tolist(), seg.pos0.tolist(), seg.kv_len.tolist())
    cache = rnd(blocks, 8, RANK + DR).bfloat16()
    qa, qr = rnd(heads, t, RANK).bfloat16().float(), rnd(t, heads, DR).bfloat16().float()
    out = torch.zeros(heads, t, RANK, device=DEV)
    want, size = reference(qa, qr, cache, seg, lens, pos0, 0.05, None)
    if form == "queries across":
        qa = qa.transpose(0, 1).contiguous().transpose(0, 1)
    elif form == "queries off":
        qa = off(qa)
    elif form == "rotated across":
        qr = torch.cat([qr, qr], 2)[..., DR:]
    elif form == "cache off":
        cache = off(cache)
    elif form == "pages apart":
        cache = torch.cat([cache, cache], 1)[:, 8:]
    elif form == "out across":
        out = out.transpose(0, 1).contiguous().transpose(0, 1)
    elif form == "wide tables":
        seg.block_tables = seg.block_tables.long()
    else:
        qa, qr = qa.bfloat16(), qr.bfloat16()
    M.latent_attention_products(out, qa, qr, cache, seg, 0.05, RANK, 32, torch.bfloat16)
    rows = torch.cat([torch.full((n,), n >= 32) for n in lens]).to(DEV)
    # weights rounded to bf16 twice at most: 2^-8 (a sum and its quotient)
    assert bool(((out.double() - want)[:, rows].abs() <= (2 ** -8 + 2 ** -12) * size[:, rows] + 1e-6).all())
    assert bool((out[:, ~rows] == 0).all())


@pytest.mark.parametrize("sink", [False, True])
def test_scores_that_overflow(sink):
    """Scores of -inf (products of 1e20 and -1e20) in the first tiles of keys: weight 0, as exp(-inf)."""
    lens, pos0, t = [130], [0], 130
    seg, blocks = make_seg(lens, pos0, [0], block_size=8)
    seg = to_dev(seg)
    seg.host = (seg.start.tolist(), seg.pos0.tolist(), seg.kv_len.tolist())
    g = torch.Generator(device=DEV).manual_seed(6)
    keys = torch.randn(blocks * 8, RANK + DR, generator=g, device=DEV)
    keys[:70, -1] = -1e20
    keys[70:, -1] = 0
    cache = torch.empty_like(keys)
    cache.view(blocks, 8, -1)[seg.block_tables[0].long()] = keys.view(blocks, 8, -1)
    cache = cache.view(blocks, 8, -1).bfloat16()
    qa, qr = torch.randn(1, t, RANK, generator=g, device=DEV), torch.randn(t, 1, DR, generator=g, device=DEV)
    qr[:, :, -1] = 1e20
    sinks = torch.ones(1, device=DEV) if sink else None
    out = torch.full((1, t, RANK), 7.0, device=DEV)
    M.latent_attention_products(out, qa, qr, cache, seg, 0.05, RANK, 32, torch.bfloat16, sinks)
    qr[:, :, -1], keys[:70, -1] = 0, 0
    see = torch.arange(130, device=DEV)
    q = torch.cat([qa[0], qr[:, 0]], 1).bfloat16().double()
    k = keys[:130].bfloat16().double()
    sc = (q @ k.T * 0.05).masked_fill((see[None] > see[:, None]) | (see < 70)[None], float("-inf"))[70:]
    if sink:
        sc = torch.cat([sc, torch.ones(60, 1, dtype=sc.dtype, device=DEV)], 1)
    p = torch.softmax(sc, 1)[:, :130]
    want, size = p @ k[:, :RANK], p @ k[:, :RANK].abs()
    # weights rounded to bf16 (half a unit: 2^-8), the rest fp32; rows that see no other score are undefined
    assert bool(((out[0, 70:].double() - want).abs() <= (2 ** -8 + 2 ** -12) * size + 1e-6).all())
