"""Latent attention of few rows on the matrix units (csrc/mixers/latent_decode.hip) against 64 bits."""
import pytest
import torch

from fasttalk_llm_microservice_amd.ops import mixers as M
from test_mixer_kernels_gpu import DEV, make_seg, to_dev

pytestmark = pytest.mark.gpu
RANK, DR = 512, 64


@pytest.mark.parametrize("sink", [False, True])
@pytest.mark.parametrize("known", [False, True])      # the longest context (slices of at least 64 keys)
@pytest.mark.parametrize("lens,pos0,heads,page", [
    ([1], [0], 16, 16),                               # one key, all other slices empty
    ([1, 1, 1], [62, 63, 64], 16, 16),                # around a tile of 64 keys
    ([1, 3, 1, 31], [2500, 0, 130, 40], 3, 4),        # several tiles a slice; part of a head tile; short segments
    ([1] * 64, list(range(0, 640, 10)), 20, 8),       # two head tiles, eight slices
])
def test_latent_decode(lens, pos0, heads, page, known, sink):
    g = torch.Generator(device=DEV).manual_seed(sum(lens) + heads)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)      # noqa: E731
    seg, _ = make_seg(lens, pos0, list(range(len(lens))), block_size=page)
    seg = to_dev(seg)
    seg.max_kv = max(p + n for p, n in zip(pos0, lens)) if known else 0
    t = sum(lens)
    cache = rnd(int(seg.block_tables.max()) + 1, page, RANK + DR).bfloat16()
    qa, qr, scale = rnd(heads, t, RANK), rnd(t, heads, DR), 0.07
    sinks = rnd(heads) * 3 if sink else None
    got = M.latent_attention(qa, qr, cache, seg, scale, RANK, sink=sinks)
    a = 0
    for s, n in enumerate(lens):
        b, kv = a + n, pos0[s] + n
        k = cache[seg.block_tables[s, :(kv + page - 1) // page].long()].reshape(-1, RANK + DR)[:kv].double()
        sc = (qa[:, a:b].double() @ k[:, :RANK].t() + (qr[a:b].double() @ k[:, RANK:].t()).transpose(0, 1)) * scale
        see = torch.arange(kv, device=DEV)[None] <= (pos0[s] + torch.arange(n, device=DEV))[:, None]
        sc = sc.masked_fill(~see, float("-inf"))
        if sinks is not None:
            sc = torch.cat([sc, sinks.double()[:, None, None].expand(heads, n, 1)], -1)
        p = sc.softmax(-1)[..., :kv]
        # fp32 scores of 576 terms (a rounding of each partial sum, of order 2 sqrt(576) times the scale: 2^-19) and
        # sums of kv terms: relative to sum_j p_j |c_j|
        bound = 2 ** -16 * (p @ k[:, :RANK].abs()) + 1e-7
        assert bool(((got[:, a:b].double() - p @ k[:, :RANK]).abs() <= bound).all())
        a = b


@pytest.mark.parametrize("sink", [False, True])
@pytest.mark.parametrize("known", [False, True])
@pytest.mark.parametrize("first,last", [(64, 128), (128, 130), (0, 70)])     # a slice of 64, the last slice's two, a first one
def test_scores_that_overflow(first, last, known, sink):
    """Scores of -inf (products of 1e20 and -1e20) throughout a slice of the keys: weight 0, as exp(-inf)."""
    kv, heads, page = 130, 16, 16
    g = torch.Generator(device=DEV).manual_seed(7)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)      # noqa: E731
    seg, _ = make_seg([1], [kv - 1], [0], block_size=page)
    seg = to_dev(seg)
    seg.max_kv = kv if known else 0
    blocks = seg.block_tables[0, :(kv + page - 1) // page].long()
    keys = rnd(blocks.numel() * page, RANK + DR)
    keys[:, -1] = 0
    keys[first:last, -1] = -1e20
    cache = torch.zeros(int(blocks.max()) + 1, page, RANK + DR, device=DEV)
    cache[blocks] = keys.view(-1, page, RANK + DR)
    cache = cache.bfloat16()
    qa, qr, scale = rnd(heads, 1, RANK), rnd(1, heads, DR), 0.07
    qr[..., -1] = 1e20
    sinks = rnd(heads) if sink else None
    got = M.latent_attention(qa, qr, cache, seg, scale, RANK, sink=sinks)[:, 0].double()
    k = keys.bfloat16().double()[:kv]
    sc = (qa[:, 0].double() @ k[:, :RANK].t() + qr[0].double() @ k[:, RANK:].t()) * scale
    if sink:
        sc = torch.cat([sc, sinks.double()[:, None]], -1)
    p = sc.softmax(-1)[:, :kv]
    # as above
    assert bool(((got - p @ k[:, :RANK]).abs() <= 2 ** -16 * (p @ k[:, :RANK].abs()) + 1e-7).all())
