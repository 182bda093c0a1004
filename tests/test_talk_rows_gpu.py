"""Prompts of score-mixing attention: which segments the rows' kernel takes (ops.mixers.talk_product_rows), and that it and the
banded products agree with the plain form over long and several segments, behind a context and with a band."""
import pytest
import torch

from fasttalk_llm_microservice_amd.ops import mixers as M
from fasttalk_llm_microservice_amd.ops import mixers_ref as ref
from test_mixer_kernels_gpu import DEV, make_seg, rnd, to_dev

pytestmark = pytest.mark.gpu


def segments(lens, pos0):
    seg, blocks = make_seg(lens, pos0, list(range(len(lens))), block_size=16)
    dev = to_dev(seg)
    dev.host = seg.host = (seg.start.tolist(), pos0, seg.kv_len.tolist())
    return seg, dev, blocks


@pytest.mark.parametrize("lens,pos0,window,keep", [([300], [0], 0, 0), ([33, 31, 64], [5, 0, 700], 100, 9), ([130, 1], [500, 40], 0, 0),
                                                   ([257], [120], 64, 64)])
@pytest.mark.parametrize("heads,kv_heads,d", [(16, 4, 128), (8, 2, 64), (3, 1, 24)])
def test_long_segments(lens, pos0, window, keep, heads, kv_heads, d):
    g = torch.Generator().manual_seed(sum(lens) + d)
    seg, dev, blocks = segments(lens, pos0)
    t, bf = sum(lens), torch.bfloat16
    kc, vc = (rnd(blocks, 16, kv_heads * d, dt=bf, g=g) for _ in range(2))
    q = rnd(t, heads * d, g=g) * d ** -0.5
    talk = rnd(heads, heads, g=g) * heads ** -0.5
    spec = M.TalkSpec(heads, kv_heads, d, d, window, keep, 20.0, talk)
    want = ref.talk_attention(q, kc, vc, seg, heads, kv_heads, d, d, window, keep, 20.0, talk)
    spec = M.TalkSpec(heads, kv_heads, d, d, window, keep, 20.0, talk.to(DEV))
    args = (q.to(DEV), None, kc.to(DEV), vc.to(DEV), dev, spec)
    # fp32 products and sums of up to 764 keys behind a softmax: a few tens of 2^-23 of values of order one
    for f, extra in ((M.talk_attention, ()), (M.talk_attention_products, (1,))):
        got = f(torch.zeros(t, heads * d, device=DEV), *args, *extra)
        torch.testing.assert_close(got.cpu(), want.view(t, -1).float(), rtol=4e-5, atol=4e-5)


def test_which_segments():
    """Lines of the rule: pairs, bands, forms of the kernel; bf16 caches only."""
    def rows_from(lens, pos0, heads=16, kv_heads=4, d=128, window=0, keep=0, dt=torch.bfloat16, device=DEV):
        _, seg, _ = segments(lens, pos0)
        return M.talk_product_rows(seg, M.TalkSpec(heads, kv_heads, d, d, window, keep, 0.0, None),
                                   torch.empty(1, 16, kv_heads * d, dtype=dt, device=device), 32)

    none = 1 << 30
    assert rows_from([1024], [0]) == none and rows_from([300], [2000]) == none and rows_from([40] * 8, [0] * 8) == none
    assert rows_from([1300], [0]) == 1300 and rows_from([300], [3000]) == 300
    assert rows_from([700, 500, 900], [1500, 0, 1500]) == 700
    assert rows_from([31, 64], [40000, 10]) == none
    assert rows_from([4096], [0], window=1024, keep=64) == none and rows_from([4096], [0], window=2500) == 4096
    for other in (dict(heads=32, kv_heads=8), dict(kv_heads=16), dict(heads=12), dict(d=136), dict(d=12), dict(dt=torch.float32),
                  dict(device="cpu")):
        assert rows_from([64], [0], **other) == 32
