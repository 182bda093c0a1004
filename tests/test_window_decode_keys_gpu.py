"""Windowed attention of decode rows (csrc/mixers/window_decode.hip) where a step of 32 keys is not whole: keys that there are
not read slot 0, whatever lies there, and count for nothing."""
import pytest
import torch

from fasttalk_llm_microservice_amd.ops import mixers as M
from test_band_attention_gpu import DEV, reference, segments

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bs", [3, 16])
@pytest.mark.parametrize("dk,dv", [(128, 128), (64, 128), (128, 64), (64, 64)])
@pytest.mark.parametrize("sigmoid", [False, True])
def test_keys_that_there_are_not(bs, dk, dv, sigmoid, monkeypatch):
    monkeypatch.setattr(M, "_plain_tiles", lambda *a: False)
    g = torch.Generator().manual_seed(dk + dv + bs)
    lens, pos0 = [1, 1, 1, 2, 1], [0, 30, 31, 255, 287]
    sp = M.WindowSpec(scale=dk ** -0.5, heads=4, kv_heads=2, dk=dk, dv=dv, window=0, sigmoid=sigmoid)
    seg, blocks = segments(lens, pos0, bs, g)
    # a block 0 that no row's table names, full of NaN
    kc = torch.randn(blocks + 1, bs, 2 * dk, generator=g).to(DEV, torch.bfloat16)
    vc = torch.randn(blocks + 1, bs, 2 * dv, generator=g).to(DEV, torch.bfloat16)
    q = torch.randn(sum(lens), 4 * dk, generator=g).to(DEV)
    assert M.native_mixers().window_decode_fits(q, kc, vc, 4, 1, 2, dk, dv)
    want = reference(q, kc[1:], vc[1:], seg, sp, 1)
    kc[0], vc[0] = float("nan"), float("nan")
    seg.block_tables.add_(1)
    got = M.window_attention(q, kc, vc, seg, sp)
    # fp32 sums of up to 288 terms
    assert float((got.double() - want).norm() / want.norm()) < 1e-6
    # a table's entry outside the cache: the row as without its keys
    if not sigmoid and bs == 16:
        full = M.window_attention(q, kc, vc, seg, sp)
        for entry in (-1, blocks + 1):
            seg.block_tables[4, 17] = entry                       # the last row's last block: its only key there is key 272 ..
            cut = M.window_attention(q, kc, vc, seg, sp)
            assert torch.equal(cut[:5], full[:5]) and bool(torch.isfinite(cut).all())
            seg.kv_len[4] = 272
            short = M.window_attention(q, kc, vc, seg, sp)
            seg.kv_len[4] = 288
            torch.testing.assert_close(cut[5], short[5], rtol=1e-6, atol=1e-6)
