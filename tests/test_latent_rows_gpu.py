"""Latent attention of prompts of few rows: which steps the rows' kernel takes (ops.mixers.latent_rows_pay), and its results over
segments of many rows against the plain form."""
import pytest
import torch

from fasttalk_llm_microservice_amd.ops import mixers as M
from fasttalk_llm_microservice_amd.ops import mixers_ref as ref
from test_mixer_kernels_gpu import DEV, make_seg, rnd, to_dev

pytestmark = pytest.mark.gpu
RANK, DR = 512, 64


def segments(lens, pos0):
    seg, blocks = make_seg(lens, pos0, list(range(len(lens))), block_size=16)
    dev = to_dev(seg)
    dev.host = seg.host = (seg.start.tolist(), pos0, seg.kv_len.tolist())
    return seg, dev, blocks


@pytest.mark.parametrize("heads", [16, 5])
@pytest.mark.parametrize("lens,pos0", [([300], [0]), ([33, 1, 64], [5, 40, 0]), ([128], [200])])
def test_many_rows(lens, pos0, heads):
    g = torch.Generator().manual_seed(sum(lens) + heads)
    seg, dev, blocks = segments(lens, pos0)
    t = sum(lens)
    cache = rnd(blocks, 16, RANK + DR, dt=torch.bfloat16, g=g)
    qa, qr = rnd(heads, t, RANK, g=g), rnd(t, heads, DR, g=g)
    want = ref.latent_attention(qa, qr, cache, seg, 0.02, RANK, None)
    got = M.latent_attention(qa.to(DEV), qr.to(DEV), cache.to(DEV), dev, 0.02, RANK)
    # fp32 scores of 576 products of order one, then a softmax: a few tens of 2^-23 times the scores' size
    torch.testing.assert_close(got.cpu(), want, rtol=1e-4, atol=1e-4)


def test_which_steps():
    def rows_kernel(lens, pos0, heads=16, rank=RANK, dt=torch.bfloat16):
        _, seg, _ = segments(lens, pos0)
        qa = torch.empty(heads, 1, rank, device=DEV)
        return M.latent_rows_pay(qa, torch.empty(1, 16, rank + DR, dtype=dt, device=DEV), seg, rank, dt, 32)

    assert rows_kernel([32], [0]) and rows_kernel([300], [0]) and rows_kernel([20, 60], [0, 0]) and rows_kernel([64], [600])
    assert not (rows_kernel([600], [0]) or rows_kernel([200] * 4, [0] * 4) or rows_kernel([64], [4000]) or rows_kernel([4096], [0]))
    assert not (rows_kernel([32], [0], heads=32) or rows_kernel([32], [0], rank=256) or rows_kernel([32], [0], dt=torch.float32))
