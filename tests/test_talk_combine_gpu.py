"""The merge of a row's key slices (csrc/mixers/talk_attn.hip talk_combine_kernel): its gate at any column of wider rows, rows of
no context, and value heads of more and fewer than 256 columns."""
import pytest
import torch

from fasttalk_llm_microservice_amd.ops import mixers as M
from fasttalk_llm_microservice_amd.ops import mixers_ref as R
from test_band_attention_gpu import DEV, segments

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("dv", [32, 128, 320, 12])
@pytest.mark.parametrize("left", [0, 3, 4])
def test_gate(dt, dv, left):
    g = torch.Generator().manual_seed(dv + left)
    lens, pos0 = [1, 1, 2], [0, 700, 63]
    seg, blocks = segments(lens, pos0, 16, g)
    kc, vc = (torch.randn(blocks, 16, 2 * d, generator=g).to(DEV, dt) for d in (32, dv))
    spec = M.TalkSpec(4, 2, 32, dv, 0, 0, 0.0, torch.eye(4, device=DEV))
    rows = 6                                                     # (two of them padding)
    q = torch.randn(rows, 4 * 32, generator=g).to(DEV)
    gate = torch.randn(rows, 4 * dv + left + 5, generator=g).to(DEV, dt)[:, left:left + 4 * dv]
    plain = M.talk_attention(torch.zeros(rows, 4 * dv, device=DEV, dtype=dt), q, None, kc, vc, seg, spec)
    got = M.talk_attention(torch.zeros(rows, 4 * dv, device=DEV, dtype=dt), q, gate, kc, vc, seg, spec)
    cpu = M.Segments(*(t.cpu() for t in (seg.start, seg.pos0, seg.slot, seg.kv_len, seg.block_tables)), seg.num, seg.max_rows, seg.max_kv,
                     seg.host)
    want = R.talk_attention(q.cpu(), kc.cpu(), vc.cpu(), cpu, 4, 2, 32, dv, 0, 0, 0.0, torch.eye(4)).view(rows, -1)
    close = dict(rtol=2e-2, atol=2e-2) if dt == torch.bfloat16 else dict(rtol=1e-4, atol=1e-4)
    torch.testing.assert_close(plain.cpu()[:4].float(), want[:4].float(), **close)
    torch.testing.assert_close(got.cpu()[:4].float(), (want * torch.sigmoid(gate.cpu().float()))[:4], **close)
    assert bool((plain[4:] == 0).all()) and bool((got[4:] == 0).all())         # padding rows are not written
