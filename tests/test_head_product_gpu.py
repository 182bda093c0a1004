"""Products of few rows with a matrix per head (csrc/mixers/head_product.hip) against 64 bits: parts of eight rows, of the
columns of a workgroup, of the rows of a matrix that its threads hold at a time."""
import pytest
import torch

from fasttalk_llm_microservice_amd.ops import mixers as M
from fasttalk_llm_microservice_amd.ops import mixers_ref as R
from test_mixer_kernels_gpu import DEV, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,heads,dn,rank,dr,dv,dt", [
    (1, 1, 8, 4, 4, 4, torch.float32), (3, 16, 128, 512, 64, 128, torch.bfloat16), (8, 5, 40, 100, 8, 36, torch.bfloat16),
    (9, 3, 1024, 132, 0, 20, torch.float32), (16, 2, 136, 1024, 16, 260, torch.bfloat16), (17, 2, 16, 32, 16, 16, torch.bfloat16),
    (7, 128, 64, 64, 32, 64, torch.bfloat16)])
@pytest.mark.parametrize("interleaved,gated", [(False, True), (True, False)])
def test_few_rows_per_head(rows, heads, dn, rank, dr, dv, dt, interleaved, gated):
    g = torch.Generator().manual_seed(rows * rank)
    q = rnd(rows, heads * (dn + dr) + 8, dt=dt, g=g)[:, :heads * (dn + dr)]
    wuk, wuv = rnd(heads, dn, rank, g=g, scale=dn ** -0.5), rnd(heads, rank, dv, g=g, scale=rank ** -0.5)
    gate = rnd(rows, heads + 3, dt=dt, g=g)[:, :heads] if gated else None
    dims = dr // 4 * 2
    table, pos = M.rope_table(50, dims, 1e4, device="cpu"), torch.randint(0, 50, (rows,), generator=g, dtype=torch.int32)
    qn, qr64 = R.latent_q_rope(q, table, dims, pos, heads, dn, dr, interleaved)
    qa64 = torch.bmm(qn.double().transpose(0, 1), wuk.double())
    qa, qr = M.latent_q_absorb(q.to(DEV), wuk.to(DEV), table.to(DEV), dims, pos.to(DEV), heads, dn, dr, interleaved)
    # fp32 sums of up to 1024 terms of about 1 / sqrt(terms)
    torch.testing.assert_close(qa.cpu().double(), qa64, rtol=1e-5, atol=4e-6)
    torch.testing.assert_close(qr.cpu(), qr64.float(), rtol=1e-5, atol=1e-5)
    got = M.head_values(qa, wuv.to(DEV), gate.to(DEV) if gated else None, dt).cpu().double()
    want = torch.bmm(qa.cpu().double(), wuv.double())
    if gated:
        want = want * torch.sigmoid(gate.double()).t()[:, :, None]
    want = want.transpose(0, 1).reshape(rows, heads * dv)
    torch.testing.assert_close(got, want, rtol=2 ** -8 if dt == torch.bfloat16 else 1e-5, atol=1e-5)
