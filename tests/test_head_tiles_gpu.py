"""Products with a matrix per head of bf16 values (csrc/mixers/head_tiles.hip) against 64 bits: the two splits of the work, rows
and columns that end inside a tile, one step along K and many, the heads of one rotation's workgroup."""
import pytest
import torch

from fasttalk_llm_microservice_amd.ops import mixers as M
from fasttalk_llm_microservice_amd.ops import mixers_ref as R
from test_mixer_kernels_gpu import DEV, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,heads,dn,rank,dr,dv,dt", [
    (1, 1, 32, 32, 4, 32, torch.float32), (5, 16, 128, 512, 64, 128, torch.bfloat16), (33, 5, 64, 96, 8, 160, torch.bfloat16),
    (300, 16, 128, 512, 64, 128, torch.bfloat16), (129, 3, 32, 1024, 0, 96, torch.float32),
    (1030, 16, 128, 512, 64, 128, torch.bfloat16), (257, 33, 160, 288, 72, 64, torch.float32),
    (500, 70, 96, 160, 16, 224, torch.bfloat16)])
@pytest.mark.parametrize("interleaved,gated", [(False, True), (True, False)])
def test_rows_per_head(rows, heads, dn, rank, dr, dv, dt, interleaved, gated):
    g = torch.Generator().manual_seed(rows * rank)
    q = rnd(rows, heads * (dn + dr) + 8, dt=dt, g=g)[:, :heads * (dn + dr)]
    wuk = rnd(heads, dn, rank, g=g, scale=dn ** -0.5).bfloat16().float()
    wuv = rnd(heads, rank, dv, g=g, scale=rank ** -0.5).bfloat16().float()
    gate = rnd(rows, heads + 3, dt=dt, g=g)[:, :heads] if gated else None
    dims = dr // 4 * 2
    table, pos = M.rope_table(50, dims, 1e4, device="cpu"), torch.randint(0, 50, (rows,), generator=g, dtype=torch.int32)
    qn, qr64 = R.latent_q_rope(q, table, dims, pos, heads, dn, dr, interleaved)
    qa64 = torch.bmm(qn.double().transpose(0, 1), wuk.double())
    tk, tv = M.head_tiles(wuk.to(DEV)), M.head_tiles(wuv.to(DEV))
    assert tk is not None and tv is not None
    qa, qr = M.latent_q_absorb(q.to(DEV), wuk.to(DEV), table.to(DEV), dims, pos.to(DEV), heads, dn, dr, interleaved, tk)
    # fp32 sums of up to 1024 terms of about 1 / sqrt(terms), of three parts each
    torch.testing.assert_close(qa.cpu().double(), qa64, rtol=1e-5, atol=4e-6)
    torch.testing.assert_close(qr.cpu(), qr64.float(), rtol=1e-5, atol=1e-5)
    got = M.head_values(qa, wuv.to(DEV), gate.to(DEV) if gated else None, dt, tv).cpu().double()
    want = torch.bmm(qa.cpu().double(), wuv.double())
    if gated:
        want = want * torch.sigmoid(gate.double()).t()[:, :, None]
    want = want.transpose(0, 1).reshape(rows, heads * dv)
    torch.testing.assert_close(got, want, rtol=2 ** -8 if dt == torch.bfloat16 else 1e-5, atol=1e-5)


def test_matrices_that_bf16_does_not_hold():
    w = torch.ones(2, 32, 64, device=DEV)
    assert M.head_tiles(w) is not None
    for v in (1.001, float("inf"), float("nan")):
        u = w.clone()
        u[1, 31, 63] = v
        assert M.head_tiles(u) is None
    assert M.head_tiles(w[:, :16].contiguous()) is None and M.head_tiles(w[:, :, :48].contiguous()) is None
