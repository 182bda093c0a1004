"""What rides in a product of few rows (csrc/mixers/few_rows.hip FewRowsRider): a second product of the same sizes, and the
token-side gate; up to 16, 32 and 64 rows and with ragged columns, against the launches they stand for."""
import pytest
import torch

from fasttalk_llm_microservice_amd.ops import mixers as M
from test_mixer_kernels_gpu import DEV, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,n,k", [(1, 2048, 128), (16, 40, 64), (17, 2048, 256), (33, 520, 2048), (64, 4608, 128), (65, 256, 128)])
def test_two_products(rows, n, k):
    g = torch.Generator().manual_seed(rows)
    p = rnd(rows, 2 * k + 16, dt=torch.bfloat16, g=g).to(DEV)
    w, w2 = (rnd(n, k, dt=torch.bfloat16, g=g, scale=k ** -0.5).to(DEV) for _ in range(2))
    y, y2 = M.linear_pair(p[:, :k], w, p[:, k:2 * k], w2)
    for got, x, m in ((y, p[:, :k], w), (y2, p[:, k:2 * k], w2)):
        want = M.linear(x, m)
        if rows <= 64 and M._few_rows_pays(rows, n, k):
            assert torch.equal(got, want)
        torch.testing.assert_close(got.double(), x.double() @ m.double().t(), rtol=2 ** -8, atol=1e-5)


@pytest.mark.parametrize("rows,sd,k", [(1, 64, 2048), (9, 36, 512), (32, 64, 2048), (64, 264, 256), (70, 64, 256)])
def test_side_gate(rows, sd, k):
    g = torch.Generator().manual_seed(sd)
    x, w = rnd(rows, k, dt=torch.bfloat16, g=g), rnd(sd, k, dt=torch.bfloat16, g=g, scale=2 * k ** -0.5)
    table, ids = rnd(50, 3 * sd, dt=torch.bfloat16, g=g), torch.randint(0, 50, (rows,), generator=g, dtype=torch.int32)
    ids[0] = 77                                                  # outside the table: its first row
    got = M.linear_side_gate(x.to(DEV), w.to(DEV), table.to(DEV), ids.to(DEV), sd, sd).cpu().double()
    z = x.double() @ w.double().t()
    t64 = table.double()[torch.where(ids < 50, ids, 0).long(), sd:2 * sd]
    want = torch.nn.functional.gelu(z, approximate="tanh") * t64
    # one rounding to bf16 at the end, and where the product is a launch of its own one before the gate
    torch.testing.assert_close(got, want, rtol=2 ** -6, atol=2 ** -9)
    assert float((got - want).norm() / want.norm()) < 2 ** -8
