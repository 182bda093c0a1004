"""Products whose last round of 256 x 256 tiles is done in halves (csrc/mixers/tile_gemm.hip): no whole round, one and two, one tile
left and half a round, halves that lie past the last row, ends inside a tile; bit for bit the whole tiles' results, and near
64 bits."""
import pytest
import torch

from fasttalk_llm_microservice_amd.ops import mixers as M
from test_tile_gemm_gpu import DEV, act64, close, rnd

pytestmark = pytest.mark.gpu
WHOLE, TAIL = 0, 9


@pytest.mark.parametrize("rows,n,k", [(1, 8, 64), (130, 600, 64), (256, 128 * 256, 192), (300, 128 * 256 + 5, 128), (385, 129 * 256, 64),
                                      (4000, 4600, 128), (4096, 24 * 256 - 12, 192), (2049, 57 * 256, 64), (1024, 257 * 64, 448)])
@pytest.mark.parametrize("act", [None, "silu", "relu_sq"])
def test_halves_of_the_last_round(rows, n, k, act):
    glu = act == "silu"
    n //= 2 if glu else 1
    x, w = rnd(rows, rows, k), rnd(n, 2 * n if glu else n, k, scale=k ** -0.5)
    b = rnd(n + 1, n) if act is None else None
    out = []
    for form in (WHOLE, TAIL):
        wide = torch.full((rows + 1, n + 8), 7.0, dtype=x.dtype, device=DEV)
        M.native_mixers().tile_gemm(wide[:rows, :n], x, w, b, M.FEW_ACTS[act], 1.5, form)
        assert bool((wide[rows] == 7.0).all()) and bool((wide[:, n:] == 7.0).all())
        out.append(wide[:rows, :n])
    assert torch.equal(out[0], out[1])
    rows = slice(max(0, rows - 200), rows)
    want = x[rows].double() @ w.double().t()
    close(out[1][rows], act64(want, act, 1.5) if act is not None else want + b.double(), k, slope=32.0 if act else 1.0)


def test_rule():
    """What is taken beyond the expected times' rule is in the form that was measured for it, whatever the sizes."""
    taken = 0
    for rows in range(1030, 4600, 170):
        for n in range(4000, 20000, 508):
            for k in (1536, 1792, 2048, 3072, 4096):
                us, tail = M.native_mixers().tile_gemm_us(rows, n, k, False)
                if M._tile_gemm_pays(rows, n, k) and us > 7 + 2.0 * rows * n * k / 1.35e9:
                    assert tail and n % 8 == 0, (rows, n, k)
                    taken += 1
    assert taken > 0 and M._tile_gemm_pays(2048, 10272, 2048) and M._tile_gemm_pays(4096, 6144, 2048)
