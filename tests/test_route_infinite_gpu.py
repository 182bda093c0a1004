"""Routers of rows with infinite logits, or with a selection bias that is no finite number: the experts that are named are those
of the router's kernels on ready logits, one expert after the other (csrc/mixers/moe_route.hip choose_in_turn)."""
import pytest
import torch

from fasttalk_llm_microservice_amd.ops import mixers as M
from test_mixer_kernels_gpu import DEV, rnd

pytestmark = pytest.mark.gpu
INF = float("inf")


def same(got, want):
    assert torch.equal(got[0], want[0])
    torch.testing.assert_close(got[1], want[1], rtol=1e-4, atol=1e-6, equal_nan=True)


@pytest.mark.parametrize("mode", ["softmax of all", "softmax", "sigmoid"])
@pytest.mark.parametrize("bad", [[(3, INF)], [(3, -INF)], [(e, -INF) for e in range(10)], [(2, INF), (7, INF), (9, -INF)]],
                         ids=["inf", "-inf", "few left", "several"])
@pytest.mark.parametrize("groups,keep", [(1, 1), (4, 2)])
@pytest.mark.parametrize("rows", [2, 64])
def test_infinite_logits(mode, bad, groups, keep, rows):
    experts, top, width = 12, 4, 512
    g = torch.Generator().manual_seed(rows)
    h, router, corr = rnd(rows, width, dt=torch.bfloat16, g=g), rnd(experts, width, g=g, scale=width ** -0.5), rnd(experts, g=g)
    # column 0 is the bad logits' own: 2^100 of the row times 2^100 of the expert, in row 1
    h[:, 0], router[:, 0] = 0.0, 0.0
    h[1, 0] = 2.0 ** 100
    for e, v in bad:
        router[e, 0] = 2.0 ** 100 * (1.0 if v > 0 else -1.0)
    h, router, corr = h.to(DEV), router.to(DEV), corr.to(DEV)
    z = h.float() @ router.t()
    assert all(float(z[1, e]) == v for e, v in bad) and bool(z[0].isfinite().all())
    if mode == "softmax of all":
        same(M.moe_route_softmax(h, router, corr, top, groups, keep), M.moe_topk(z, corr, top, groups, keep))
    elif mode == "sigmoid":
        same(M.moe_route_top_logits(h, router, None, top, True, 1.5, groups, keep), M.moe_top_sigmoid(z, top, 1.5, groups, keep))
    else:
        same(M.moe_route_top_logits(h, router, None, top), M.moe_top_logits(z, top))


@pytest.mark.parametrize("v", [INF, -INF, float("nan")])
def test_selection_bias(v):
    g = torch.Generator().manual_seed(7)
    h, router, corr = rnd(3, 512, dt=torch.bfloat16, g=g).to(DEV), rnd(12, 512, g=g).to(DEV), rnd(12, g=g).to(DEV)
    corr[[1, 4, 5, 6, 7, 8, 9, 10, 11]] = v
    same(M.moe_route_softmax(h, router, corr, 4, 1, 1), M.moe_topk(h.float() @ router.t(), corr, 4, 1, 1))


def test_rows_of_a_prompt():
    """Above 64 rows the experts of such a row are distinct, as the router for sixteen rows a workgroup names them."""
    g = torch.Generator().manual_seed(9)
    h, router, corr = rnd(100, 2048, dt=torch.bfloat16, g=g).to(DEV), rnd(12, 2048, g=g).to(DEV), rnd(12, g=g).to(DEV)
    h[1, 5], h[2, 0] = float("nan"), 2.0 ** 100
    router[3, 0] = 2.0 ** 100
    parts = M.route_parts(router)
    assert M.moe_route_fits(h, parts, 12)
    same(M.moe_route_softmax(h, router, corr, 4, 1, 1), M.moe_route(h, parts, corr, 12, 4, "grouped_softmax", 1.0, 1, 1))
    same(M.moe_route_top_logits(h, router, corr, 4), M.moe_route(h, parts, corr, 12, 4, "top_logits", 1.0, 1, 1))
