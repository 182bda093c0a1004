"""Routers with their logits in one launch (csrc/mixers/moe_route.hip moe_route_tile_kernel) against the routers on
64-bit logits: part-filled tiles of 16 rows and 16 experts, groups, ties."""
import pytest
import torch

from fasttalk_llm_microservice_amd.ops import mixers as M
from fasttalk_llm_microservice_amd.ops import mixers_ref as R
from test_mixer_kernels_gpu import DEV, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("routing", ["grouped_softmax", "top_logits", "top_sigmoid"])
@pytest.mark.parametrize("rows,experts,top,groups,keep", [(1, 1, 1, 1, 1), (16, 6, 2, 1, 1), (17, 32, 4, 4, 2),
                                                         (100, 33, 3, 3, 2), (9, 64, 8, 8, 4), (33, 64, 64, 64, 64)])
def test_moe_route(routing, rows, experts, top, groups, keep):
    if routing == "top_logits":
        groups = keep = 1
    g = torch.Generator().manual_seed(rows + experts)
    h, router = rnd(rows, 2048, dt=torch.bfloat16, g=g), rnd(experts, 2048, g=g, scale=2048 ** -0.5)
    bias = rnd(experts, g=g, scale=0.1)
    parts = M.route_parts(router.to(DEV))
    assert M.moe_route_fits(h.to(DEV), parts, experts)
    idx, wts = M.moe_route(h.to(DEV), parts, bias.to(DEV), experts, top, routing, 1.7, groups, keep)
    few = None
    if routing == "grouped_softmax":            # the kernel of few rows, a workgroup each
        few = M.moe_route_softmax(h.to(DEV), router.to(DEV), bias.to(DEV), top, groups, keep)
    z = h.double() @ router.double().t()
    if routing == "grouped_softmax":
        i64, w64 = R.moe_topk(z.float(), bias, top, groups, keep)
    else:
        z = (z + bias.double()).float()
        i64, w64 = R.moe_top_sigmoid(z, top, 1.7, groups, keep) if routing == "top_sigmoid" else R.moe_top_logits(z, top)
        w64 = w64 * (1.7 if routing == "top_logits" else 1.0)
    # logits differ from the 64-bit ones by fp32 sums of 2048 terms (2^-19): no choice of these hangs on that
    assert torch.equal(idx.cpu(), i64.int())
    torch.testing.assert_close(wts.cpu(), w64.float(), rtol=2e-5, atol=1e-6)
    if few is not None:
        assert torch.equal(few[0].cpu(), i64.int())
        torch.testing.assert_close(few[1].cpu(), w64.float(), rtol=2e-5, atol=1e-6)


def test_ties_go_to_the_lower_index():
    h = torch.ones(3, 2048, dtype=torch.bfloat16, device=DEV)
    router = torch.zeros(40, 2048, device=DEV)
    router[7] = 1.0
    idx, wts = M.moe_route(h, M.route_parts(router), None, 40, 5, "top_logits")
    assert idx.tolist() == [[7, 0, 1, 2, 3]] * 3 and bool((wts[:, 0] > 0.99).all())


def test_layer_of_many_experts_in_a_decode_step():
    """More experts than one workgroup's rows pay for: the library product and the choice kernel, with the same choice."""
    from fasttalk_llm_microservice_amd.models.mixers import MoEFF
    g = torch.Generator().manual_seed(2)
    sizes = {"router": (96, 128), "correction": (96,)}
    size = lambda n: sizes.get(n, (128, 32) if n.endswith("down") else (32, 128))      # noqa: E731
    moe = MoEFF(lambda n: rnd(*size(n), g=g, scale=0.1), 96, 4, 7.0, 8, 4, None, torch.bfloat16, DEV)
    h = rnd(5, 128, dt=torch.bfloat16, g=g).to(DEV)
    idx, wts = moe.route(h)
    i2, w2 = M.moe_route_softmax(h, moe.router, moe.correction, 4, 8, 4)
    assert torch.equal(idx, i2)
    torch.testing.assert_close(wts, w2, rtol=1e-5, atol=1e-7)     # fp32 logits of 128 terms in another order
