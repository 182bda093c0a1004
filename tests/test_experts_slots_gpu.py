"""Experts of fewer (row, choice) pairs than experts (csrc/mixers/few_rows.hip: the grid has a row per choice, and the next
round's loads are in flight under a round's products) against the same sums in 64 bits: up to 64 experts and past them, repeated
choices, indices outside the experts, a grid row per choice in both products, one or none, k of one round and of uneven ones, short (no
loads ahead) and long in both products and in either."""
import pytest
import torch

from fasttalk_llm_microservice_amd.ops import mixers as M

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("experts", [3, 63, 64, 65])
@pytest.mark.parametrize("rows,top", [(1, 1), (1, 2), (2, 6), (10, 6), (16, 4)])
@pytest.mark.parametrize("ff,width,act", [(24, 40, "relu_sq"), (136, 1032, "silu_glu"), (1048, 1032, "relu_sq"), (1048, 40, "silu_glu")])
def test_choices(experts, rows, top, ff, width, act):
    g = torch.Generator(device=DEV).manual_seed(experts * rows + top)
    rnd = lambda *s, scale=1.0: (torch.randn(*s, generator=g, device=DEV) * scale).bfloat16()   # noqa: E731
    h = rnd(rows, width)
    w1, w2 = rnd(experts, (1 if act == "relu_sq" else 2) * ff, width, scale=width ** -0.5), rnd(experts, width, ff, scale=ff ** -0.5)
    idx = torch.randint(-1, experts + 2, (rows, top), generator=g, device=DEV).int()
    idx[0, 0] = experts - 1
    wts = torch.rand(rows, top, generator=g, device=DEV)
    got = M.experts_few(h, idx, wts, w1, w2, act)
    e = torch.where((idx < 0) | (idx >= experts), 0, idx).long()
    u = torch.einsum("rw,rtfw->rtf", h.double(), w1.double()[e])
    y = torch.relu(u) ** 2 if act == "relu_sq" else u[..., :ff] * torch.sigmoid(u[..., :ff]) * u[..., ff:]
    want = torch.einsum("rt,rtf,rtwf->rw", wts.double(), y, w2.double()[e])
    size = torch.einsum("rt,rtf,rtwf->rw", wts.double(), y.abs(), w2.double()[e].abs())
    # the activations are rounded to bf16 in between (one unit, 2^-8, where a sum lies near a boundary), the rest is fp32
    assert bool(((got.double() - want).abs() <= size * 2.0 ** -8 + 1e-5).all())
