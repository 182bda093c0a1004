"""Experts on many rows: pairs sorted by expert, two grouped products, one weighted sum."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _act(act, u, limit):
    if act == "relu_sq":
        return u.relu() ** 2
    g, up = u.chunk(2, 1)
    if act == "silu_glu":
        return g * torch.sigmoid(g) * up
    g = g.clamp(max=limit)
    return g * torch.sigmoid(1.702 * g) * (up.clamp(-limit, limit) + 1)


@pytest.mark.parametrize("act", ["clamp_glu", "silu_glu", "relu_sq"])
@pytest.mark.parametrize("rows,experts,top,width,ff,choice", [
    (65, 5, 2, 64, 72, "random"),         # an activation tile that is not full, k past a step of 64
    (300, 1, 1, 72, 8, "random"),         # one expert, the smallest inner width
    (257, 40, 6, 256, 136, "random"),     # 64-row tiles, most of them part-filled
    (1100, 4, 3, 128, 128, "random"),     # 128-row tiles; more pairs than one turn of the sort per expert
    (1500, 16, 3, 64, 64, "few"),         # experts without a row, one with nearly all of them
])
def test_experts_many_matches_fp64(act, rows, experts, top, width, ff, choice):
    from fasttalk_llm_microservice_amd.ops import mixers as M
    gen = torch.Generator(device="cuda").manual_seed(rows + ff)
    rnd = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    glu = act != "relu_sq"
    h = rnd(rows, width).bfloat16()
    wgu = (rnd(experts, (2 if glu else 1) * ff, width) * width ** -0.5).bfloat16()
    wdown = (rnd(experts, width, ff) * ff ** -0.5).bfloat16()
    score = rnd(rows, experts)
    if choice == "few":
        score[:, 3] += 8
        score[:, 5:9] -= 50
    idx = score.topk(top).indices.int().contiguous()
    wts = torch.rand(rows, top, generator=gen, device="cuda")
    shared = rnd(rows, width).bfloat16()
    gate_w = (rnd(width) * width ** -0.5).bfloat16()
    assert M.experts_many_ok(h, wgu, wdown)
    want = torch.zeros(rows, width, dtype=torch.float64, device="cuda")
    size = torch.zeros_like(want)
    for e in range(experts):
        y = _act(act, h.double() @ wgu[e].double().t(), 7.0)
        w = (wts.double() * (idx == e)).sum(1, keepdim=True)
        want += w * (y @ wdown[e].double().t())
        size += w * (y.abs() @ wdown[e].double().abs().t())
    # two bf16 roundings, each of at most half a unit in the eighth bit: 2^-8 of the activation (a term of the
    # second product) and 2^-8 of the second product; fp32 sums of at most 256 terms are far below that
    bound = 2 ** -7 * size + 1e-5
    for sh, gw in ((None, None), (shared, None), (shared, gate_w)):
        got = M.experts_many(h, idx, wts, wgu, wdown, act, 7.0, sh, gw)
        ref = want
        if sh is not None:
            ref = ref + sh.double() * (torch.sigmoid(h.double() @ gw.double())[:, None] if gw is not None else 1.0)
        assert ((got.double() - ref).abs() <= bound + 1e-5 * ref.abs()).all()
