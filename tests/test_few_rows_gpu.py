"""Products of few rows and experts of few rows (csrc/mixers/few_rows.hip) against the same sums in
64 bits, at the edges of their tiles: row blocks of 16, column tiles of 16 and 32, steps of 64 in k
with whole and partial last steps, and each number of waves the sizes choose."""
import pytest
import torch
import torch.nn.functional as F

from fasttalk_llm_microservice_amd.ops import mixers as M

pytestmark = pytest.mark.gpu
DEV = "cuda"
ACTS = ["gelu_tanh", "relu", "silu", "clamp_glu", "relu_sq"]


def rnd(g, *shape, scale=1.0):
    return (torch.randn(*shape, generator=g) * scale).to(DEV, torch.bfloat16)


def act64(u, act, limit):
    if act == "relu_sq":
        return torch.relu(u) ** 2
    g, u = u.chunk(2, -1)
    if act == "clamp_glu":
        g, u = g.clamp(max=limit), u.clamp(-limit, limit) + 1
        return g * torch.sigmoid(1.702 * g) * u
    return {"gelu_tanh": lambda z: F.gelu(z, approximate="tanh"), "relu": torch.relu, "silu": F.silu}[act](g) * u


def close(got, want, k, slope=1.0):
    """bf16 output: half a unit in the last place (2^-9), plus fp32 sums of k terms of order 1 (rounding of
    each partial sum, sqrt(k) of them) seen through an activation of this slope."""
    err = (got.double() - want).abs()
    bound = want.abs() * 2.0 ** -8 + slope * (k ** 0.5 * 2.0 ** -22 + 2.0 ** -20)
    assert bool((err <= bound).all()), float((err - bound).max())


@pytest.mark.parametrize("rows", [1, 15, 16, 17, 33, 64])
@pytest.mark.parametrize("n,k", [(8, 8), (20, 72), (16, 64), (40, 1000), (2056, 1024), (48, 4160), (8200, 256), (16400, 64)])
def test_plain_products(rows, n, k):
    g = torch.Generator().manual_seed(rows * 1000 + n + k)
    wide = rnd(g, rows, k + 24)
    x, w, b = wide[:, 16:16 + k], rnd(g, n, k, scale=k ** -0.5), rnd(g, n)
    assert M._few_rows(x, w)
    want = x.double() @ w.double().t()
    y, f = torch.empty(rows, n, dtype=x.dtype, device=DEV), torch.empty(rows, n, device=DEV)
    M.native_mixers().few_rows_gemm(y, x, w, None, 0, 0.0)
    close(y, want, k)
    M.native_mixers().few_rows_gemm(y, x, w, b, 0, 0.0)
    close(y, want + b.double(), k)
    close(M.linear(x, w, b), want + b.double(), k)
    M.native_mixers().few_rows_gemm(f, x, w, None, 0, 0.0)
    assert float((f.double() - want).abs().max()) <= 2.0 ** -20 * k ** 0.5


@pytest.mark.parametrize("act", ACTS)
@pytest.mark.parametrize("rows,ff,k", [(1, 8, 16), (7, 24, 2048), (17, 1040, 264), (64, 64, 4096)])
def test_activations(act, rows, ff, k):
    g = torch.Generator().manual_seed(ff + k)
    x, w = rnd(g, rows, k), rnd(g, ff if act == "relu_sq" else 2 * ff, k, scale=k ** -0.5)
    close(M.linear_act(x, w, act, 1.5), act64(x.double() @ w.double().t(), act, 1.5), k, slope=32.0)


@pytest.mark.parametrize("act,name", [("clamp_glu", "clamp_glu"), ("relu_sq", "relu_sq"), ("silu_glu", "silu")])
@pytest.mark.parametrize("rows,experts,top,ff,width,shared", [
    (1, 4, 2, 8, 16, None), (5, 3, 3, 40, 96, "gate"), (17, 6, 2, 72, 128, "plain"),
    (64, 32, 6, 64, 256, "gate"), (64, 2, 1, 48, 64, None), (33, 1, 1, 32, 32, "plain")])
def test_experts(act, name, rows, experts, top, ff, width, shared):
    g = torch.Generator().manual_seed(rows + ff)
    mult = 1 if act == "relu_sq" else 2
    fs, gate = ff + 8, shared == "gate"
    h = rnd(g, rows, width)
    w1, w2 = rnd(g, experts, mult * ff, width, scale=width ** -0.5), rnd(g, experts, width, ff, scale=ff ** -0.5)
    sh = (rnd(g, mult * fs + gate, width, scale=width ** -0.5), rnd(g, width, fs, scale=fs ** -0.5)) if shared else None
    # every row chooses distinct experts; with one expert of two chosen by all, its list is full
    idx = torch.stack([torch.randperm(experts, generator=g)[:top] for _ in range(rows)]).int().to(DEV)
    wts = torch.rand(rows, top, generator=g).to(DEV)
    assert M.experts_few_ok(h, w1, w2, sh)
    got = M.experts_few(h, idx, wts, w1, w2, act, 1.5, sh, 0.75, gate)
    want = torch.zeros(rows, width, dtype=torch.float64, device=DEV)
    mag = torch.zeros_like(want)

    def one(a, b, x, limit):
        y = act64(x @ a.double().t(), name, limit).to(torch.bfloat16).double()
        return y @ b.double().t(), y.abs() @ b.double().abs().t()

    for r in range(rows):
        for k in range(top):
            e = int(idx[r, k])
            d, m = one(w1[e], w2[e], h[r:r + 1].double(), 1.5)
            want[r] += float(wts[r, k]) * d[0]
            mag[r] += float(wts[r, k]) * m[0]
    if sh:
        n1 = mult * fs
        d, m = one(sh[0][:n1], sh[1], h.double(), 0.75)
        f = torch.sigmoid(h.double() @ sh[0][n1].double())[:, None] if gate else 1.0
        want, mag = want + f * d, mag + f * m
    # the activations are rounded to bf16 in between (a sum near a rounding boundary may go either way: one unit,
    # 2^-8 of the magnitudes that meet), the rest is fp32
    err = (got.double() - want).abs()
    assert bool((err <= mag * 2.0 ** -8 + 1e-5).all()), float(err.max())
    torch.testing.assert_close(got, M.experts_few(h, idx, wts, w1, w2, act, 1.5, sh, 0.75, gate), rtol=0, atol=0)


@pytest.mark.parametrize("rows,experts,top", [(16, 8, 6), (17, 4, 6), (32, 8, 2), (64, 6, 3), (64, 32, 6)])
@pytest.mark.parametrize("act", ["clamp_glu", "relu_sq"])
def test_repeated_choices_keep_to_their_rows(act, rows, experts, top):
    """More pairs than rows for one expert (rows of NaN choose it again and again, indices outside the experts count as
    it): every row's result is that of the row alone."""
    g = torch.Generator().manual_seed(rows + top)
    width, ff, few = 64, 40, min(top, experts)
    w1 = rnd(g, experts, (1 if act == "relu_sq" else 2) * ff, width, scale=width ** -0.5)
    w2 = rnd(g, experts, width, ff, scale=ff ** -0.5)
    h, router = rnd(g, rows, width), torch.randn(experts, width, generator=g).to(DEV)
    h[:5] = float("nan")
    idx, wts = M.moe_route_top_logits(h, router, None, few)
    idx, wts = torch.cat([idx, idx[:, :top - few]], 1).contiguous(), torch.cat([wts, wts[:, :top - few]], 1).contiguous()
    idx[6, 0], idx[7, top - 1] = -1, experts
    idx[8:12] = 0
    idx[rows // 2:, 1] = 0
    spoiled = torch.full((rows * top * width,), float("nan"), device=DEV)     # what a row left out would read
    del spoiled
    got = M.experts_few(h, idx, wts, w1, w2, act, 1.5)
    alone = torch.cat([M.experts_few(h[r:r + 1], idx[r:r + 1].contiguous(), wts[r:r + 1], w1, w2, act, 1.5)
                       for r in range(rows)])
    assert bool(alone[5:].isfinite().all()) and bool(alone[:5].isnan().all())
    assert torch.equal(got[5:], alone[5:]) and bool(got[:5].isnan().all())
