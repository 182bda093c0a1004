"""Grouped products in tiles of 256 rows with shorter last pieces (csrc/mixers/tile_gemm.hip, tile_groups_kernel) against the same
sums in 64 bits: group sizes at the edges of each tile, one to a few stages of k (the groups begin at another of them in turn), more
groups than a wave has lanes, plain, gated and through an index."""
import pytest
import torch

from fasttalk_llm_microservice_amd.ops import mixers as M

pytestmark = pytest.mark.gpu
DEV = "cuda"
GROUPS = 8                       # tile_groups_kernel among tile_gemm.hip's forms
EDGES = [0, 1, 63, 64, 65, 127, 128, 129, 255, 256, 257, 320, 321, 384, 385, 512, 513]


def rnd(seed, *shape, scale=1.0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(*shape, generator=g, device=DEV) * scale).bfloat16()


def close(got, want, k, slope=1.0):
    """bf16 output: half a unit in the last place, plus fp32 sums of k terms of order 1 through an activation of this slope."""
    err = (got.double() - want).abs()
    bound = want.abs() * 2.0 ** -8 + slope * (k ** 0.5 * 2.0 ** -22 + 2.0 ** -20)
    assert bool((err <= bound).all()), float((err - bound).max())


def product(a, w, counts, act=None):
    out = torch.full((a.shape[0], w.shape[1] // (2 if act else 1)), 7.0, dtype=a.dtype, device=DEV)
    M.native_mixers().grouped_gemm(out, a, w, torch.tensor(counts).cumsum(0).int().to(DEV), M.FEW_ACTS[act], 0.0, GROUPS)
    return out


@pytest.mark.parametrize("counts", [EDGES, [3] * 70 + [700] + [0] * 5 + [40] * 60, [0] * 63 + [130] + [0] * 64 + [1]])
@pytest.mark.parametrize("k", [64, 192, 576, 1088])
def test_plain_groups(counts, k):
    e = len(counts)
    n = 8 * (-(-128 // e) * 256 // 8) - 248          # 128 tiles of columns or more over all groups, the last one 8 wide
    rows = sum(counts)
    a, w = rnd(e, rows, k), rnd(e + 1, e, n, k, scale=k ** -0.5)
    got = product(a, w, counts)
    s = 0
    for g, c in enumerate(counts):
        close(got[s:s + c], a[s:s + c].double() @ w[g].double().t(), k)
        s += c


@pytest.mark.parametrize("k", [64, 576])
@pytest.mark.parametrize("n", [8, 136])
def test_gated_groups(k, n):
    a, w = rnd(n, sum(EDGES), k), rnd(n + 1, len(EDGES), 2 * n, k, scale=k ** -0.5)
    got = product(a, w, EDGES, "silu")
    s = 0
    for g, c in enumerate(EDGES):
        u = a[s:s + c].double() @ w[g].double().t()
        close(got[s:s + c], u[:, :n] * torch.sigmoid(u[:, :n]) * u[:, n:], k, slope=8.0)
        s += c


@pytest.mark.parametrize("rows,experts,top", [(70, 16, 2), (300, 16, 4), (900, 16, 4), (2100, 16, 3)])
@pytest.mark.parametrize("act", ["silu_glu", "relu_sq"])
def test_experts(rows, experts, top, act):
    """The two products of experts_many one after the other, the first through the index of sorted rows."""
    width, ff = 2048, 1088                           # (9 tiles of gated columns; the second product's k is 17 stages)
    g = torch.Generator(device=DEV).manual_seed(rows)
    h = rnd(rows, rows, width)
    wgu = rnd(1, experts, (2 if act == "silu_glu" else 1) * ff, width, scale=width ** -0.5)
    wdown = rnd(2, experts, width, ff, scale=ff ** -0.5)
    idx = torch.rand(rows, experts, generator=g, device=DEV).topk(top).indices.int().contiguous()
    wts = torch.rand(rows, top, generator=g, device=DEV)
    got = M.experts_many(h, idx, wts, wgu, wdown, act)
    want, size = torch.zeros(rows, width, dtype=torch.float64, device=DEV), torch.zeros(rows, width, dtype=torch.float64, device=DEV)
    for e in range(experts):
        u = h.double() @ wgu[e].double().t()
        y = u.relu() ** 2 if act == "relu_sq" else u[:, :ff] * torch.sigmoid(u[:, :ff]) * u[:, ff:]
        w = (wts.double() * (idx == e)).sum(1, keepdim=True)
        want += w * (y @ wdown[e].double().t())
        size += w * (y.abs() @ wdown[e].double().abs().t())
    # two bf16 roundings, each half a unit in the eighth bit: 2^-8 of each term of the second product and of its sum
    assert bool(((got.double() - want).abs() <= 2.0 ** -7 * size + 1e-5).all())


@pytest.mark.parametrize("before,count", [([0, 0, 0], 700), ([300, 40, 900], 1000), ([1, 513, 64], 449)])
def test_equal_rows(before, count):
    """A row's result is the same bits wherever its tile lies: in each of its group's, whole or short, and behind others' rows."""
    k, n, e = 1088, 16 * 256, 16
    w = rnd(1, e, n, k, scale=k ** -0.5)
    row = rnd(2, 1, k)
    counts = [before[i % 3] for i in range(7)] + [count] + [20] * (e - 8)
    a = row.expand(sum(counts), k).contiguous()
    got = product(a, w, counts)
    alone = product(row.expand(e * 30, k).contiguous(), w, [30] * e)
    s = 0
    for g, c in enumerate(counts):
        assert torch.equal(got[s:s + c], alone[30 * g:30 * g + 1].expand(c, n))
        s += c
