"""Products of many rows (csrc/mixers/tile_gemm.hip) against the same sums in 64 bits: every form of tile at its edges (row and
column remainders, one to a few stages of k, rows that are no whole 16-byte pieces), with each epilogue, and grouped."""
import pytest
import torch
import torch.nn.functional as F

from fasttalk_llm_microservice_amd.ops import mixers as M

pytestmark = pytest.mark.gpu
DEV = "cuda"
FORMS = [(0, 256, 256), (1, 256, 128), (2, 192, 128), (3, 128, 128), (4, 64, 128), (5, 64, 64), (6, 64, 32), (7, 32, 64)]


def rnd(seed, *shape, scale=1.0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(*shape, generator=g, device=DEV) * scale).bfloat16()


def act64(u, act, limit):
    if act is None:
        return u
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


@pytest.mark.parametrize("form,bm,bn", FORMS)
@pytest.mark.parametrize("k", [64, 128, 192, 448, 1088])
def test_plain_products(form, bm, bn, k):
    for rows, n in ((1, 8), (bm - 1, bn), (bm + 1, bn + 8), (2 * bm + 17, 2 * bn - 12), (9 * bm, bn + 3)):
        wide = rnd(rows + n, rows, k + 24)
        x, w, b = wide[:, 16:16 + k], rnd(k, n, k, scale=k ** -0.5), rnd(n, n)
        want = x.double() @ w.double().t()
        out = torch.full((rows, n + 8), 7.0, dtype=x.dtype, device=DEV)      # rows apart: nothing past them is written
        M.native_mixers().tile_gemm(out[:, :n], x, w, None, 0, 0.0, form)
        close(out[:, :n], want, k)
        assert bool((out[:, n:] == 7.0).all())
        y = torch.empty(rows, n, dtype=x.dtype, device=DEV)
        M.native_mixers().tile_gemm(y, x, w, b, 0, 0.0, form)
        close(y, want + b.double(), k)


@pytest.mark.parametrize("form,bm,bn", FORMS)
@pytest.mark.parametrize("act", ["gelu_tanh", "relu", "silu", "clamp_glu", "relu_sq"])
def test_activations(act, form, bm, bn):
    for rows, ff, k in ((bm + 5, bn // 2 + 8, 320), (3, 20, 64)):
        x, w = rnd(rows, rows, k), rnd(ff, ff if act == "relu_sq" else 2 * ff, k, scale=k ** -0.5)
        y = torch.empty(rows, ff, dtype=x.dtype, device=DEV)
        M.native_mixers().tile_gemm(y, x, w, None, M.FEW_ACTS[act], 1.5, form)
        close(y, act64(x.double() @ w.double().t(), act, 1.5), k, slope=32.0)


@pytest.mark.parametrize("rows,n,k,act", [(65, 272, 2048, None), (300, 2048, 128, None), (700, 1024, 256, "silu"),
                                          (1500, 512, 512, "relu_sq")])
def test_rule_takes_them(rows, n, k, act):
    """Through the entry points, at sizes where the rule says so; one element of k more, and the library's product serves."""
    x, w = rnd(1, rows, k), rnd(2, n, k, scale=k ** -0.5)
    assert M._tile_gemm(x, w, None, act, 1.5) is not None
    y = M.linear(x, w) if act is None else M.linear_act(x, w, act, 1.5)
    close(y, act64(x.double() @ w.double().t(), act, 1.5), k, slope=32.0)
    x, w = rnd(1, rows, k + 8), rnd(2, n, k + 8, scale=k ** -0.5)
    assert M._tile_gemm(x, w, None, act, 1.5) is None
    assert M._tile_gemm(rnd(1, rows, k + 4)[:, 4:], rnd(2, n, k), None) is None        # rows off 16 bytes


@pytest.mark.parametrize("counts", [[300, 0, 1, 257, 256, 0, 700], [50, 64, 128, 129, 0, 90], [1] * 70 + [9000]])
@pytest.mark.parametrize("n,k", [(264, 64), (40, 192)])
def test_groups(counts, n, k):
    rows, e = sum(counts), len(counts)
    a, w = rnd(e, rows, k), rnd(e + 1, e, n, k, scale=k ** -0.5)
    offs = torch.tensor(counts).cumsum(0).int().to(DEV)
    got = M.grouped_mm(a, w, offs)
    s = 0
    for g, c in enumerate(counts):
        close(got[s:s + c], a[s:s + c].double() @ w[g].double().t(), k)
        s += c
