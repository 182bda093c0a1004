"""Activations of the gated products far from zero (csrc/mixers/few_rows.h fr_act): gates of exact values over the ranges where
the exponential leaves the normal numbers, through every kernel that has the activation in its epilogue, against 64 bits."""
import pytest
import torch
import torch.nn.functional as F

from fasttalk_llm_microservice_amd.ops import mixers as M

pytestmark = pytest.mark.gpu
DEV = "cuda"
LIMIT = 7.0
# gates from, to and step: whole multiples of the step are the sum of two bf16 numbers
SWEEP = {"silu": (-110.0, 110.0, 2.0 ** -7), "gelu_tanh": (-13.0, 13.0, 2.0 ** -10), "clamp_glu": (-66.0, 66.0, 2.0 ** -7),
         "relu": (-110.0, 110.0, 2.0 ** -5), "relu_sq": (-110.0, 110.0, 2.0 ** -5)}


def gates(act):
    lo, hi, step = SWEEP[act]
    v = torch.arange(lo, hi, step, dtype=torch.float64, device=DEV)
    coarse = v.bfloat16()
    fine = (v - coarse.double()).bfloat16()
    assert bool((coarse.double() + fine.double() == v).all())
    return v, coarse, fine


def act64(g, u, act):
    if act == "relu_sq":
        return torch.relu(g) ** 2
    if act == "clamp_glu":
        g = g.clamp(max=LIMIT)
        return g * torch.sigmoid(1.702 * g) * (u.clamp(-LIMIT, LIMIT) + 1)
    return {"gelu_tanh": lambda z: F.gelu(z, approximate="tanh"), "relu": torch.relu, "silu": F.silu}[act](g) * u


def close(got, g, u, act):
    """The argument of the exponential is exact or, for gelu and clamp, off by three roundings: of 2^7, 2^7 * 3 * 2^-24 = 2^-15.4
    of the result, beside the 2^-9 of its own rounding.  Sigmoids below the smallest normal number may be 0: 2^-126 * 2^7 * 2."""
    want = act64(g, u, act)
    if act == "gelu_tanh":           # (64 bits of 1 + tanh lose the tail as well)
        want = g * torch.sigmoid(2 * 0.7978845608028654 * (g + 0.044715 * g ** 3)) * u
    assert bool(torch.isfinite(got).all()), g[~torch.isfinite(got).expand(g.shape)][:8]
    err = (got.double() - want).abs()
    assert bool((err <= want.abs() * 2.0 ** -8 + 2.0 ** -117).all()), float((err / (want.abs() + 2.0 ** -117)).max())


def columns(act, k):
    """Weights whose products with a row of ones at 0 and 1 are the gates, and 1 for the up matrix."""
    v, coarse, fine = gates(act)
    n = len(v)
    w = torch.zeros(n if act == "relu_sq" else 2 * n, k, dtype=torch.bfloat16, device=DEV)
    w[:n, 0], w[:n, 1] = coarse, fine
    w[n:, 0] = 1.0
    return v, w


@pytest.mark.parametrize("act", list(SWEEP))
@pytest.mark.parametrize("rows", [3, 30, 40])
def test_products_of_few_rows(act, rows):
    v, w = columns(act, 128)
    x = torch.zeros(rows, 128, dtype=torch.bfloat16, device=DEV)
    x[:, :2] = 1.0
    y = torch.empty(rows, len(v), dtype=torch.bfloat16, device=DEV)
    M.native_mixers().few_rows_gemm(y, x, w, None, M.FEW_ACTS[act], LIMIT)
    close(y, v.expand(rows, -1), torch.ones_like(v).expand(rows, -1), act)


@pytest.mark.parametrize("act", list(SWEEP))
@pytest.mark.parametrize("form", range(8))
def test_tiles(act, form):
    v, w = columns(act, 64)
    x = torch.zeros(3, 64, dtype=torch.bfloat16, device=DEV)
    x[:, :2] = 1.0
    y = torch.empty(3, len(v), dtype=torch.bfloat16, device=DEV)
    M.native_mixers().tile_gemm(y, x, w, None, M.FEW_ACTS[act], LIMIT, form)
    close(y, v.expand(3, -1), torch.ones_like(v).expand(3, -1), act)


@pytest.mark.parametrize("act", ["silu", "gelu_tanh", "clamp_glu"])
@pytest.mark.parametrize("width,experts", [(64, 2), (72, 2), (64, 128)])
def test_experts_of_many_rows(act, width, experts):
    """A row a gate, equal experts that hand the activation on: tall groups (tiles), rows that are no whole stages, short groups."""
    v, coarse, fine = gates(act)
    v, coarse, fine = v[::5], coarse[::5], fine[::5]
    t = len(v)
    h = torch.zeros(t, width, dtype=torch.bfloat16, device=DEV)
    h[:, 0], h[:, 1], h[:, 2] = coarse, fine, 1.0
    wgu = torch.zeros(experts, 2 * width, width, dtype=torch.bfloat16, device=DEV)
    wgu[:, :width, :2] = 1.0
    wgu[:, width:, 2] = 1.0
    wdown = torch.eye(width, dtype=torch.bfloat16, device=DEV).repeat(experts, 1, 1)
    idx = (torch.arange(t, device=DEV) % experts).int()[:, None].contiguous()
    y = M.experts_many(h, idx, torch.ones(t, 1, device=DEV), wgu, wdown, act, LIMIT)
    close(y, v[:, None].expand(-1, width), torch.ones(t, width, dtype=torch.float64, device=DEV), act)


@pytest.mark.parametrize("act,lo,hi", [("silu", -104.5, -88.0), ("gelu_tanh", -10.75, -10.0), ("clamp_glu", -61.5, -51.5)])
def test_experts_of_few_rows(act, lo, hi):
    width, experts = 64, 4
    v = torch.linspace(lo, hi, 64, dtype=torch.float64, device=DEV)
    coarse = v.bfloat16()
    fine = (v - coarse.double()).bfloat16()
    v = coarse.double() + fine.double()
    h = torch.zeros(64, width, dtype=torch.bfloat16, device=DEV)
    h[:, 0], h[:, 1], h[:, 2] = coarse, fine, 1.0
    wgu = torch.zeros(experts, 2 * width, width, dtype=torch.bfloat16, device=DEV)
    wgu[:, :width, :2] = 1.0
    wgu[:, width:, 2] = 1.0
    wdown = torch.eye(width, dtype=torch.bfloat16, device=DEV).repeat(experts, 1, 1)
    idx = (torch.arange(64, device=DEV) % experts).int()[:, None].contiguous()
    y = M.experts_few(h, idx, torch.ones(64, 1, device=DEV), wgu, wdown, act, LIMIT)
    close(y, v[:, None].expand(-1, width), torch.ones(64, width, dtype=torch.float64, device=DEV), act)
