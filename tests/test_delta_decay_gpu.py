"""Decays of the channel delta rule's chunk form (csrc/mixers/mx_common.h: delta_decay) over all the pre-activations and rates that
they can have, against the recurrence in 64 bits."""
import pytest
import torch

from fasttalk_llm_microservice_amd.ops import mixers as M

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("values", [(-3e38, -200.0, -90.0, -20.0, -1e-3), (0.0, 1e-3, 1.0, 20.0, 20.5), (-1.0, 88.0, 104.0, 3e38, float("inf"))])
def test_decays(values, dt):
    rows, heads, dk, dv = 130, 2, 16, 16
    g = torch.Generator(device=DEV).manual_seed(len(values))
    qkv = torch.randn(rows, 2 * heads * dk + heads * dv, generator=g, device=DEV).to(dt)
    a = torch.tensor(values, device=DEV)[torch.randint(0, len(values), (rows, heads * dk), generator=g, device=DEV)].to(dt)
    b = torch.randn(rows, heads, generator=g, device=DEV).to(dt)
    a_log, bias = torch.tensor([-3.0, 3.0], device=DEV), torch.zeros(heads * dk, device=DEV)
    i32 = lambda *v: torch.tensor(v, dtype=torch.int32, device=DEV)   # noqa: E731
    state, o = torch.zeros(1, heads, dk, dv, device=DEV), torch.empty(rows, heads * dv, device=DEV)
    M.native_mixers().gated_delta_rule(o, qkv, a, b, a_log, bias, state, i32(0, rows), i32(0), i32(0), 1, rows, heads, heads, dk, dv,
                                       False, 33)
    q, k, v = (t.double().view(rows, heads, -1) for t in qkv.split([heads * dk, heads * dk, heads * dv], 1))
    unit = lambda t: t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6)   # noqa: E731
    q, k = unit(q) * dk ** -0.5, unit(k)
    z = a.double().view(rows, heads, dk)
    # (x with x > 40 is its own softplus in 64 bits to within e^-40)
    decay = torch.exp(-torch.exp(a_log.double())[None, :, None] * torch.nn.functional.softplus(z, threshold=40.0))
    beta = torch.sigmoid(b.double())
    s, want = torch.zeros(heads, dk, dv, dtype=torch.float64, device=DEV), []
    for t in range(rows):
        s = s * decay[t][:, :, None]
        s = s + k[t][:, :, None] * (beta[t][:, None] * (v[t] - torch.einsum("hkv,hk->hv", s, k[t])))[:, None]
        want.append(torch.einsum("hkv,hk->hv", s, q[t]).reshape(-1))
    # fp32 sums over at most 64 + 16 terms of order 1 a chunk, decays of 2^-23 times their logarithm's size, 64 of them a product
    assert float((o.double() - torch.stack(want)).abs().max()) <= 5e-5
    assert float((state[0].double() - s).abs().max()) <= 5e-5
