"""One row per sequence of the recurrences (csrc/mixers/state_step.hip) against 64 bits: padding and fresh slots,
part-filled column and row tiles, shared key heads, column ranges of wider rows."""
import pytest
import torch
import torch.nn.functional as F

from fasttalk_llm_microservice_amd.ops import mixers as M
from test_mixer_kernels_gpu import DEV, DTYPES, make_seg, rnd, to_dev

pytestmark = pytest.mark.gpu

# (key size, value size): one row tile and part of one, several, the largest; columns that do not fill 32
SIZES = [(3, 4), (32, 32), (40, 36), (128, 128), (200, 64), (256, 20)]



def step64(q, k, v, g, state, seg, delta=None):
    """S <- g S + k x^T and S^T q for each row in 64 bits; x = v, or with ``delta`` (beta) its correction."""
    state, out = state.double(), torch.zeros(*v.shape, dtype=torch.float64)
    for s in range(seg.num):
        slot = int(seg.slot[s])
        if slot < 0:
            continue
        S = g[s][:, :, None] * (state[slot] if int(seg.pos0[s]) > 0 else torch.zeros_like(state[slot]))
        x = v[s]
        if delta is not None:
            x = delta[s][:, None] * (x - (S * k[s][:, :, None]).sum(1))
        S = S + k[s][:, :, None] * x[:, None, :]
        out[s], state[slot] = (S * q[s][:, :, None]).sum(1), S
    return out.flatten(1), state


def close(got, want):
    """fp32 sums of at most 256 products of order 1, and fp32 exponentials: a few tens of 2^-23."""
    torch.testing.assert_close(got.cpu().double(), want, rtol=2e-5, atol=2e-5)


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("dk,dv", SIZES)
def test_steps(dt, dk, dv):
    g = torch.Generator().manual_seed(dk + dv)
    seg, _ = make_seg([1, 1, 1, 1], [7, 0, 3, 900], [2, 0, -1, 4])
    t, heads, kvh = 4, 4, 2
    wide = lambda n: rnd(t, n + 9, dt=dt, g=g)[:, 2:2 + n]      # noqa: E731
    state = rnd(5, heads, dk, dv, g=g)
    parts = lambda x, *n: [p.double().view(t, -1, w) for p, w in zip(x.split([a * b for a, b in n], 1), [b for _, b in n])]  # noqa: E731
    unit = lambda x: x / (x.square().sum(-1, keepdim=True) + 1e-6).sqrt()                  # noqa: E731
    rep = lambda x: x.repeat_interleave(heads // kvh, 1)                                   # noqa: E731
    dev = lambda *x: [y.to(DEV) for y in x]                                                # noqa: E731

    qkv, a, b = wide(2 * kvh * dk + heads * dv), wide(heads * dk), wide(heads)
    a_log, bias = rnd(heads, g=g) * 0.5, rnd(heads * dk, g=g)
    q, k, v = parts(qkv, (kvh, dk), (kvh, dk), (heads, dv))
    decay = (-a_log.double().exp()[:, None] * F.softplus(a.double().view(t, heads, dk) + bias.double().view(heads, dk))).exp()
    want, s64 = step64(rep(unit(q)) * dk ** -0.5, rep(unit(k)), v, decay, state, seg, torch.sigmoid(b.double()))
    s2 = state.to(DEV)
    close(M.gated_delta_rule(*dev(qkv, a, b, a_log, bias), s2, to_dev(seg), heads, kvh, dk, dv), want)
    close(s2, s64)

    qkv, a = wide(heads * (2 * dk + dv) + 5), wide(heads * dk)
    q, k, v = parts(qkv[:, :heads * (2 * dk + dv)], (heads, dk), (heads, dk), (heads, dv))
    decay = torch.sigmoid(a.double() + bias.double()).view(t, heads, dk) ** (1 / 3.0)
    want, s64 = step64(q * dk ** -0.5, k, v, decay, state, seg)
    s2 = state.to(DEV)
    close(M.gated_linear_attention(*dev(qkv, a, bias), 3.0, s2, to_dev(seg), heads, dk, dv), want)
    close(s2, s64)

    xbc, dts, skip, hb = wide(heads * dv + 2 * kvh * dk), wide(heads), rnd(heads, g=g), rnd(heads, g=g)
    x, k, q = parts(xbc, (heads, dv), (kvh, dk), (kvh, dk))
    step = F.softplus(dts.double() + hb.double())
    decay = (-a_log.double().exp() * step).exp()[:, :, None].expand(t, heads, dk)
    want, s64 = step64(rep(q), rep(k), x * step[:, :, None], decay, state, seg)
    live = (seg.slot[:seg.num] >= 0)[:, None, None]
    want = want + (skip.double()[:, None] * x * live).flatten(1)
    s2 = state.to(DEV)
    close(M.ssd_scan(*dev(xbc, dts, a_log, hb, skip), s2, to_dev(seg), heads, kvh, dk, dv), want)
    close(s2, s64)
