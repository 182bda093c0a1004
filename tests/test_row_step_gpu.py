"""One row per sequence of a recurrent mixer in one launch (csrc/mixers/row_step.hip) against 64 bits: padding and fresh slots,
part-filled row and column tiles, every number of taps, column ranges of wider rows; and which steps it leaves alone."""
import pytest
import torch
import torch.nn.functional as F

from fasttalk_llm_microservice_amd.ops import mixers as M
from test_mixer_kernels_gpu import DEV, DTYPES, make_seg, rnd, to_dev
from test_state_step_gpu import step64

pytestmark = pytest.mark.gpu

# (key size, value size): part of a row tile, one, several, the largest; columns that fill no wave, some, all
SIZES = [(3, 4), (16, 16), (33, 20), (64, 100), (128, 128), (200, 64), (256, 128)]


def conv64(x, w, hist, seg, bias=None):
    """silu of the convolution over time of one row per sequence, in 64 bits; the histories behind it."""
    x, w, out, new = x.double(), w.double(), torch.zeros(*x.shape, dtype=torch.float64), hist.double().clone()
    for s in range(seg.num):
        slot = int(seg.slot[s])
        if slot < 0:
            continue
        old = hist[slot].double() if int(seg.pos0[s]) > 0 else torch.zeros_like(hist[slot], dtype=torch.float64)
        rows = torch.cat([old, x[s:s + 1]])
        y = (rows * w.t()).sum(0)
        out[s], new[slot] = F.silu(y if bias is None else y + bias.double()), rows[1:]
    return out, new


def close(got, want, dt):
    """fp32 sums of at most 256 products of order 1, and fp32 exponentials: a few tens of 2^-23; bf16 results half a unit more."""
    tol = 4e-5 if dt == torch.float32 else 2.0 ** -8
    torch.testing.assert_close(got.cpu().double(), want, rtol=tol, atol=4e-5)


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("taps", [2, 3, 4])
@pytest.mark.parametrize("dk,dv", SIZES)
def test_row_step(dt, taps, dk, dv):
    g = torch.Generator().manual_seed(dk + dv + taps)
    seg, _ = make_seg([1, 1, 1, 1], [7, 0, 3, 900], [2, 0, -1, 4])
    t, heads, c = 4, 3, 3 * (2 * dk + dv)
    wide = lambda n: rnd(t, n + 9, dt=dt, g=g)[:, 2:2 + n]      # noqa: E731
    dev = lambda *x: [y.to(DEV) for y in x]                      # noqa: E731
    unit = lambda x: x / (x.square().sum(-1, keepdim=True) + 1e-6).sqrt()                  # noqa: E731
    heads_of = lambda x, n: x.double().view(t, heads, n)         # noqa: E731
    live = (seg.slot[:seg.num] >= 0)[:, None].double()

    def gated(o, gate, norm, silu):
        o, z = heads_of(o, dv), heads_of(gate, dv)
        o = o / (o.square().mean(-1, keepdim=True) + 1e-5).sqrt() * norm.double()
        return (o * (F.silu(z) if silu else torch.sigmoid(z))).flatten(1) * live

    for kind in (M.ROW_CHANNEL, M.ROW_HEAD):
        x, a, b, gate = wide(c), wide(heads * dk if kind == M.ROW_CHANNEL else heads), wide(heads), wide(heads * dv)
        w, hist, state = rnd(c, taps, g=g), rnd(5, taps - 1, c, g=g), rnd(5, heads, dk, dv, g=g)
        a_log, bias, norm = rnd(heads, g=g) * 0.5, rnd(a.shape[1], g=g), rnd(dv, g=g)
        y, h64 = conv64(x, w, hist, seg)
        q, k, v = (heads_of(p.contiguous(), n) for p, n in zip(y.split([heads * dk, heads * dk, heads * dv], 1), (dk, dk, dv)))
        z = heads_of((a.double() + bias.double()).contiguous(), a.shape[1] // heads)
        decay = (-a_log.double().exp()[:, None] * F.softplus(z)).exp().expand(t, heads, dk)
        o, s64 = step64(unit(q) * dk ** -0.5, unit(k), v, decay, state, seg, torch.sigmoid(b.double()))
        h2, s2 = dev(hist, state)
        got = M.row_step(kind, *dev(x, a, b, gate, w), h2, *dev(a_log, bias), 1.0, norm.to(DEV), 1e-5, kind == M.ROW_HEAD, s2,
                         to_dev(seg), heads, heads, dk, dv)
        close(got, gated(o, gate, norm, kind == M.ROW_HEAD), dt)
        close(s2, s64, torch.float32)
        close(h2, h64, torch.float32)

    x, a, gate = wide(c + 5), wide(heads * dk), wide(heads * dv)
    state, bias, norm = rnd(5, heads, dk, dv, g=g), rnd(heads * dk, g=g), rnd(dv, g=g)
    q, k, v = (heads_of(p.contiguous(), n) for p, n in zip(x.split([heads * dk, heads * dk, heads * dv, 5], 1), (dk, dk, dv)))
    decay = torch.sigmoid(heads_of((a.double() + bias.double()).contiguous(), dk)) ** (1 / 3.0)
    o, s64 = step64(q * dk ** -0.5, k, v, decay, state, seg)
    s2 = state.to(DEV)
    got = M.row_step(M.ROW_LINEAR, *dev(x, a), None, gate.to(DEV), None, None, None, bias.to(DEV), 3.0, norm.to(DEV), 1e-5, True,
                     s2, to_dev(seg), heads, heads, dk, dv)
    close(got, gated(o, gate, norm, True), dt)
    close(s2, s64, torch.float32)


# (heads, groups, state rows, value size): one wave, part-filled row tiles of each form, heads of several waves, the largest
GROUP_SIZES = [(2, 2, 16, 32), (2, 1, 3, 32), (3, 1, 33, 32), (6, 3, 64, 64), (4, 1, 65, 64), (8, 2, 128, 128), (2, 2, 128, 256)]


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("taps", [2, 3, 4])
@pytest.mark.parametrize("heads,groups,n,dv", GROUP_SIZES)
def test_group_step(dt, taps, heads, groups, n, dv):
    """State-space mixers.  The state of a fresh slot is not looked at: it holds NaN."""
    g = torch.Generator().manual_seed(heads + n + dv + taps)
    seg, _ = make_seg([1, 1, 1, 1], [7, 0, 3, 900], [2, 0, -1, 4])
    t, inner = 4, heads * dv
    c = inner + 2 * groups * n
    p = rnd(t, inner + c + heads + 3, dt=dt, g=g)
    z, x, step, _ = p.split([inner, c, heads, 3], 1)
    w, bias, hist, state = rnd(c, taps, g=g), rnd(c, g=g), rnd(5, taps - 1, c, g=g), rnd(5, heads, n, dv, g=g)
    a_log, dt_bias, skip, norm = rnd(heads, g=g) * 0.5, rnd(heads, g=g), rnd(heads, g=g), rnd(inner, g=g)
    bias = None if taps == 3 else bias
    y, h64 = conv64(x, w, hist, seg, bias)
    v, b, k = y.split([inner, groups * n, groups * n], 1)
    v = v.contiguous().view(t, heads, dv)
    b, k = (m.contiguous().view(t, groups, n).repeat_interleave(heads // groups, 1) for m in (b, k))
    dstep = F.softplus(step.double() + dt_bias.double())
    decay = (-a_log.double().exp() * dstep).exp()[:, :, None].expand(t, heads, n)
    o, s64 = step64(k, b * dstep[:, :, None], v, decay, state, seg)
    o = ((o.view(t, heads, dv) + skip.double()[:, None] * v).flatten(1) * F.silu(z.double())).view(t, groups, -1)
    live = (seg.slot[:seg.num] >= 0)[:, None].double()
    want = (o / (o.square().mean(-1, keepdim=True) + 1e-5).sqrt()).flatten(1) * norm.double() * live
    state[0], hist[0] = float("nan"), float("nan")
    pd, h2, s2 = p.to(DEV), hist.to(DEV), state.to(DEV)
    z, x, step, _ = pd.split([inner, c, heads, 3], 1)
    got = M.group_step(x, z, step, w.to(DEV), None if bias is None else bias.to(DEV), h2, a_log.to(DEV), dt_bias.to(DEV),
                       skip.to(DEV), norm.to(DEV), 1e-5, groups, s2, to_dev(seg), heads, groups, n, dv)
    close(got, want, dt)
    close(s2, s64, torch.float32)
    close(h2, h64, torch.float32)


def test_steps_left_alone():
    """Several rows a segment, shared key heads, one tap or five, value sizes of no whole fours or beyond 128: the launches before."""
    seg, _ = make_seg([1, 1], [7, 0], [1, 0])
    long, _ = make_seg([2], [7], [1])
    state = torch.zeros(2, 2, 32, 128, device=DEV)
    x = torch.zeros(2, 4, device=DEV)

    def takes(seg=seg, taps=4, kvh=2, dk=32, dv=128, kind=M.ROW_HEAD):
        w = torch.zeros(4, taps, device=DEV) if taps else None
        try:
            return M.row_step(kind, x, x, x, x, w, x, x, x, 1.0, x, 1e-5, True, state, to_dev(seg), 2, kvh, dk, dv) is not None
        except RuntimeError:              # (taken, and the shapes of this call refused)
            return True

    assert takes() and takes(taps=2) and takes(dk=256) and takes(dv=4)
    assert not (takes(seg=long) or takes(kvh=1) or takes(taps=1) or takes(taps=5) or takes(dv=126) or takes(dv=132) or
                takes(dk=257) or takes(kind=M.ROW_LINEAR))

    def group(seg=seg, taps=4, norm_groups=2, n=32, dv=128):
        try:
            return M.group_step(x, x, x, torch.zeros(4, taps, device=DEV), None, x, x, x, x, x, 1e-5, norm_groups, state, to_dev(seg),
                                2, 2, n, dv) is not None
        except RuntimeError:
            return True

    assert group() and group(taps=2) and group(n=64) and group(dv=512)
    assert not (group(seg=long) or group(norm_groups=1) or group(taps=1) or group(taps=5) or group(dv=48) or group(dv=544) or
                group(n=65) or group(n=129, dv=512))
