"""The state-space scan's chunks on the bf16 matrix units (csrc/mixers/state_scan.hip) against the recurrence in 64 bits: chunk
edges, segments beside each other and beside short ones, states that go on, padding segments, decays from none to all."""
import pytest
import torch

from fasttalk_llm_microservice_amd.ops import mixers as M

pytestmark = pytest.mark.gpu
DEV = "cuda"
N = 128


def case(lens, heads, groups, dv, seed=0, shift=-3.0, wide=0):
    g = torch.Generator(device=DEV).manual_seed(seed + sum(lens))
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)   # noqa: E731
    t, width = sum(lens), heads * dv + 2 * groups * N
    xbc = (rnd(t, width + wide) * 0.7).bfloat16()[:, :width]
    return (xbc, rnd(t, heads + 3).bfloat16()[:, :heads], rnd(heads).abs(), rnd(heads) + shift, rnd(heads),
            rnd(len(lens), heads, N, dv))


def reference(xbc, dt, a_log, dt_bias, skip, state, lens, pos, heads, groups, dv):
    t = xbc.shape[0]
    x, b, c = xbc.double().split([heads * dv, groups * N, groups * N], 1)
    x, (b, c) = x.view(t, heads, dv), (z.view(t, groups, N).repeat_interleave(heads // groups, 1) for z in (b, c))
    step = torch.nn.functional.softplus(dt.double() + dt_bias.double())
    decay = torch.exp(-torch.exp(a_log.double()) * step)
    y, out, size, r = torch.zeros(t, heads, dv, dtype=torch.float64, device=DEV), [], 0.0, 0
    for i, n in enumerate(lens):
        s = state[i].double() * (pos[i] > 0)
        for k in range(r, r + n):
            s = s * decay[k][:, None, None] + b[k][:, :, None] * (step[k][:, None] * x[k])[:, None]
            y[k] = torch.einsum("hnv,hn->hv", s, c[k]) + skip.double()[:, None] * x[k]
        r += n
        size = max(size, float(s.abs().max()))
        out.append(s)
    return y.reshape(t, -1), torch.stack(out), size


def run(args, lens, pos, heads, groups, dv, slots=None, least=64):
    xbc, dt, a_log, dt_bias, skip, state = args
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)   # noqa: E731
    start = [sum(lens[:i]) for i in range(len(lens) + 1)]
    y, state = torch.full((xbc.shape[0], heads * dv), 7.0, device=DEV), state.clone()
    assert M.native_mixers().state_scan_takes(y, xbc, heads, groups, N, dv, max(lens))
    M.native_mixers().ssd_scan(y, xbc, dt, a_log, dt_bias, skip, state, i32(start), i32(pos), i32(slots or list(range(len(lens)))),
                               len(lens), max(lens), heads, groups, N, dv, min(lens) < least, least)
    return y, state


@pytest.mark.parametrize("lens,pos", [([64], [0]), ([65], [5]), ([127, 128, 129], [0, 3, 0]), ([1000], [9]), ([64, 1, 40, 200, 1], [0, 7, 0, 1, 2]),
                                      ([192], [0]), ([257, 80], [4, 0])])
@pytest.mark.parametrize("heads,groups,dv", [(4, 2, 16), (2, 1, 48), (3, 3, 128)])
@pytest.mark.parametrize("shift", [-3.0, 3.0, -30.0])
def test_rows(lens, pos, heads, groups, dv, shift):
    """(a shift of 3: most decays are below e^-3; of -30: nothing decays and nothing is added)"""
    args = case(lens, heads, groups, dv, shift=shift, wide=8)
    y, state = run(args, lens, pos, heads, groups, dv)
    want, left, size = reference(*args, lens, pos, heads, groups, dv)
    # fp32 sums of 128 products with the state and up to 64 with pair weights, each of them exact to 2^-24 of its size
    bound = 2.0 ** -21 * (size * 128 ** 0.5 * 4 + float(want.abs().max()))
    assert float((y.double() - want).abs().max()) <= bound
    assert float((state.double() - left).abs().max()) <= 2.0 ** -21 * max(size, 1.0)


def test_padding_segments():
    heads, groups, dv, lens = 4, 2, 32, [100, 70, 130]
    args = case(lens, heads, groups, dv)
    good, states = run(args, lens, [0, 0, 0], heads, groups, dv)
    y, left = run(args, lens, [0, 0, 0], heads, groups, dv, slots=[0, -1, 2])
    assert torch.equal(y[:100], good[:100]) and torch.equal(y[170:], good[170:]) and bool((y[100:170] == 0).all())
    assert torch.equal(left[1], args[5][1]) and torch.equal(left[0], states[0])


@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("row", [0, 1, 14, 15, 16, 17, 30, 33, 47, 52, 63, 64, 67, 69])
def test_a_row_that_is_not_finite(bad, row):
    """Rows before it do not see it, wherever in its chunk it lies, nor do other segments, heads and columns."""
    heads, groups, dv, lens = 4, 2, 32, [100, 70, 130]
    args = case(lens, heads, groups, dv)
    good, _ = run(args, lens, [0, 0, 0], heads, groups, dv)
    at, n = 100 + row, heads * dv
    for col, seen in ((5, slice(5, 6)), (n + 3, slice(0, 2 * dv)), (n + groups * N + 3, slice(0, 2 * dv))):     # x, B, C
        keep = args[0][at, col].clone()
        args[0][at, col] = bad
        y, _ = run(args, lens, [0, 0, 0], heads, groups, dv)
        args[0][at, col] = keep
        assert torch.equal(y[:at], good[:at]) and torch.equal(y[170:], good[170:])
        others = torch.ones(n, dtype=torch.bool, device=DEV)
        others[seen] = False
        assert torch.equal(y[:, others], good[:, others])
        own = y[at:170 if col < n + groups * N else at + 1, seen]
        assert not bool(torch.isfinite(own).any())
        if col >= n + groups * N:                         # a row of C is its own output's alone
            assert torch.equal(y[at + 1:], good[at + 1:])
    args[1][at, 1] = bad if bad > 0 else float("nan")      # (a step of softplus(-inf) is none)
    y, _ = run(args, lens, [0, 0, 0], heads, groups, dv)
    others = [0, 2, 3]
    assert torch.equal(y[:at], good[:at]) and torch.equal(y[170:], good[170:])
    assert torch.equal(y.view(-1, heads, dv)[:, others], good.view(-1, heads, dv)[:, others])
    assert not bool(torch.isfinite(y[at:170].view(-1, heads, dv)[:, 1]).any())


def test_decays_of_any_size():
    """What a single row leaves to each later one, to a few units in the last place: sums of decays that fp32 does not hold, results
    below the smallest normal number, within a chunk and over its end."""
    dv, n, at = 16, 128, 40
    big, small = 24.5, -14.0                             # softplus(24.5) = 24.5 and softplus(-14) = 8.3e-7 in fp32
    for steps, x0, c0 in (([big, big, small, small], 1.0, 1.0), ([big, big, small, big, big], 2.0 ** 100, 2.0 ** 20),
                          ([small] * 3 + [big] + [small] * 60, 1.0, 1.0)):
        t = at + 1 + len(steps)
        xbc = torch.zeros(t, dv + 2 * n, device=DEV)
        xbc[at, :dv], xbc[at, dv], xbc[:, dv + n] = x0, 1.0, c0
        dt = torch.zeros(t, 1, device=DEV)
        dt[at + 1:, 0] = torch.tensor(steps)
        zero = torch.zeros(1, device=DEV)
        args = (xbc.bfloat16(), dt.bfloat16(), zero, zero, zero, torch.zeros(1, 1, n, dv, device=DEV))
        y, state = run(args, [t], [0], 1, 1, dv, least=1)
        step = torch.nn.functional.softplus(dt[:, 0]).double()
        want = torch.exp(-(step.cumsum(0)[at:] - step[:at + 1].sum())) * step[at] * x0
        # up to three factors, each within two units in the last place of 2^-24 (of 2^-149 below the smallest normal number), and as
        # many products of three parts, each rounded once
        for got, w, f in ((y[at:, 0].double(), want * c0, x0 * c0), (state[0, 0, 0, :1].double(), want[-1:], x0)):
            assert bool(((got - w).abs() <= 2.0 ** -20 * w + 2.0 ** -148 * f).all()), (got / w - 1).abs().max()
