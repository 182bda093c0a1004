"""Recurrences of long segments in chunk form (csrc/mixers/chunk_state.hip) against the same walk in 64
bits: segment lengths around the chunk of 64 rows and the form's lower bound, sequences that continue,
padding, sizes off the tiles.  Its error may not exceed that of the row-by-row kernel."""
import pytest
import torch

from fasttalk_llm_microservice_amd.ops import mixers as M

pytestmark = pytest.mark.gpu
DEV = "cuda"
D = torch.float64


def segments(lens, pos0, slots):
    start = [0]
    for n in lens:
        start.append(start[-1] + n)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)   # noqa: E731
    kv = [p + n for p, n in zip(pos0, lens)]
    return M.Segments(i32(start), i32(pos0), i32(slots), i32(kv), torch.zeros(len(lens), 1, dtype=torch.int32, device=DEV),
                      len(lens), max(lens), max(kv), host=(start, list(pos0), kv))


def walk(seg, state, step):
    """step(row, S) -> (S, output row); states as the kernels leave them."""
    state, out = state.to(D).clone(), {}
    for s in range(seg.num):
        slot, pos = int(seg.slot[s]), seg.host[1][s]
        if slot < 0:
            continue
        S = state[slot] if pos > 0 else torch.zeros_like(state[slot])
        for r in range(seg.host[0][s], seg.host[0][s + 1]):
            S, out[r] = step(r, S)
        state[slot] = S
    return state, out


def check(run, want_state, want, dv, monkeypatch):
    """run() -> (outputs, states), once in chunk form and once row by row."""
    got = run()
    monkeypatch.setattr(M, "CHUNK_ROWS", 1 << 30)
    base = run()
    rows = sorted(want)
    w = torch.stack([want[r] for r in rows])
    for i, (x, y) in enumerate(((w, lambda t: t[rows].to(D)), (want_state, lambda t: t.to(D)))):
        e, b = (float((y(t[i]) - x).norm() / x.norm()) for t in (got, base))
        # fp32 sums of 64-row blocks and their carry: a few units of 2^-23
        assert e < 2e-6 and e < 1.5 * b + 1e-7, (e, b)
    return got


SHAPES = [([64], [0]), ([31, 32, 1, 65], [0, 5, 9, 0]), ([127, 200, 40], [64, 0, 3]), ([520], [0])]


@pytest.mark.parametrize("dt_", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("lens,pos0", SHAPES)
@pytest.mark.parametrize("heads,groups,n,dv", [(4, 2, 128, 128), (6, 3, 20, 24), (3, 1, 64, 72)])
def test_state_space(dt_, lens, pos0, heads, groups, n, dv, monkeypatch):
    g = torch.Generator().manual_seed(sum(lens) + n)
    T = sum(lens)
    slots = list(range(len(lens)))
    if len(lens) > 3:
        slots[1] = -1                                       # a padding segment of chunk length
    seg = segments(lens, pos0, slots)
    xbc = (torch.randn(T, heads * dv + 2 * groups * n, generator=g) * 0.5).to(DEV, dt_)
    dt = torch.randn(T, heads + 3, generator=g).to(DEV, dt_)[:, 3:]
    a_log, bias, skip = (torch.rand(heads, generator=g).to(DEV) for _ in range(3))
    bias = bias - 2.0
    s0 = torch.randn(len(lens), heads, n, dv, generator=g).to(DEV)
    x64, grp = xbc.to(D), torch.arange(heads, device=DEV) // (heads // groups)
    step64 = torch.nn.functional.softplus(dt.to(D) + bias.to(D))
    dec = torch.exp(-torch.exp(a_log.to(D)) * step64)

    def step(r, S):
        x = x64[r, :heads * dv].view(heads, dv)
        B = x64[r, heads * dv:heads * dv + groups * n].view(groups, n)[grp]
        C = x64[r, heads * dv + groups * n:].view(groups, n)[grp]
        S = dec[r][:, None, None] * S + step64[r][:, None, None] * B[:, :, None] * x[:, None]
        return S, ((S * C[:, :, None]).sum(1) + skip.to(D)[:, None] * x).flatten()

    ws, wo = walk(seg, s0, step)

    def run():
        st = s0.clone()
        return M.ssd_scan(xbc, dt, a_log, bias, skip, st, seg, heads, groups, n, dv), st

    y, _ = check(run, ws, wo, dv, monkeypatch)
    if -1 in slots:
        i = slots.index(-1)
        assert bool((y[seg.host[0][i]:seg.host[0][i + 1]] == 0).all())
