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
    monkeypatch.setattr(M, "_chunks_pay", lambda *a: True)
    both = []
    for rows in (32, 1 << 30):
        monkeypatch.setattr(M, "CHANNEL_CHUNK_ROWS", rows)
        monkeypatch.setattr(M, "SSD_CHUNK_ROWS", rows)
        both.append(run())
    got, base = both
    rows = sorted(want)
    w = torch.stack([want[r] for r in rows])
    for i, (x, y) in enumerate(((w, lambda t: t[rows].to(D)), (want_state, lambda t: t.to(D)))):
        e, b = (float((y(t[i]) - x).norm() / x.norm()) for t in (got, base))
        # fp32 sums of 64-row blocks and their carry: a few units of 2^-23
        assert e < 2e-6 and e < 1.5 * b + 1e-7, (e, b)
    return got


# (the last: workgroups that look for their segment among more than 64, a long one of padding rows)
SHAPES = [([64], [0]), ([31, 32, 1, 65], [0, 5, 9, 0]), ([127, 200, 40], [64, 0, 3]), ([520], [0]),
          ([40, 65] + [1] * 66 + [513], [0, 3] + [7] * 66 + [2])]


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


@pytest.mark.parametrize("dt_", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("lens,pos0", SHAPES)
@pytest.mark.parametrize("heads,kvh,dk,dv", [(4, 2, 128, 128), (3, 3, 20, 24), (2, 1, 64, 72), (2, 2, 12, 16)])
@pytest.mark.parametrize("fast", [False, True], ids=["slow", "fast"])
def test_channel_delta(dt_, lens, pos0, heads, kvh, dk, dv, fast, monkeypatch):
    """``fast``: channels that forget within a few rows (decays down to e^-30), beside slow ones."""
    g = torch.Generator().manual_seed(sum(lens) + dk)
    T, slots = sum(lens), list(range(len(lens)))
    if len(lens) > 3:
        slots[1] = -1
    seg = segments(lens, pos0, slots)
    rnd = lambda *s: torch.randn(*s, generator=g).to(DEV, dt_)   # noqa: E731
    qkv, a, b = rnd(T, 2 * kvh * dk + heads * dv), rnd(T, heads * dk), rnd(T, heads)
    a_log = (torch.rand(heads, generator=g) + (1.5 if fast else -1.0)).to(DEV)
    bias = ((torch.rand(heads * dk, generator=g) - 0.5) * (12.0 if fast else 2.0) - 1.0).to(DEV)
    s0 = torch.randn(len(lens), heads, dk, dv, generator=g).to(DEV)
    x = qkv.to(D)
    unit = lambda v: v / torch.sqrt((v * v).sum(-1, keepdim=True) + 1e-6)   # noqa: E731
    q = unit(x[:, :kvh * dk].view(T, kvh, dk)).repeat_interleave(heads // kvh, 1) * dk ** -0.5
    k = unit(x[:, kvh * dk:2 * kvh * dk].view(T, kvh, dk)).repeat_interleave(heads // kvh, 1)
    v, beta = x[:, 2 * kvh * dk:].view(T, heads, dv), torch.sigmoid(b.to(D))
    sp = torch.nn.functional.softplus(a.to(D) + bias.to(D)).view(T, heads, dk)
    dec = torch.exp(-torch.exp(a_log.to(D))[None, :, None] * sp)

    def step(r, S):
        S = dec[r][:, :, None] * S
        u = beta[r][:, None] * (v[r] - (S * k[r][:, :, None]).sum(1))
        S = S + k[r][:, :, None] * u[:, None]
        return S, (S * q[r][:, :, None]).sum(1).flatten()

    ws, wo = walk(seg, s0, step)

    def run():
        st = s0.clone()
        return M.gated_delta_rule(qkv, a, b, a_log, bias, st, seg, heads, kvh, dk, dv), st

    y, _ = check(run, ws, wo, dv, monkeypatch)
    if -1 in slots:
        i = slots.index(-1)
        assert bool((y[seg.host[0][i]:seg.host[0][i + 1]] == 0).all())


@pytest.mark.parametrize("dt_", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("lens,pos0", SHAPES)
@pytest.mark.parametrize("heads,dk,dv", [(4, 128, 128), (3, 20, 24), (2, 64, 72), (2, 12, 16)])
@pytest.mark.parametrize("fast", [False, True], ids=["slow", "fast"])
def test_channel_linear(dt_, lens, pos0, heads, dk, dv, fast, monkeypatch):
    g = torch.Generator().manual_seed(sum(lens) + dk)
    T, slots = sum(lens), list(range(len(lens)))
    if len(lens) > 3:
        slots[1] = -1
    seg = segments(lens, pos0, slots)
    tau = 0.5 if fast else 8.0
    p = torch.randn(T, heads * (2 * dk + dv) + 8, generator=g).to(DEV, dt_)
    a = torch.randn(T, heads * dk, generator=g).to(DEV, dt_)
    bias = (torch.rand(heads * dk, generator=g) * (16.0 if fast else 3.0) - (8.0 if fast else 0.0)).to(DEV)
    s0 = torch.randn(len(lens), heads, dk, dv, generator=g).to(DEV)
    x = p.to(D)
    n = heads * dk
    q, k, v = x[:, :n].view(T, heads, dk) * dk ** -0.5, x[:, n:2 * n].view(T, heads, dk), x[:, 2 * n:2 * n + heads * dv].view(T, heads, dv)
    dec = torch.exp(torch.nn.functional.logsigmoid(a.to(D) + bias.to(D)) / tau).view(T, heads, dk)

    def step(r, S):
        S = dec[r][:, :, None] * S + k[r][:, :, None] * v[r][:, None]
        return S, (S * q[r][:, :, None]).sum(1).flatten()

    ws, wo = walk(seg, s0, step)

    def run():
        st = s0.clone()
        return M.gated_linear_attention(p, a, bias, tau, st, seg, heads, dk, dv), st

    check(run, ws, wo, dv, monkeypatch)


@pytest.mark.parametrize("dt_", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("dk,dv", [(18, 24), (7, 136), (101, 9)])
def test_channel_sizes_off_quads(dt_, dk, dv, monkeypatch):
    """Key sizes that are no multiple of the loads' four entries, more value tiles than waves."""
    test_channel_delta(dt_, [65, 130], [0, 7], 2, 1, dk, dv, False, monkeypatch)
    test_channel_linear(dt_, [65, 130], [0, 7], 2, dk, dv, True, monkeypatch)


@pytest.mark.parametrize("lens", [[1, 1], [5, 2], [300, 4]])
def test_longest_segment_as_a_bound(lens):
    """``max_rows`` beyond the step's rows: the same results as with the longest segment itself."""
    g = torch.Generator().manual_seed(11)
    heads, dk, dv, T = 2, 32, 32, sum(lens)
    rnd = lambda *s: (0.3 * torch.randn(*s, generator=g)).to(DEV)      # noqa: E731
    qkv, a, b, al, bias = rnd(T, 6 * 32), rnd(T, 64), rnd(T, 2), rnd(2), rnd(64)
    s0, out = rnd(2, heads, dk, dv), []
    for bound in (max(lens), 4096):
        seg = segments(lens, [3, 0], [0, 1])
        seg.max_rows = bound
        st = [s0.clone() for _ in range(3)]
        out.append([M.gated_delta_rule(qkv, a, b, al, bias, st[0], seg, heads, heads, dk, dv),
                    M.gated_linear_attention(qkv, a, bias, 4.0, st[1], seg, heads, dk, dv),
                    M.ssd_scan(qkv, b, al, al, al, st[2], seg, heads, heads, dk, dv)] + st)
    for x, y in zip(*out):
        # walk and chunk form, or step and walk: fp32 sums of a few hundred terms of order 1
        torch.testing.assert_close(x, y, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("first", [95.0, 60.0])
def test_state_space_forgets_at_once(first, monkeypatch):
    """Rates e^a_log up to infinity (e^95 in fp32): decays are 0, a row sees itself alone."""
    g = torch.Generator().manual_seed(12)
    heads, n, dv, T = 2, 16, 16, 130
    seg = segments([T], [5], [0])
    xbc = torch.randn(T, heads * dv + 2 * n, generator=g).to(DEV)
    dt, bias, skip = torch.randn(T, heads, generator=g).to(DEV), torch.zeros(heads, device=DEV), torch.ones(heads, device=DEV)
    a_log, s0 = torch.tensor([first, 0.0], device=DEV), torch.randn(1, heads, n, dv, generator=g).to(DEV)
    monkeypatch.setattr(M, "_chunks_pay", lambda *a: True)
    out = []
    for rows in (64, 1 << 30):
        monkeypatch.setattr(M, "SSD_CHUNK_ROWS", rows)
        st = s0.clone()
        out.append((M.ssd_scan(xbc, dt, a_log, bias, skip, st, seg, heads, 1, n, dv), st))
    for x, y in zip(*out):
        assert bool(y.isfinite().all())
        torch.testing.assert_close(x, y, rtol=1e-5, atol=1e-5)       # fp32 sums of a few hundred terms of order 1


@pytest.mark.parametrize("dt_", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads,kvh,dk", [(16, 16, 66), (18, 6, 128), (4, 2, 256), (8, 8, 64)])
def test_delta_preparation_of_many_rows(dt_, heads, kvh, dk):
    """Enough rows for the preparation that takes four rows a wave (but for channels of 64), a part-filled item at the
    end: the results of the segments alone, whose rows are prepared one by one."""
    g = torch.Generator().manual_seed(dk)
    count = 12288 // (heads + kvh) // 81 + 1
    T, dv = 81 * count, 16
    rnd = lambda *s: torch.randn(*s, generator=g).to(DEV, dt_)      # noqa: E731
    qkv, a, b = rnd(T, 2 * kvh * dk + heads * dv), rnd(T, heads * dk + 2)[:, 2:], rnd(T, heads)
    al, bias = torch.rand(heads, generator=g).to(DEV), torch.randn(heads * dk, generator=g).to(DEV)
    s0 = torch.randn(count, heads, dk, dv, generator=g).to(DEV)
    st = s0.clone()
    o = M.gated_delta_rule(qkv, a, b, al, bias, st, segments([81] * count, [3] * count, list(range(count))), heads, kvh, dk, dv)
    for i in range(count):
        r, si = slice(81 * i, 81 * i + 81), s0[i:i + 1].clone()
        alone = M.gated_delta_rule(qkv[r], a[r], b[r], al, bias, si, segments([81], [3], [0]), heads, kvh, dk, dv)
        # sums of dk squares in another order: a few units of 2^-23 of numbers of order 1 to 10, carried over 81 rows
        torch.testing.assert_close(o[r], alone, rtol=1e-4, atol=1e-4)
        torch.testing.assert_close(st[i:i + 1], si, rtol=1e-4, atol=1e-4)
