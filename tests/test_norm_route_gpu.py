"""Decode rows of a mixture layer: the norm step and the router behind it in one launch (csrc/mixers/moe_route.hip
route_rows_kernel), and the norm steps that sum the experts' results themselves (csrc/mixers/rows.hip ExpertRows)."""
import pytest
import torch

from fasttalk_llm_microservice_amd.ops import mixers as M
from fasttalk_llm_microservice_amd.ops import mixers_ref as R
from test_mixer_kernels_gpu import DEV, rnd

pytestmark = pytest.mark.gpu


# one pass and several, a router of fewer and more pieces than are in flight, one and two pieces of a row per thread
@pytest.mark.parametrize("routing,form", [("grouped_softmax", "rms"), ("top_logits", "layer"), ("top_sigmoid", "plain")])
@pytest.mark.parametrize("rows,width,experts,top,groups,keep,ydt", [
    (1, 256, 1, 1, 1, 1, torch.bfloat16), (256, 512, 6, 2, 1, 1, torch.bfloat16), (3, 2048, 17, 4, 1, 1, torch.float32), (64, 2048, 32, 4, 4, 2, torch.bfloat16),
    (2, 4096, 64, 8, 8, 4, torch.bfloat16), (5, 4352, 33, 3, 3, 2, torch.float32), (2, 8192, 64, 64, 64, 64, torch.bfloat16)])
def test_norm_route(routing, form, rows, width, experts, top, groups, keep, ydt):
    if routing == "top_logits":
        groups = keep = 1
    g = torch.Generator().manual_seed(rows + width)
    x, y = rnd(rows, width, g=g), rnd(rows, width + 8, dt=ydt, g=g)[:, :width]
    w, wb, b = (1 + rnd(width, g=g, scale=0.1), rnd(width, g=g), rnd(width, g=g))
    router, bias = rnd(experts, width, g=g, scale=width ** -0.5), rnd(experts, g=g, scale=0.1)
    wb, b = (wb if form == "rms" else None), (b if form == "layer" else None)
    d = [None if t is None else t.to(DEV) for t in (x, y, wb, w, b, router, bias)]
    assert M.norm_route_fits(*d[:6])
    h, (idx, wts) = M.norm_route(*d[:5], 1e-5, *d[5:], top, routing, 1.7, groups, keep)
    if form == "layer":
        want = R.add_layer_norm_rows(x, y, w, b, 1e-5, torch.float32)
    else:
        want, _ = R.add_rms_norm_rows(x, y, wb, 1e-5, None, w, torch.float32, False)
    torch.testing.assert_close(d[0].cpu(), x, rtol=1e-5, atol=1e-5)          # fp32 sums in another order
    torch.testing.assert_close(h.float().cpu(), want, rtol=2 ** -8, atol=1e-5)      # one rounding to bf16
    z = h.cpu().double() @ router.double().t()
    if routing == "grouped_softmax":
        i64, w64 = R.moe_topk(z.float(), bias, top, groups, keep)
    else:
        z = (z + bias.double()).float()
        i64, w64 = R.moe_top_sigmoid(z, top, 1.7, groups, keep) if routing == "top_sigmoid" else R.moe_top_logits(z, top)
        w64 = w64 * (1.7 if routing == "top_logits" else 1.0)
    # fp32 logits of a few thousand terms: a choice may only differ between experts that are as good as level
    same = idx.cpu() == i64.int()
    by = z.float() if routing != "grouped_softmax" else torch.softmax(z.float(), -1) + bias
    level = by.gather(1, idx.cpu().long()) - by.gather(1, i64.long())
    assert bool((same | (level.abs() < 2e-5)).all())
    torch.testing.assert_close(wts.cpu(), w64.float(), rtol=2e-4, atol=1e-5)


def test_router_of_rows_with_nan_names_the_same_experts():
    g = torch.Generator().manual_seed(1)
    h, router, bias = rnd(3, 512, dt=torch.bfloat16, g=g).to(DEV), rnd(12, 512, g=g).to(DEV), rnd(12, g=g).to(DEV)
    h[1, 5] = float("nan")
    idx, wts = M.moe_route_top_logits(h, router, bias, 3)
    i32, w32 = M.moe_route_top_logits(h.float(), router, bias, 3)            # (the kernel of fp32 rows)
    assert torch.equal(idx, i32)
    torch.testing.assert_close(wts, w32, rtol=1e-5, atol=1e-7, equal_nan=True)


@pytest.mark.parametrize("rows,width,top", [(1, 1032, 1), (3, 2048, 4), (5, 4096, 8), (2, 16384, 5)])
@pytest.mark.parametrize("shared", ["no", "as it is", "gated"])
def test_norm_steps_sum_the_experts(rows, width, top, shared):
    g = torch.Generator().manual_seed(rows * top)
    d, wts = rnd(rows * top, width, g=g).to(DEV), rnd(rows, top, g=g).abs().to(DEV)
    ds = rnd(rows, width, g=g).to(DEV) if shared != "no" else None
    gate = rnd(rows, g=g).to(DEV) if shared == "gated" else None
    parts = M.ExpertParts(d, wts, ds, gate)
    y = (wts[:, :, None] * d.view(rows, top, width)).sum(1)
    if ds is not None:
        y = y + ds * (torch.sigmoid(gate)[:, None] if gate is not None else 1.0)
    x, w, wb, b, add = rnd(rows, width, g=g), rnd(width, g=g), rnd(width, g=g), rnd(width, g=g), rnd(width, g=g)
    w, wb, b, add = (t.to(DEV) for t in (w, wb, b, add))
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)      # noqa: E731
    # a sequence's first token, one further on, and a row without a slot
    pos, slot = [0, 7, 3, 5, 9][:rows], [2, 0, -1, 4, 1][:rows]
    seg = M.Segments(start=i32(list(range(rows + 1))), pos0=i32(pos), slot=i32(slot), kv_len=i32([p + 1 for p in pos]),
                     block_tables=i32([[0]] * rows), num=rows, max_rows=1)
    state = rnd(5, width, g=g)
    states = [state.to(DEV), state.to(DEV)]
    calls = [lambda x, y: M.add_rms_norm_rows(x, y, wb, 1e-5, add, w, torch.bfloat16, True),
             lambda x, y: M.add_rms_norm_rows(x, y, None, 1e-5, None, w, torch.bfloat16),
             lambda x, y: M.add_rms_norm_rows(x, y, wb, 1e-5, None, None, torch.bfloat16),
             lambda x, y: M.add_layer_norm_rows(x, y, w, b, 1e-5, torch.bfloat16),
             lambda x, y: M.add_norm_shift_rows(x, y, wb, w, b, 1e-5, torch.bfloat16, states[isinstance(y, torch.Tensor)], seg)]
    for call in calls:
        xs = [x.to(DEV), x.to(DEV)]
        got, want = call(xs[0], parts), call(xs[1], y)
        torch.testing.assert_close(xs[0], xs[1], rtol=1e-5, atol=2e-5)       # fp32 sums in another order
        for a, c in zip(*(t if isinstance(t, tuple) else (t,) for t in (got, want))):
            assert (a is None) == (c is None)
            if a is not None:
                torch.testing.assert_close(a.float(), c.float(), rtol=2 ** -7, atol=1e-4)    # a rounding to bf16 on each side
    torch.testing.assert_close(*states, rtol=1e-5, atol=1e-4)


# in registers and not (rows / width), experts' results
@pytest.mark.parametrize("rows,width", [(1, 1032), (7, 2048), (3, 16392), (2, 30)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_layer_norm_behind_the_last_one(rows, width, dt):
    g = torch.Generator().manual_seed(width)
    x, y = rnd(rows, width, g=g).to(DEV), rnd(rows, width, g=g).to(DEV)
    w, b, nw, nb = (rnd(width, g=g).to(DEV) for _ in range(4))
    x2 = x.clone()
    got = M.add_layer_norm_rows(x, y, w, b, 1e-5, dt, (nw, nb))
    M.add_layer_norm_rows(x2, y, w, b, 1e-5, dt)
    assert torch.equal(x, x2)
    assert got.dtype == dt and torch.equal(got, M.layer_norm_rows(x2, nw, nb, 1e-5, dt))       # the same sums
    if dt == torch.bfloat16 and 1024 < width <= 16384:
        parts = M.ExpertParts(y, torch.ones(rows, 1, device=DEV), None, None)
        x3 = (x2 - M.layer_norm_rows(y, w, b, 1e-5, torch.float32))
        got = M.add_layer_norm_rows(x3, parts, w, b, 1e-5, dt, (nw, nb))
        want = M.layer_norm_rows(x3, nw, nb, 1e-5, torch.float32)
        torch.testing.assert_close(got.float(), want, rtol=2 ** -8, atol=1e-5)                 # one rounding to bf16


@pytest.mark.parametrize("rows,n", [(1, 8), (33, 4104)])
def test_capped_logits(rows, n):
    g = torch.Generator().manual_seed(n)
    x, w = rnd(rows, 256, dt=torch.bfloat16, g=g).to(DEV), rnd(n, 256, dt=torch.bfloat16, g=g).to(DEV)
    z = M.linear_f32(x, w)
    assert torch.equal(M.linear_f32(x, w, 30.0), M.tanh_cap_(z.clone(), 30.0))


@pytest.mark.parametrize("routing", ["grouped_softmax", "top_logits", "top_sigmoid"])
@pytest.mark.parametrize("rows", [65, 256, 257, 512, 513])
def test_layer_routes_alike_by_either_kernel(rows, routing):
    """A mixture's choice where a workgroup takes a row and where it takes sixteen, and behind its norm step."""
    from fasttalk_llm_microservice_amd.models.mixers import MoEFF
    g = torch.Generator().manual_seed(rows)
    sizes = {"router": (12, 2048), "correction": (12,), "router.b": (12,)}
    size = lambda n: sizes.get(n, (2048, 16) if n.endswith("down") else (16, 2048))      # noqa: E731
    groups, keep = (1, 1) if routing == "top_logits" else (4, 2)
    moe = MoEFF(lambda n: rnd(*size(n), g=g, scale=2048 ** -0.5), 12, 3, 7.0, groups, keep, None, torch.bfloat16, DEV, routing=routing)
    h = rnd(rows, 2048, dt=torch.bfloat16, g=g).to(DEV)
    idx, wts = moe.route(h)
    limited = routing != "top_logits"
    i2, w2 = M.moe_route(h, moe.router_parts, moe.correction if routing == "grouped_softmax" else moe.router_bias, 12, 3, routing,
                         1.0, groups if limited else 1, keep if limited else 1)
    near = (wts - w2).abs().max(1).values < 1e-4       # fp32 logits of 2048 terms in another order: level experts may change places
    assert bool((torch.equal(idx, i2) or float((idx != i2).any(1).float().mean()) < 0.01)) and bool(near.all())
    x, y, w = rnd(rows, 2048, g=g).to(DEV), rnd(rows, 2048, g=g).to(DEV), torch.ones(2048, device=DEV)
    got = moe.norm_route(x, y, None, w, None, 1e-5, torch.bfloat16)
    assert (got is not None) == (rows <= 256)
    if got is not None:
        i3, w3 = moe.route(got[0])
        assert torch.equal(i3, got[1][0])
        torch.testing.assert_close(w3, got[1][1], rtol=1e-5, atol=1e-7)
