"""Row kernels that hold a row in registers, at the edges of their widths: one and several register chunks (2048
entries each), widths and addresses that are not whole fours, and the widest rows beyond which the general kernels run."""
import pytest
import torch

from fasttalk_llm_microservice_amd.ops import mixers as M
from fasttalk_llm_microservice_amd.ops import mixers_ref as R
from test_mixer_kernels_gpu import DEV, DTYPES, rnd, tol

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("width,left", [(4, 4), (33, 4), (2048, 4), (2052, 4), (2052, 3), (5000, 8), (16384, 4), (16388, 4)])
def test_norms(dt, width, left):
    g = torch.Generator().manual_seed(width + left)
    wide = lambda d: rnd(3, width + left, dt=d, g=g)[:, left:]             # noqa: E731
    vec = lambda: 1 + rnd(width, g=g, scale=0.2)                            # noqa: E731
    w, b, x = vec(), vec(), rnd(3, width, g=g)
    dev = lambda *ts: [None if t is None else t.to(DEV) for t in ts]        # noqa: E731
    close = lambda a, e: torch.testing.assert_close(a.cpu().float(), e.float(), **tol(a.dtype))   # noqa: E731
    close(M.layer_norm_rows(*dev(x, w, b), 1e-5, dt), R.layer_norm_rows(x, w, b, 1e-5, dt))
    for y in (None, wide(dt)):
        x1, x2 = x.clone(), x.to(DEV)
        close(M.add_layer_norm_rows(x2, *dev(y, w, b), 1e-5, dt), R.add_layer_norm_rows(x1, y, w, b, 1e-5, dt))
        close(x2, x1)
    for y1, y2, nw in ((None, None, w), (wide(dt), None, None), (wide(torch.float32), wide(dt), w)):
        x1, x2 = x.clone(), x.to(DEV)
        want = R.add_scaled_rms_norm_rows(x1, y1, y2, 0.4, nw, 1e-5, dt)
        got = M.add_scaled_rms_norm_rows(x2, *dev(y1, y2), 0.4, *dev(nw), 1e-5, dt)
        close(x2, x1)
        assert (got is None) == (want is None)
        if want is not None:
            close(got, want)
    a, c = wide(dt), wide(dt)
    close(M.dual_rms_mean(*dev(a, c, w, b), 1e-5), R.dual_rms_mean(a, c, w, b, 1e-5, 0.5))


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("groups,gs,left", [(1, 4, 4), (3, 256, 4), (2, 260, 4), (2, 512, 3), (1, 2048, 8), (1, 2052, 4)])
def test_gate_group_norm(dt, groups, gs, left):
    g = torch.Generator().manual_seed(gs)
    y, w = rnd(5, groups * gs, g=g), 1 + rnd(groups * gs, g=g, scale=0.2)
    z = rnd(5, groups * gs + left, dt=dt, g=g)[:, left:]
    torch.testing.assert_close(M.gate_group_norm(y.to(DEV), z.to(DEV), w.to(DEV), 1e-5, groups, dt).cpu().float(),
                               R.gate_group_norm(y, z, w, 1e-5, groups, dt).float(), **tol(dt))


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("norm,rot,hd,nqh,nkh", [(True, 0, 128, 16, 4), (True, 128, 128, 16, 4), (False, 64, 128, 3, 1),
                                                 (True, 8, 12, 4, 2), (False, 12, 12, 4, 2), (True, 16, 64, 100, 28),
                                                 (True, 0, 64, 120, 9)])
def test_attn_prep(dt, norm, rot, hd, nqh, nkh):
    g = torch.Generator().manual_seed(hd + rot)
    nq, nk, nv, t = nqh * hd, nkh * hd, nkh * 20, 6
    qkv = rnd(t, nq + nk + nv + 4, dt=dt, g=g)[:, 4:]
    wq, wk = (1 + rnd(nq, g=g, scale=0.2), 1 + rnd(nk, g=g, scale=0.2)) if norm else (None, None)
    table = M.rope_table(40, rot, 50.0) if rot else None
    pos, slots = torch.tensor([3, 0, 39, 7, 1, 20]).int(), torch.tensor([5, 0, -1, 7, 2, 1]).int()
    kc1, vc1 = torch.zeros(2, 4, nk, dtype=dt), torch.zeros(2, 4, nv, dtype=dt)
    kc2, vc2 = kc1.to(DEV), vc1.to(DEV)
    q1 = R.attn_prep(qkv, nq, nk, wq, wk, 1e-5, table, rot, hd, pos, slots, kc1, vc1)
    mv = lambda x: x.to(DEV) if x is not None else None   # noqa: E731
    q2 = M.attn_prep(mv(qkv), nq, nk, mv(wq), mv(wk), 1e-5, mv(table), rot, hd, mv(pos), mv(slots), kc2, vc2)
    torch.testing.assert_close(q2.cpu(), q1, rtol=2e-5, atol=2e-5)
    torch.testing.assert_close(kc2.cpu().float(), kc1.float(), **tol(dt))
    torch.testing.assert_close(vc2.cpu().float(), vc1.float(), **tol(dt))


@pytest.mark.parametrize("rows,width,left", [(600, 512, 4), (600, 516, 4), (512, 516, 4), (513, 1024, 4), (600, 1028, 4), (64, 2050, 4),
                                             (65, 2050, 4), (64, 1023, 4), (600, 2052, 3)])
def test_norms_by_rows(rows, width, left):
    """Both sides of the rule on rows, widths and addresses."""
    g = torch.Generator().manual_seed(rows + width)
    dt = torch.bfloat16
    wide = lambda: rnd(rows, width + left, dt=dt, g=g)[:, left:]            # noqa: E731
    w, b, x = 1 + rnd(width, g=g, scale=0.2), rnd(width, g=g), rnd(rows, width, g=g)
    close = lambda a, e: torch.testing.assert_close(a.cpu().float(), e.float(), **tol(a.dtype))   # noqa: E731
    y, c = wide(), wide()
    for f, args in (("add_layer_norm_rows", lambda d: (x.clone().to(d), y.to(d), w.to(d), b.to(d), 1e-5, dt)),
                    ("add_scaled_rms_norm_rows", lambda d: (x.clone().to(d), y.to(d), c.to(d), 0.4, w.to(d), 1e-5, dt)),
                    ("dual_rms_mean", lambda d: (y.to(d), c.to(d), w.to(d), b.to(d), 1e-5, 0.5)),
                    ("layer_norm_rows", lambda d: (x.to(d), w.to(d), b.to(d), 1e-5, dt))):
        got, want = args(DEV), args("cpu")
        if f != "layer_norm_rows" and left == 3:                     # (.to makes rows dense: offset them on the GPU again)
            got = tuple(torch.cat([t[:, :3], t], 1)[:, 3:] if t is not None and hasattr(t, "dim") and t.dim() == 2 and t.dtype == dt
                        else t for t in got)
        close(getattr(M, f)(*got), getattr(R, f)(*want))
        if "add" in f:
            close(got[0], want[0])


@pytest.mark.parametrize("rows,nqh", [(512, 3), (513, 3), (513, 7)])
def test_attn_prep_by_rows(rows, nqh):
    """Both sides of the rule on rows and sizes (512 entries, 512 rows)."""
    g, dt, hd, rot = torch.Generator().manual_seed(rows), torch.bfloat16, 64, 16
    nq, nk, nv = nqh * hd, hd, 20
    qkv = rnd(rows, nq + nk + nv + 4, dt=dt, g=g)[:, 4:]
    wq, wk, table = 1 + rnd(nq, g=g, scale=0.2), 1 + rnd(nk, g=g, scale=0.2), M.rope_table(40, rot, 50.0)
    pos, slots = torch.arange(rows).int() % 40, torch.arange(rows).int() - 1
    kc, vc = torch.zeros(-(-rows // 4), 4, nk, dtype=dt), torch.zeros(-(-rows // 4), 4, nv, dtype=dt)
    kd, vd = kc.to(DEV), vc.to(DEV)
    want = R.attn_prep(qkv, nq, nk, wq, wk, 1e-5, table, rot, hd, pos, slots, kc, vc)
    wide = torch.cat([qkv[:, :4], qkv], 1).to(DEV)[:, 4:]
    got = M.attn_prep(wide, nq, nk, wq.to(DEV), wk.to(DEV), 1e-5, table.to(DEV), rot, hd, pos.to(DEV), slots.to(DEV), kd, vd)
    torch.testing.assert_close(got.cpu(), want, rtol=2e-5, atol=2e-5)
    torch.testing.assert_close(kd.cpu().float(), kc.float(), **tol(dt))
    torch.testing.assert_close(vd.cpu().float(), vc.float(), **tol(dt))
