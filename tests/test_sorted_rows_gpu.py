"""Norm steps that sum a mixture's sorted results as they read them (rows.hip SortedRows) against 64 bits: widths of every number
of register chunks and part-filled ones, more choices than are read at once, shared experts with and without a gate."""
import pytest
import torch

from fasttalk_llm_microservice_amd.ops import mixers as M
from test_mixer_kernels_gpu import DEV, rnd

pytestmark = pytest.mark.gpu
EPS = 1e-5


def rms(x, w):
    return x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * w.double()


def layer(x, w, b):
    x = x - x.mean(-1, keepdim=True)
    return x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * w.double() + b.double()


@pytest.mark.parametrize("shared", ["none", "plain", "gated"])
@pytest.mark.parametrize("top", [1, 4, 5])
@pytest.mark.parametrize("width", [1032, 2048, 2056, 4104, 8200])
def test_norm_steps(width, top, shared):
    g = torch.Generator().manual_seed(width + top)
    rows, bf = 5, torch.bfloat16
    d, h, sh, gw = (rnd(*s, dt=bf, g=g) for s in ((rows * top, width), (rows, width), (rows, width), (width,)))
    gw = (gw.float() * width ** -0.5).to(bf)
    place, wts = torch.randperm(rows * top, generator=g).int(), torch.rand(rows, top, generator=g)
    x, w1, w2, w3, w4 = rnd(rows, width, g=g), *(rnd(width, g=g) for _ in range(4))
    y = (d.double()[place.long()].view(rows, top, width) * wts.double()[:, :, None]).sum(1)
    if shared != "none":
        y += sh.double() * (torch.sigmoid(h.double() @ gw.double())[:, None] if shared == "gated" else 1.0)
    c = lambda t: t.to(DEV)                            # noqa: E731
    parts = M.SortedParts(c(d), c(place), c(wts), None if shared == "none" else c(sh), c(h), c(gw) if shared == "gated" else None)

    def close(got, want):
        """fp32: sums of a few products of order one and means of up to 8200, a few tens of 2^-23; bf16 half a unit more."""
        tol = 2e-5 if got.dtype == torch.float32 else 2.0 ** -8
        torch.testing.assert_close(got.cpu().double(), want, rtol=tol, atol=2e-5)

    for wb in (None, w1):
        x1 = x.double() + (y if wb is None else rms(y, wb))
        xd = c(x)
        out, cast = M.add_rms_norm_rows(xd, parts, None if wb is None else c(wb), EPS, None, c(w2), bf, True)
        close(xd, x1), close(cast, x1), close(out, rms(x1, w2))
    x1 = x.double() + layer(y, w1, w2)
    for nxt in (None, (w3, w4)):
        xd = c(x)
        got = M.add_layer_norm_rows(xd, parts, c(w1), c(w2), EPS, bf, nxt and tuple(map(c, nxt)))
        close(xd, x1), close(got, x1 if nxt is None else layer(x1, *nxt))


@pytest.mark.parametrize("top", [1, 2, 5, 9])
@pytest.mark.parametrize("width", [1032, 2056, 4104, 8200])
def test_unsorted_parts(width, top):
    """Mixtures' results in fp32 and a product's parts (rows.hip ExpertRows, AnyRows): fewer and more than are read at once."""
    g = torch.Generator().manual_seed(width + top)
    rows, bf = 5, torch.bfloat16
    d, d2, sh = rnd(rows * top, width, g=g), rnd(rows * top, width, g=g), rnd(rows, width, g=g)
    gate, wts = rnd(rows, g=g), torch.rand(rows, top, generator=g)
    x, w1, w2 = (rnd(*s, g=g) for s in ((rows, width), (width,), (width,)))
    c = lambda t: t.to(DEV)                            # noqa: E731
    sums = lambda t: t.double().view(rows, top, width).sum(1)      # noqa: E731
    y = (d.double().view(rows, top, width) * wts.double()[:, :, None]).sum(1) + sh.double() * torch.sigmoid(gate.double())[:, None]

    def close(got, want):
        """As above; sums of up to nine terms of order one."""
        tol = 4e-5 if got.dtype == torch.float32 else 2.0 ** -8
        torch.testing.assert_close(got.cpu().double(), want, rtol=tol, atol=4e-5)

    for parts, rows_y in ((M.ExpertParts(c(d), c(wts), c(sh), c(gate)), y), (M.ExpertParts(c(d), None, None, None), sums(d))):
        xd = c(x)
        out, _ = M.add_rms_norm_rows(xd, parts, c(w1), EPS, None, c(w2), bf)
        x1 = x.double() + rms(rows_y, w1)
        close(xd, x1), close(out, rms(x1, w2))
    if top > 1:
        a, b = M.ExpertParts(c(d), None, None, None), M.ExpertParts(c(d2), None, None, None)
        xd = c(x)
        out = M.add_scaled_rms_norm_rows(xd, a, b, 0.5, c(w2), EPS, bf)
        x1 = x.double() + 0.5 * (sums(d) + sums(d2))
        close(xd, x1), close(out, rms(x1, w2))
        close(M.dual_rms_mean(a, b, c(w1), c(w2), EPS, 0.5, rows), 0.5 * (rms(sums(d), w1) + rms(sums(d2), w2)))
