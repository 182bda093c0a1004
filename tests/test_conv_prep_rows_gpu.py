"""Convolution, norm and rotation of q, k and v (window_attn.hip) and the delta rule's inputs (head_state.hip) at the step sizes
where a wave takes another number of rows, with segments that begin and end inside a wave's rows, against the PyTorch ops."""
import pytest
import torch

from fasttalk_llm_microservice_amd.ops import mixers as M
from test_kerarax_gpu import _segments

pytestmark = pytest.mark.gpu


def both(f):
    return [[t.double().cpu() for t in f(dev)] for dev in ("cuda", "cpu")]


def move(seg, dev):
    return M.Segments(**{**seg.__dict__, **{k: getattr(seg, k).to(dev) for k in ("start", "pos0", "slot", "kv_len", "block_tables")}})


@pytest.mark.parametrize("heads,total", [(3, 255), (3, 256), (3, 639), (3, 640), (28, 272), (28, 274), (62, 255), (62, 256), (62, 504),
                                         (62, 505), (3, 1639), (3, 1280)])
@pytest.mark.parametrize("dk,interleaved", [(24, False), (128, True), (200, False)])
def test_rows_of_a_wave(heads, total, dk, interleaved):
    g = torch.Generator().manual_seed(total + dk)
    rows = [1, 1, 6, 30]
    rows += [total - sum(rows) - 1, 1]
    pos0, slots = [17, 0, 3, 0, 40, 9], [2, 0, 3, 1, 5, 4]
    seg, slot_map, nb = _segments("cuda", rows, pos0, slots, 16, pad=2)
    H, G, taps = heads, 1, 4
    nq, nk, nv = H * dk, G * dk, G * dk
    c = nq + nk + nv
    qkv = (0.7 * torch.randn(total, c, generator=g)).bfloat16()
    conv_w, hist0 = 0.5 * torch.randn(c, taps, generator=g), torch.randn(6, taps - 1, c, generator=g)
    wq, wk = 1 + 0.2 * torch.randn(dk, generator=g), 1 + 0.2 * torch.randn(dk, generator=g)
    rot = dk // 8 * 4
    table = M.rope_table(total + 64, rot, 1e4, device="cpu")

    def attn(dev):
        hist = hist0.clone().to(dev)
        kc, vc = (torch.zeros(nb, 16, n, dtype=torch.bfloat16, device=dev) for n in (nk, nv))
        q = M.conv_attn_prep(qkv.to(dev), nq, nk, conv_w.to(dev), hist, move(seg, dev), wq.to(dev), wk.to(dev), 1e-5, dk,
                             slot_map.to(dev), kc, vc, table.to(dev), rot, interleaved)
        return q, hist, kc, vc

    a, b = torch.randn(total, H, generator=g).bfloat16(), torch.randn(total, H, generator=g).bfloat16()
    a_log, dt = torch.randn(H, generator=g), torch.randn(H, generator=g)
    x = (0.7 * torch.randn(total, 2 * G * dk + H * dk, generator=g)).bfloat16()

    def delta(dev):
        hist = hist0.clone().to(dev)
        return (*M.conv_delta_prep(x.to(dev), a.to(dev), b.to(dev), conv_w.to(dev), hist, a_log.to(dev), dt.to(dev),
                                   move(seg, dev), H, G, dk, dk), hist)

    for f in (attn, delta):
        for n, (got, want) in enumerate(zip(*both(f))):
            # fp32 sums of four products and of dk squares; the caches (attn's last two) are rounded to bf16
            tol = 2 ** -7 if f is attn and n >= 2 else 2e-5
            torch.testing.assert_close(got, want, rtol=tol, atol=tol, msg=lambda m, n=n: f"{f.__name__} {n}: {m}")
