"""A step's first rows and the norm that reads them in one launch (csrc/mixers/rows.hip embed_norm_kernel): edges of the register
chunks, ids out of range, padding rows, pairs across segments and steps, positions; and rows that are no whole fours."""
import pytest
import torch

from fasttalk_llm_microservice_amd.ops import mixers as M
from fasttalk_llm_microservice_amd.ops import mixers_ref as R
from test_mixer_kernels_gpu import DEV, DTYPES, rnd, tol

pytestmark = pytest.mark.gpu


def segments(dev):
    """Segments of one, three and two rows, the last in no slot, and two rows of padding; the second starts its sequence."""
    t = lambda *v: torch.tensor(v, dtype=torch.int32, device=dev)        # noqa: E731
    return M.Segments(start=t(0, 1, 4, 6), pos0=t(7, 0, 5), slot=t(2, 0, -1), kv_len=t(8, 3, 7), block_tables=None, num=3, max_rows=3)


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("width", [4, 1028, 2048, 2052, 8192, 16384, 50, 16388])
@pytest.mark.parametrize("form", ["plain", "pair", "positions"])
def test_first_rows(dt, width, form):
    g = torch.Generator().manual_seed(width)
    table, pair = rnd(40, width, dt=dt, g=g), rnd(12, width, dt=dt, g=g)
    ids = torch.tensor([3, 39, 40, 0, 7, -1, 5, 38], dtype=torch.int32)
    pos = torch.tensor([7, 0, 1, 2, 3299, 131071, 0, 0], dtype=torch.int32)
    w, b = 1 + rnd(width, g=g, scale=0.2), rnd(width, g=g, scale=0.2)
    freqs = M.sinusoid_freqs(width) if form == "positions" else None
    known = ids.clamp(0, 39) * (ids < 40)
    for norm in ((None, None), (w, None), (w, b)):
        if width > 16384 and norm[1] is None and norm[0] is not None:
            continue                                                       # (RMS norms go no further)
        last = [torch.tensor([11, 12, 13, 14], dtype=torch.int32, device=d) for d in ("cpu", DEV)]
        got, want = [], []
        for d, put, last_tok in (("cpu", want, last[0]), (DEV, got, last[1])):
            seg = segments(d)
            mv = lambda t: None if t is None else t.to(d)                  # noqa: E731
            at = (mv(pair), 7, 5, 11, seg, last_tok) if form == "pair" else None
            put += M.embed_norm_rows(mv(known if d == "cpu" or form == "pair" else ids), mv(table), 2.5, 1e-5, dt, *map(mv, norm), mv(pos),
                                     mv(freqs), at)
        close = tol(torch.float32)
        if norm[1] is None:
            torch.testing.assert_close(got[0].cpu(), want[0], **close)
        if norm[0] is None:
            assert got[1] is None
        else:
            torch.testing.assert_close(got[1].cpu().float(), want[1].float(), **tol(dt))
            if norm[1] is not None:
                torch.testing.assert_close(got[0].cpu(), want[0], **close)
        if form == "pair":
            assert last[1].tolist() == last[0].tolist() == [0, 12, 3, 14]
