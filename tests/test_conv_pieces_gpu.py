"""Short convolution in 16-byte pieces of channels: edges of its row tiles (8) and of the history it leaves."""
import pytest
import torch

from fasttalk_llm_microservice_amd.ops import mixers as M
from fasttalk_llm_microservice_amd.ops import mixers_ref as R
from test_mixer_kernels_gpu import DEV, DTYPES, make_seg, rnd, to_dev, tol

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("taps", [2, 3, 4])
@pytest.mark.parametrize("lens", [[1, 1, 1, 1], [8, 2, 3, 7], [9, 1, 16, 8], [40, 17, 3, 1]])
@pytest.mark.parametrize("c,left", [(8, 8), (1032, 16), (1032, 3)])    # left 3: not on 16 bytes, the general kernel
def test_conv_pieces(dt, taps, lens, c, left):
    g = torch.Generator().manual_seed(c + taps)
    seg, _ = make_seg(lens, [5, 0, 1, 0], [2, 0, 3, 1] if lens[0] != 8 else [2, 0, -1, 1])
    wide = rnd(sum(lens), left + c + 8 - left % 8, dt=dt, g=g)
    w, b, hist = rnd(c, taps, g=g), rnd(c, g=g), rnd(4, taps - 1, c, g=g)
    for bias in (None, b):
        h1, h2 = hist.clone(), hist.clone().to(DEV)
        y1 = R.short_conv_silu(wide[:, left:left + c], w, h1, seg, bias)
        y2 = M.short_conv_silu(wide.to(DEV)[:, left:left + c], w.to(DEV), h2, to_dev(seg),
                               None if bias is None else bias.to(DEV))
        torch.testing.assert_close(y2.cpu().float(), y1.float(), **tol(dt))
        torch.testing.assert_close(h2.cpu(), h1, rtol=0, atol=0)


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("taps", [2, 3, 4])
@pytest.mark.parametrize("lens,c", [([400, 9, 8, 1], 1032), ([8, 2, 3, 7], 39088), ([41, 16, 17, 33], 7688)])
def test_conv_pieces_of_many_rows(dt, taps, lens, c):
    """Work enough for the pieces kernel: part-filled row tiles, histories left by both kernels, padding."""
    test_conv_pieces(dt, taps, lens, c, 8)
