"""Products of more than a few rows with long sums, k cut into parts that the norm step adds (csrc/mixers/tile_gemm.hip tile_parts)."""
import pytest
import torch

from fasttalk_llm_microservice_amd.ops import mixers as M
from test_few_rows_gpu import rnd

pytestmark = pytest.mark.gpu
DEV = "cuda"


# edges of row and column tiles, parts of unlike lengths (k = 65, 67 and 130 stages), rows of a wider array, each form
@pytest.mark.parametrize("rows", [65, 128, 193, 257, 300, 577, 769, 1024])
@pytest.mark.parametrize("n,k", [(2048, 4160), (1288, 8320), (3076, 4288), (64, 4096)])
def test_parts(rows, n, k):
    g = torch.Generator().manual_seed(rows + n + k)
    N = M.native_mixers()
    parts = N.tile_parts(rows, n, k)
    if parts == 1:
        with pytest.raises(RuntimeError):
            N.tile_gemm_parts(torch.empty(rows, n, device=DEV), rnd(g, rows, k), rnd(g, n, k), None)
        return
    x, w, b = rnd(g, rows, k + 24)[:, 16:16 + k], rnd(g, n, k, scale=k ** -0.5), rnd(g, n)
    for bias in (None, b):
        d = torch.full((rows * parts, n), float("nan"), device=DEV)
        N.tile_gemm_parts(d, x, w, bias)
        share = -(-(k // 64) // parts) * 64
        for p in range(parts):
            at = slice(p * share, min(k, (p + 1) * share))
            want = x[:, at].double() @ w[:, at].double().t() + (bias.double() if bias is not None and p == 0 else 0)
            # fp32 sums of k terms of order 1 / sqrt(k)
            assert float((d.view(rows, parts, n)[:, p].double() - want).abs().max()) <= 2.0 ** -20 * k ** 0.5


def test_which_products():
    """Rows of bf16 up to 1024, long sums of few columns; the norm step adds the parts as it adds the product's rows."""
    w = torch.randn(2048, 8192, device=DEV).to(torch.bfloat16)
    forms = set()
    for rows in (65, 256, 300, 777, 1024):
        x = torch.randn(rows, 8192, device=DEV).to(torch.bfloat16)
        y = M.linear_out(x, w, True)
        assert isinstance(y, M.ExpertParts) and y.d.shape == (rows * M.native_mixers().tile_parts(rows, 2048, 8192), 2048)
        forms.add(y.d.shape[0] // rows)
        res, nw = torch.randn(rows, 2048, device=DEV), torch.ones(2048, device=DEV)
        r2 = res.clone()
        h, _ = M.add_rms_norm_rows(res, y, nw, 1e-6, next_w=nw, out_dtype=torch.bfloat16)
        h2, _ = M.add_rms_norm_rows(r2, x.float() @ w.float().t(), nw, 1e-6, next_w=nw, out_dtype=torch.bfloat16)
        torch.testing.assert_close(res, r2, rtol=1e-4, atol=1e-4)                # (both fp32 sums of 8192 terms of order 1)
        torch.testing.assert_close(h.float(), h2.float(), rtol=2.0 ** -7, atol=1e-4)      # (one rounding to bf16 either way)
    assert len(forms) > 1 and all(M.native_mixers().tile_parts(r, 2048, 4096) in (2, 4) for r in range(65, 257))
    x = torch.ones(1025, 8192, device=DEV, dtype=torch.bfloat16)
    assert all(isinstance(M.linear_out(*a), torch.Tensor) for a in ((x, w, True), (x[:300], w, False), (x[:300, :4032], w[:, :4032].contiguous(), True),
                                                                    (x[:300].float(), w.float(), True)))


@pytest.mark.parametrize("rows,width,p1,p2", [(1, 2048, 2, 4), (3, 1032, 4, 3), (130, 4096, 3, 2), (5, 4352, 1, 4), (2, 2048, 4, 1)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_norms_of_two_rows(rows, width, p1, p2, dt):
    """The scaled add of two sublayers' rows and the mean of two norms, of parts, of rows beside them, and of both."""
    g = torch.Generator().manual_seed(rows + width)
    f32 = lambda *s: torch.randn(*s, generator=g).to(DEV)      # noqa: E731
    a, b = ((f32(rows * p, width) if p > 1 else rnd(g, rows, width).to(dt)) for p in (p1, p2))
    made = [M.ExpertParts(y, None, None, None) if p > 1 else y for y, p in ((a, p1), (b, p2))]
    ya, yb = (y.view(rows, p, width).double().sum(1).float() for y, p in ((a, p1), (b, p2)))
    wa, wb, x = f32(width), f32(width), f32(rows, width)
    torch.testing.assert_close(M.dual_rms_mean(*made, wa, wb, 1e-5, 0.5, rows), M.dual_rms_mean(ya, yb, wa, wb, 1e-5, 0.5), rtol=1e-5, atol=1e-5)
    x1, x2 = x.clone(), x.clone()
    got, want = (M.add_scaled_rms_norm_rows(r, *y, 0.4, wa, 1e-5, dt) for r, y in ((x1, made), (x2, (ya, yb))))
    torch.testing.assert_close(x1, x2, rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(got.float(), want.float(), rtol=2.0 ** -7 if dt == torch.bfloat16 else 1e-5, atol=1e-5)
    for bad in (M.ExpertParts(f32(rows * 2, width), f32(rows, 2), None, None), M.ExpertParts(f32(rows * 2, width), None, f32(rows, width), None)):
        with pytest.raises(ValueError):
            M.add_scaled_rms_norm_rows(x1, bad, None, 0.4, wa, 1e-5, dt)
