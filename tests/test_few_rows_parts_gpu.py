"""Products of few rows with k cut into parts (csrc/mixers/few_rows.hip few_rows_parts) and the norm steps that add the parts:
edges of row blocks, of column tiles and of the shares of k, each form that the sizes choose."""
import pytest
import torch

from fasttalk_llm_microservice_amd.ops import mixers as M
from test_few_rows_gpu import rnd

pytestmark = pytest.mark.gpu
DEV = "cuda"


# two and four parts by the rule, and numbers of parts whose last one is short or that have no whole steps
@pytest.mark.parametrize("rows", [1, 16, 17, 33, 64])
@pytest.mark.parametrize("n,k,parts", [(1032, 1024, 0), (2048, 2048, 0), (1288, 4104, 0), (2048, 8192, 0), (2056, 2056, 0), (3584, 4096, 0),
                                       (20, 72, 2), (36, 328, 3), (24, 2000, 8)])
def test_parts(rows, n, k, parts):
    g = torch.Generator().manual_seed(rows + n + k)
    wide = rnd(g, rows, k + 24)
    x, w, b = wide[:, 16:16 + k], rnd(g, n, k, scale=k ** -0.5), rnd(g, n)
    parts = parts or M.native_mixers().few_rows_parts(n, k)
    assert parts > 1
    for bias in (None, b):
        d = torch.empty(rows * parts, n, device=DEV)
        M.native_mixers().few_rows_gemm_parts(d, x, w, bias)
        want = x.double() @ w.double().t() + (0 if bias is None else bias.double())
        # fp32 sums of k terms of order 1 / sqrt(k), and of the parts
        assert float((d.view(rows, parts, n).double().sum(1) - want).abs().max()) <= 2.0 ** -20 * k ** 0.5
        share = -(-(-(-k // 64)) // parts) * 64
        first = x[:, :share].double() @ w[:, :share].double().t() + (0 if bias is None else bias.double())
        assert float((d.view(rows, parts, n)[:, 0].double() - first).abs().max()) <= 2.0 ** -20 * k ** 0.5


def test_which_products():
    """Rows of bf16 whose product a norm step reads; not beyond 64 rows, of many columns or of short sums, nor in fp32."""
    w = torch.zeros(2048, 2048, dtype=torch.bfloat16, device=DEV)
    x = torch.ones(64, 2048, dtype=torch.bfloat16, device=DEV)
    y = M.linear_out(x, w, True)
    assert isinstance(y, M.ExpertParts) and y.d.shape == (128, 2048)
    assert isinstance(M.linear_out(x, w, False), torch.Tensor)
    assert isinstance(M.linear_out(torch.ones(65, 2048, dtype=torch.bfloat16, device=DEV), w, True), torch.Tensor)
    assert isinstance(M.linear_out(x.float(), w.float(), True), torch.Tensor)
    assert [M.native_mixers().few_rows_parts(*s) for s in ((4096, 4096), (2048, 1016), (3072, 1024), (2048, 1024), (3072, 2048), (2048, 4096))] \
        == [1, 1, 1, 2, 4, 4]
    with pytest.raises(RuntimeError):                                            # (parts without any k)
        M.native_mixers().few_rows_gemm_parts(torch.empty(64 * 40, 2048, device=DEV), x, w, None)


@pytest.mark.parametrize("rows,width,parts", [(1, 2048, 2), (3, 1280, 4), (17, 4096, 2), (5, 4352, 4)])
@pytest.mark.parametrize("layer", [False, True])
def test_norm_steps_add_the_parts(rows, width, parts, layer):
    """As the same steps of the rows already added: the sums differ in the last place at most."""
    g = torch.Generator().manual_seed(rows + width)
    f32 = lambda *s: torch.randn(*s, generator=g).to(DEV)      # noqa: E731
    d, x, wb, w, b = f32(rows * parts, width), f32(rows, width), f32(width), f32(width), f32(width)
    y = d.view(rows, parts, width).double().sum(1).float()
    made = M.ExpertParts(d, None, None, None)
    close = dict(rtol=2.0 ** -7, atol=2e-5)                    # (bf16 results: one rounding either way)
    x1, x2 = x.clone(), x.clone()
    if layer:
        got, want = (M.add_layer_norm_rows(a, p, w, b, 1e-5, torch.bfloat16) for a, p in ((x1, made), (x2, y)))
    else:
        got, want = (M.add_rms_norm_rows(a, p, wb, 1e-5, None, w, torch.bfloat16)[0] for a, p in ((x1, made), (x2, y)))
    torch.testing.assert_close(x1, x2, rtol=1e-5, atol=2e-5)
    torch.testing.assert_close(got.float(), want.float(), **close)
    if width % 256 == 0:
        router = f32(24, width) * width ** -0.5
        args = (None if layer else wb, w, b if layer else None)
        x1, x2 = x.clone(), x.clone()
        assert M.norm_route_fits(x1, made, *args, router)
        (h1, (i1, w1)), (h2, (i2, w2)) = (M.norm_route(a, p, *args, 1e-5, router, None, 4, "top_logits") for a, p in ((x1, made), (x2, y)))
        torch.testing.assert_close(x1, x2, rtol=1e-5, atol=2e-5)
        torch.testing.assert_close(h1.float(), h2.float(), **close)
        z = h2.double() @ router.double().t()      # a choice may differ between experts as good as level to h's rounding
        assert bool(((i1 == i2) | ((z.gather(1, i1.long()) - z.gather(1, i2.long())).abs() < 0.05)).all())
    assert not M.norm_route_fits(x, M.ExpertParts(d, torch.ones(rows, parts, device=DEV), None, None), wb, w, None, wb)
