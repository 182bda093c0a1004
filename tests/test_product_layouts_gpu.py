"""Operands of products that the kernels do not take, the library's product does: rows that overlap in memory (a row that is repeated
by a stride of 0, windows of one row), weights of one row, a bias that is broadcast, a gated form's matrices with a row more."""
import pytest
import torch

from fasttalk_llm_microservice_amd.ops import mixers as M

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("rows", [3, 100, 700, 1500])
@pytest.mark.parametrize("stride", [0, 8, 64])
@pytest.mark.parametrize("act", [None, "silu", "relu_sq"])
def test_overlapping_rows(rows, stride, act):
    g = torch.Generator(device=DEV).manual_seed(rows)
    flat = torch.randn(rows * 64 + 512, generator=g, device=DEV).bfloat16()
    x = flat.as_strided((rows, 512), (stride, 1))
    w = (torch.randn(512, 512, generator=g, device=DEV) / 512 ** 0.5).bfloat16()
    got = M.linear(x, w) if act is None else M.linear_act(x, w, act)
    want = M.linear(x.contiguous(), w) if act is None else M.linear_act(x.contiguous(), w, act)
    # bf16 sums of 512 terms of order 1, rounded before the activation or behind it
    torch.testing.assert_close(got.float(), want.float(), rtol=2.0 ** -6, atol=2.0 ** -7)


@pytest.mark.parametrize("rows", [65, 100])
def test_one_output_column(rows):
    """A weight of one dimension: a product per row, as torch's linear gives it."""
    g = torch.Generator(device=DEV).manual_seed(1)
    x, w = torch.randn(rows, 512, generator=g, device=DEV).bfloat16(), torch.randn(512, generator=g, device=DEV).bfloat16()
    assert torch.equal(M.linear(x, w), torch.nn.functional.linear(x, w))


@pytest.mark.parametrize("shape", [(1,), (1, 512), (100, 512)])
def test_bias_of_another_shape(shape):
    g = torch.Generator(device=DEV).manual_seed(2)
    x, w, b = (torch.randn(*s, generator=g, device=DEV).bfloat16() for s in ((100, 512), (512, 512), shape))
    assert torch.equal(M.linear(x, w, b), torch.nn.functional.linear(x, w, b))


@pytest.mark.parametrize("act", ["clamp_glu"])
def test_matrices_with_one_row_more(act):
    g = torch.Generator(device=DEV).manual_seed(3)
    x, w = (torch.randn(*s, generator=g, device=DEV).bfloat16() for s in ((100, 512), (1025, 512)))
    got, want = M.linear_act(x, w, act, 7.0), M.clamp_swiglu(torch.nn.functional.linear(x, w), 7.0)
    assert torch.equal(got, want)


@pytest.mark.parametrize("rows,n,k,act,kept", [(65, 256, 2048, None, False), (128, 2048, 8192, None, False), (128, 2048, 2048, None, True),
                                               (200, 4096, 2048, "silu", True)])
def test_captured_steps(rows, n, k, act, kept):
    """A step that is replayed has no host time to save: where the tiles are behind for that, the vendor's product is captured."""
    g = torch.Generator(device=DEV).manual_seed(4)
    x, w = torch.randn(rows, k, generator=g, device=DEV).bfloat16(), (torch.randn(n, k, generator=g, device=DEV) * k ** -0.5).bfloat16()
    run = lambda: M.linear(x, w) if act is None else M.linear_act(x, w, act)      # noqa: E731
    eager = run().clone()
    assert M._tile_gemm(x, w, None, act) is not None
    with M.replayed_step():
        assert (M._tile_gemm(x, w, None, act) is not None) == kept
        warm = run()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph), M.replayed_step():
        y = run()
    assert M._tile_gemm(x, w, None, act) is not None
    torch.testing.assert_close(warm.float(), eager.float(), rtol=2.0 ** -6, atol=2.0 ** -7)      # bf16 sums in another order
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, warm)
        run()
