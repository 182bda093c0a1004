"""A row's sampled token does not depend on how many rows are sampled with it: the draw and the above-masses in one
launch for few rows, in two for more (csrc/kernels/sampling.hip kAboveRows), top-k rows in the same launch."""
import pytest
import torch

from fasttalk_llm_microservice_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


# one slice with ids, slices of uneven length, the largest vocabulary
@pytest.mark.parametrize("vocab", [8, 4104, 131072])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_rows_alone_and_together(vocab, dtype):
    g = torch.Generator().manual_seed(vocab)
    n = 12
    logits = (3 * torch.randn(n, vocab, generator=g)).to(dtype).to(DEV)
    logits[5, : vocab - 3] = float("-inf")
    logits[6] = float("-inf")
    temp = torch.tensor([0.7, 0.0, 1.0, 0.8, 0.9, 0.7, 0.7, 1.3, 0.7, 0.8, 0.6, 0.7], device=DEV)
    top_p = torch.tensor([0.9, 0.9, 1.0, 0.95, 0.5, 0.9, 0.9, 0.05, 0.9, 1.0, 0.9, 0.9], device=DEV)
    top_k = torch.tensor([0, 0, 0, 40, 5, 0, 0, 0, 64, 1, 0, 100], dtype=torch.int32, device=DEV)
    seeds = torch.arange(n, device=DEV) * 7919
    mask = torch.full((n, (vocab + 31) // 32), -1, dtype=torch.int32, device=DEV)
    mask[2, 0] = 5
    for step in range(6):
        steps = torch.full((n,), step, dtype=torch.int32, device=DEV)
        args = (logits, temp, top_p, top_k, seeds, steps)
        together = ops.sample(*args, mask=mask)
        for k in (1, 4, 8, 9):
            parts = [ops.sample(*(t[i:i + k].contiguous() for t in args), mask=mask[i:i + k].contiguous())
                     for i in range(0, n, k)]
            assert torch.equal(torch.cat(parts), together)
