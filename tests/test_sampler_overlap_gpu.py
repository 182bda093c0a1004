"""Draws whose target lies where two threads' ranges of the fp32 prefix sums overlap (csrc/kernels/sampling.hip
samp_draw_kernel): the lower thread's id is the candidate, in every workgroup that draws the row, whatever their timing."""
import numpy as np
import pytest
import torch

from fasttalk_llm_microservice_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
M64 = (1 << 64) - 1


def mix(x):
    x = (x + 0x9E3779B97F4A7C15) & M64
    x = ((x ^ (x >> 30)) * 0xBF58476D1CE4E5B9) & M64
    x = ((x ^ (x >> 27)) * 0x94D049BB133111EB) & M64
    return x ^ (x >> 31)


def unmix(y):
    """x with mix(x) = y"""
    def shift(v, s):
        x = v
        for _ in range(64 // s + 1):
            x = v ^ (x >> s)
        return x
    y = shift(y, 31)
    y = shift((y * pow(0x94D049BB133111EB, -1, 1 << 64)) & M64, 27)
    y = shift((y * pow(0xBF58476D1CE4E5B9, -1, 1 << 64)) & M64, 30)
    return (y - 0x9E3779B97F4A7C15) & M64


def uniforms(s0):
    return [((mix((s0 + r * 0xD1B54A32D192ED03) & M64) >> 40) + 0.5) * 2.0 ** -24 for r in range(4)]


def seed_for(first, accept):
    """A seed whose first uniform at step 0 has these 24 bits and whose second one is accepted."""
    for low in range(10000):
        s0 = unmix(first << 40 | low)
        if accept(uniforms(s0)[1]):
            seed = unmix(s0) ^ 0x632BE59BD9B4E019
            return seed - (1 << 64) if seed >> 63 else seed
    raise AssertionError("no seed")


@pytest.mark.parametrize("rows", [1, 8, 9, 40])
@pytest.mark.parametrize("top_p,threads", [(1.0, 0), (0.9, 256)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_lower_thread_wins(rows, top_p, threads, dtype):
    # masses 1/2 in thread 0, 2^-24 in thread 63 (where there are some, in its second eight ids), 1 in thread 64: thread 63's range is [1/2, 1/2 +
    # 2^-24), and thread 64's begins at (1/2 + 2^-24 + 1) - 1, in fp32 1/2.  A temperature of log2(e) makes them exact.
    f = np.float32
    low, high = 8 * (63 + threads) + 7, 8 * 64
    before = f(f(0.5) + f(2.0 ** -24))
    assert before > 0.5 and f(f(before + f(1.0)) - f(1.0)) == 0.5
    # the first target: u * 1.5 = 1/2
    u = (5592405 + 0.5) * 2.0 ** -24
    assert f(f(u) * f(1.5)) == 0.5
    vocab = 131072                 # 4096 ids a slice: eight a thread of 1024, twice eight a thread of a candidate's 256
    logits = torch.full((rows, vocab), float("-inf"), dtype=dtype, device=DEV)
    logits[:, 0], logits[:, low], logits[:, high] = -1.0, -24.0, 0.0
    seed = seed_for(5592405, lambda v: v < 0.3)          # (the second one is in thread 0's range)
    full = lambda v, dt: torch.full((rows,), v, dtype=dt, device=DEV)      # noqa: E731
    # at top-p 0.9 everything is more likely than the first candidate, which is refused; the second, id 0, is taken
    want = low if top_p == 1.0 else 0
    for _ in range(20):
        got = ops.sample(logits, full(1.4426950408889634, torch.float32), full(top_p, torch.float32), full(0, torch.int32),
                         full(seed, torch.int64), full(0, torch.int32))
        assert got.tolist() == [want] * rows
