"""A decode step's inputs written by the runtime (csrc/runtime/step_inputs.cpp) against the plain loop over the sequences,
and an eager step's arrays through the uploader's one image."""
import numpy as np
import pytest
import torch

from fasttalk_llm_microservice_amd.engine import runner as R
from fasttalk_llm_microservice_amd.engine.sampling_params import SamplingParams
from fasttalk_llm_microservice_amd.engine.sequence import Sequence
from fasttalk_llm_microservice_amd.runtime import rt


def sequences(n, seed=0):
    g = np.random.default_rng(seed)
    out = []
    for i in range(n):
        toks = g.integers(0, 1 << 20, size=int(g.integers(1, 200))).tolist()
        s = Sequence(f"s{i}", toks, SamplingParams(temperature=0.1 * i, top_p=1.0 - 0.01 * i, top_k=i, seed=(1 << 62) - i))
        for t in range(i % 4):
            s.append(7 + t)
        s.inflight, s.preemptions, s.state_slot = i % 3, i % 2, 3 * i
        s.block_ids = g.permutation(1 << 16)[:(s.n_tokens + s.inflight + 15) // 16 + i % 2].tolist()
        out.append(s)
    return out


@pytest.mark.parametrize("n,nb,mb", [(1, 1, 8), (3, 8, 8), (8, 8, 8), (0, 2, 4)])
@pytest.mark.parametrize("stateful", [False, True])
def test_decode_inputs(n, nb, mb, stateful):
    cols, bs = 40, 16
    seqs = sequences(n)
    st = R._Staging(mb, cols, pin=False, gpu=False)
    st.h_in.fill_(-9)
    keep = st.h_in.clone()
    most = rt().fill_decode(seqs, bs, mb, nb, stateful, st.hs, st.hbt, st.hf, st.hseed)
    assert most == max([1] + [len(s.block_ids) for s in seqs])
    want = R._Staging(mb, cols, pin=False, gpu=False)
    want.h_in.copy_(keep)
    hs = want.hs.reshape(8, mb)
    for i, s in enumerate(seqs):
        p = s.n_tokens - 1 + s.inflight
        hs[:6, i] = (s.last_token, p, s.block_ids[p // bs] * bs + p % bs, p + 1, s.params.top_k,
                     s.num_output + s.inflight + 131 * s.preemptions)
        want.hbt[i, :len(s.block_ids)] = s.block_ids
        want.hf[i], want.hf[mb + i], want.hseed[i] = s.params.temperature, s.params.top_p, s.params.seed
        if stateful:
            hs[6, i] = s.state_slot
    for i in range(n, nb):
        hs[:6, i] = (0, 0, -1, 0, 0, 0)
        want.hbt[i, 0] = 0
        want.hf[i], want.hf[mb + i] = 0.0, 1.0
        if stateful:
            hs[6, i] = -1
    assert torch.equal(st.h_in, want.h_in)


def test_decode_inputs_are_refused():
    st = R._Staging(4, 4, pin=False, gpu=False)
    args = (16, 4, 2, False, st.hs, st.hbt, st.hf, st.hseed)
    s = sequences(1)[0]
    s.block_ids = list(range(5))                 # a table wider than the image
    with pytest.raises(IndexError):
        rt().fill_decode([s], *args)
    s.block_ids = []                             # a position without a page
    with pytest.raises(IndexError):
        rt().fill_decode([s], *args)
    with pytest.raises(ValueError):
        rt().fill_decode(sequences(3), *args)    # more rows than the bucket
    with pytest.raises(ValueError):
        rt().fill_decode([], 16, 4, 5, False, st.hs, st.hbt, st.hf, st.hseed)


def test_uploaded_arrays():
    g = np.random.default_rng(1)
    up = R._Uploader(torch.device("cpu"), pin=False)
    for size in (0, 1, 15, 16, 1000, 3):
        arrays = [g.integers(-9, 9, size).astype(np.int32), g.normal(size=size).astype(np.float32),
                  g.integers(-(1 << 60), 1 << 60, size), g.integers(0, 9, (size, 3)).astype(np.int32),
                  g.integers(0, 9, (2, size)).astype(np.int32)[:, ::-1], g.normal(size=2)]
        for a, v in zip(arrays, up(arrays)):
            assert tuple(v.shape) == a.shape and np.array_equal(v.numpy(), a)
    assert [v.numel() for v in up([])] == []
    with pytest.raises(TypeError):
        up([np.zeros(4, np.int16)])
