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


def mixed_reference(dseqs, pseqs, ntoks, starts, bs, segments):
    """The same rows as a plain loop."""
    rows, segs = [], []
    for s in dseqs:
        p = s.n_tokens - 1 + s.inflight
        segs.append((s, p, [(s.last_token, p)]))
    for s, n, a in zip(pseqs, ntoks, starts):
        a = s.num_computed if a is None else a
        segs.append((s, a, [(int(s.tokens[p]), p) for p in range(a, a + n)]))
    table = lambda seqs, m: np.array([s.block_ids + [0] * (m - len(s.block_ids)) for s in seqs]).reshape(-1, m)   # noqa: E731
    widest = lambda seqs: max([len(s.block_ids) for s in seqs] or [1])   # noqa: E731
    for s, _, r in segs:
        rows += [(t, p, s.block_ids[p // bs] * bs + p % bs) for t, p in r]
    out = {"ids": [r[0] for r in rows], "pos": [r[1] for r in rows], "slots": [r[2] for r in rows],
           "seq_lens": [a + len(r) for _, a, r in segs[len(dseqs):]], "qsl": np.cumsum([0] + list(ntoks)),
           "bt": table(pseqs, widest(pseqs)) if pseqs else np.zeros((1, 1))}
    if dseqs:
        out.update(d_bt=table(dseqs, widest(dseqs)), d_sl=[a + 1 for _, a, _ in segs[:len(dseqs)]])
    if segments:
        out.update(sg_start=np.cumsum([0] + [len(r) for _, _, r in segs]), sg_pos0=[a for _, a, _ in segs],
                   sg_slot=[s.state_slot for s, _, _ in segs], sg_len=[a + len(r) for _, a, r in segs],
                   sg_bt=table(dseqs + pseqs, widest(dseqs + pseqs)), num_segs=len(segs),
                   max_rows=max(len(r) for _, _, r in segs), max_kv=max(a + len(r) for _, a, r in segs))
    return out


@pytest.mark.parametrize("nd,np_", [(0, 1), (1, 0), (3, 0), (0, 4), (5, 3)])
@pytest.mark.parametrize("segments", [False, True])
def test_mixed_rows(nd, np_, segments):
    seqs = sequences(nd + np_, seed=nd + np_)
    dseqs, pseqs, starts, ntoks = seqs[:nd], seqs[nd:], [], []
    for i, s in enumerate(pseqs):
        s.num_computed = s.n_tokens // 3
        starts.append(None if i % 2 else s.n_tokens // 2)
        ntoks.append(max(1, (s.n_tokens - (s.num_computed if i % 2 else s.n_tokens // 2)) - i % 3))
    got = rt().mixed_rows(dseqs, pseqs, ntoks, starts, 16, segments)
    want = mixed_reference(dseqs, pseqs, ntoks, starts, 16, segments)
    assert set(got) == set(want)
    for k, w in want.items():
        if isinstance(w, int):
            assert got[k] == w, k
        else:
            assert got[k].dtype == np.int32 and got[k].shape == np.shape(w) and np.array_equal(got[k], w), k


def test_mixed_rows_are_refused():
    s = sequences(1)[0]
    for args in (([], [], [], []), ([], [s], [1, 1], [0]), ([], [s], [1], [])):
        with pytest.raises(ValueError):
            rt().mixed_rows(*args, 16, True)
    for n, a in ((s.n_tokens + 1, 0), (1, s.n_tokens), (0, 0), (1, -1)):      # tokens that the sequence does not have
        with pytest.raises(IndexError):
            rt().mixed_rows([], [s], [n], [a], 16, True)
    s.block_ids = s.block_ids[:-2]                                            # a position without a page
    with pytest.raises(IndexError):
        rt().mixed_rows([], [s], [s.n_tokens], [0], 16, True)


def test_prompt_ids():
    for toks in ([], [3], list(range(5000)), [np.int64(4), True, 7], (1, 2), np.arange(9)):
        s = Sequence("s", toks, SamplingParams(max_tokens=1))
        assert s.n_tokens == len(toks) and np.array_equal(s.tokens, np.asarray(toks, dtype=np.int32).reshape(-1))
    for bad, err in (([1 << 31], OverflowError), ([1 << 70], OverflowError), ([None], TypeError)):
        with pytest.raises(err):
            Sequence("s", bad, SamplingParams())
