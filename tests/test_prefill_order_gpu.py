"""Order of the prefill attention's work (csrc/kernels/attn_prefill.hip): items longest first and all heads of one before the
next where they take several rounds of the CUs, with the results of a sequence alone."""
import pytest
import torch

from fasttalk_llm_microservice_amd import ops

DEV = "cuda"


@pytest.mark.parametrize("q_lens,cached", [([4096], 0), ([2048], 0), ([777], 0), ([64, 2000, 300], 0), ([400] * 5, 100), ([30] * 40, 0)])
def test_plan_longest_first(q_lens, cached):
    seq_lens = [q + cached for q in q_lens]
    items, comb = ops.build_prefill_tiles(q_lens, 64, seq_lens=seq_lens, nkv=8, num_cus=256)
    seen = {}
    sizes = []
    for b, s, rng, slot in items:
        nkt = -(-(cached + s + min(64, q_lens[b] - s)) // 64)
        lo, hi = (0, nkt) if rng == 0xFFFF else (rng >> 16, rng & 0xFFFF)
        seen.setdefault((b, s), []).append((lo, hi, slot))
        sizes.append(hi - lo)
    assert set(seen) == {(b, s) for b, q in enumerate(q_lens) for s in range(0, q, 64)}
    parts = {(b, s): (first, n) for b, s, first, n in comb}
    for (b, s), got in seen.items():
        got.sort()
        assert got[0][0] == 0 and got[-1][1] == -(-(cached + s + min(64, q_lens[b] - s)) // 64)
        assert all(x[1] == y[0] for x, y in zip(got, got[1:]))
        if len(got) > 1:
            assert [x[2] for x in got] == list(range(parts[b, s][0], sum(parts[b, s])))
    if len(items) * 8 > 256:
        assert sizes == sorted(sizes, reverse=True)


@pytest.mark.gpu
@pytest.mark.parametrize("nq,nkv", [(32, 8), (8, 8), (6, 3), (8, 1)])
def test_together_as_alone(nq, nkv):
    g = torch.Generator().manual_seed(nq)
    d, bs, n = 64, 16, 300 // nkv + 2          # one item a sequence: more workgroups than CUs
    lens = [5 + int(x) for x in torch.randint(0, 60 if nq > nkv else 250, (n,), generator=g)]
    lens = [min(v, ops.prefill_tile_tokens(nq, nkv)) for v in lens]
    nb = [-(-v // bs) for v in lens]
    kc, vc = (torch.randn(sum(nb), nkv, *s, generator=g).to(DEV, torch.bfloat16) for s in ((bs, d), (d, bs)))
    q = torch.randn(sum(lens), nq * d, generator=g).to(DEV, torch.bfloat16)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)      # noqa: E731
    first = [sum(nb[:i]) for i in range(n)]

    def run(seqs):
        rows = [sum(lens[:i]) for i in seqs]
        x = torch.cat([q[r:r + lens[i]] for r, i in zip(rows, seqs)])
        bt = torch.zeros(len(seqs), max(nb), dtype=torch.int32)
        for k, i in enumerate(seqs):
            bt[k, :nb[i]] = torch.arange(first[i], first[i] + nb[i])
        tiles, comb = ops.build_prefill_tiles([lens[i] for i in seqs], ops.prefill_tile_tokens(nq, nkv),
                                              seq_lens=[lens[i] for i in seqs], nkv=nkv)
        assert not comb
        out = torch.empty_like(x)
        start = [0]
        for i in seqs:
            start.append(start[-1] + lens[i])
        ops.prefill_attention(out, x, kc, vc, bt.to(DEV), i32([lens[i] for i in seqs]), i32(start), i32(tiles).flatten(), len(tiles),
                              nq, nkv, d, d ** -0.5)
        return out, len(tiles)

    together, items = run(list(range(n)))
    assert items * nkv > 256
    assert torch.equal(together, torch.cat([run([i])[0] for i in range(n)]))
