"""Values into their transposed cache blocks (csrc/kernels/rope_kv.hip): tokens whose slots follow each other from any place of a
block on, in runs that end inside sixteen tokens, scattered and left out; bf16 and fp8, bit for bit the reference's."""
import pytest
import torch

from fasttalk_llm_microservice_amd import ops
from fasttalk_llm_microservice_amd.ops import ref

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("bs,fp8", [(16, False), (8, False), (12, False), (16, True), (20, True), (24, True)])
@pytest.mark.parametrize("d,nkv", [(128, 2), (64, 3)])
@pytest.mark.parametrize("runs", [[(0, 1)], [(0, 16)], [(5, 48)], [(8, 7), (40, 30), (-1, 3), (96, 17)], [(24, 8), (39, 9), (80, 95)]])
def test_values(bs, d, nkv, fp8, runs):
    g = torch.Generator().manual_seed(bs + d)
    slots = [s + i if s >= 0 else -1 for s, n in runs for i in range(n)]
    t, nq, blocks = len(slots), 4, 24
    assert max(slots) < blocks * bs
    qkv = torch.randn(t, (nq + 2 * nkv) * d, generator=g).bfloat16().to(DEV)
    pos, cs = torch.arange(t, dtype=torch.int32, device=DEV), ref.rope_cos_sin(d, 512, 1e4, None, DEV)
    slots = torch.tensor(slots, dtype=torch.int32, device=DEV)
    shape = (blocks, nkv, bs, d), (blocks, nkv, d, bs)
    dt = torch.float8_e4m3fn if fp8 else torch.bfloat16
    (k1, v1), (k2, v2) = ([torch.ones(s, device=DEV).to(dt) for s in shape] for _ in range(2))
    ops.rope_kv_write(qkv.clone(), pos, cs, slots, k1, v1, nq, nkv, d)
    ref.rope_kv_write(qkv.clone(), pos, cs, slots, k2, v2, nq, nkv, d)
    assert torch.equal(v1.view(torch.uint8), v2.view(torch.uint8))
