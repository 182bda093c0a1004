"""Head norm with gate by whole fours of a head (csrc/mixers/rows.hip head_rms_gate_fours_kernel) against 64 bits: every head
size, one and four heads at a time, ends of the grid, and operands it leaves to the other kernel; the sigmoid at its ends."""
import pytest
import torch

from fasttalk_llm_microservice_amd.ops import mixers as M
from test_mixer_kernels_gpu import DEV, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,heads,dv", [(1, 1, 16), (3, 5, 32), (7, 3, 64), (2731, 3, 128), (4099, 1, 256), (1025, 33, 64), (5, 2, 36)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("off", [0, 1])
def test_head_rms_gate(rows, heads, dv, dt, off):
    g = torch.Generator().manual_seed(rows + dv)
    o, w = rnd(rows, heads * dv, g=g).to(DEV), rnd(dv, g=g).to(DEV)
    gate = (8 * rnd(rows, heads * dv + 8, g=g)).to(dt).to(DEV)[:, off:off + heads * dv]
    gate[0, :4] = torch.tensor([200.0, -200.0, float("inf"), 0.0], dtype=dt)
    for silu in (False, True):
        if silu:
            gate[0, 1] = -90.0
        got = M.head_rms_gate(o, w, gate, 1e-5, heads, dv, dt, silu=silu)
        x, z = o.double().view(rows, heads, dv), gate.double().view(rows, heads, dv)
        want = x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5) * w.double() * torch.sigmoid(z) * (z if silu else 1.0)
        fin = torch.isfinite(want).view(rows, -1)
        # fp32 sums of up to 256 terms and a few roundings; bf16: one rounding of the result
        torch.testing.assert_close(got.double()[fin], want.view(rows, -1)[fin], rtol=2 ** -8 if dt == torch.bfloat16 else 2e-6, atol=1e-30)
        assert bool(torch.isinf(got[~fin]).all())


def test_sigmoid_in_its_tail():
    """z sigmoid(z) in fp32: within a few units in the last place as far as the sigmoid is any number, half the smallest one's
    step times |z| below the normal numbers, -0 beyond."""
    z = torch.cat([torch.linspace(-104.5, -30, 1 << 16), torch.linspace(-30, 110, 1 << 16), torch.tensor([-1e5, -1e30, -3.4e38])]).to(DEV)
    got = M.silu_glu(torch.stack([z, torch.ones_like(z)], 1).contiguous())[:, 0].double()
    want = z.double() * torch.sigmoid(z.double())
    err = (got - want).abs()
    # the exponential's, the sum's and the reciprocal's roundings, and that of the product: 4 units of 2^-24 at most
    bound = want.abs() * 2.0 ** -22 + z.double().abs().clamp(max=105.0) * 2.0 ** -149
    assert bool((err <= bound).all()), (float(z[(err - bound).argmax()]), float((err / bound).max()))
