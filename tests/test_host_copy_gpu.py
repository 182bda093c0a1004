"""Copies between the device and pinned host memory by a kernel (csrc/kernels/kv_copy.hip): sizes and addresses that are no whole
16-byte pieces, both directions, one address again and again, and what is refused."""
import pytest
import torch

from fasttalk_llm_microservice_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [0, 1, 3, 4, 5, 1023, 4096, 300001])
@pytest.mark.parametrize("off", [0, 1, 4])
@pytest.mark.parametrize("dtype", [torch.int32, torch.float32, torch.int64])
def test_words(n, off, dtype):
    h = torch.zeros(n + 8, dtype=dtype, pin_memory=True)
    d = torch.zeros(n + 8, dtype=dtype, device="cuda")
    for turn in range(3):                       # (nothing of the turn before is left in a cache)
        x = torch.randint(-9, 9, (n,)).to(dtype)
        h[off:off + n] = x
        ops.native().host_copy(d[3:3 + n], h[off:off + n])
        torch.cuda.synchronize()
        assert torch.equal(d[3:3 + n].cpu(), x) and int(d[:3].abs().sum() + d[3 + n:].abs().sum()) == 0
        d[3:3 + n] += 1
        ops.native().host_copy(h[off:off + n], d[3:3 + n])
        torch.cuda.synchronize()
        assert torch.equal(h[off:off + n], x + 1)
        d.zero_()


def test_memory_freed_under_a_copy():
    """Pinned memory that is freed while a copy is queued is not given to the next tensor before that has run."""
    n = 1 << 16
    a = torch.randn(4096, 4096, device="cuda")
    d = torch.zeros(n, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    for to_host, held in ((False, False), (True, False), (True, True)):
        h = torch.full((n,), 5, dtype=torch.int32, pin_memory=True)
        at = h.data_ptr()
        for _ in range(40):                     # (milliseconds of work in front of the copy)
            b = a @ a
        ops.native().host_copy(*((h, d) if to_host else (d, h)), held=held)
        if held:                                # (the wait that was to come does not)
            ops.native().host_in_use(h)
        done = torch.cuda.Event()
        done.record()
        del h
        new = torch.full((n,), 9, dtype=torch.int32, pin_memory=True)
        assert not done.query() and new.data_ptr() != at
        done.synchronize()
        assert bool((new == 9).all()) and bool((d == 5).all())
    del b


def test_refused():
    d, pinned = torch.zeros(8, dtype=torch.int32, device="cuda"), torch.zeros(8, dtype=torch.int32, pin_memory=True)
    for a, b in ((d, torch.zeros(8, dtype=torch.int32)), (d, d), (pinned, pinned), (d[:4], pinned), (d[::2], pinned[:4]),
                 (d.short(), pinned.short()), (d.float(), pinned)):
        with pytest.raises(RuntimeError):
            ops.native().host_copy(a, b)
