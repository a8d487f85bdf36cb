"""Chunked device-to-host copies (device.HostFetch) equal a direct one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 7, (1 << 21) - 1, 1 << 21, (1 << 21) + 1, 2 * (1 << 21) + 5, 5 * (1 << 21) + 3])
def test_host_fetch_equals_direct_copy(n):
    import torch
    from minkasi_amd import device
    t = torch.arange(n, dtype=torch.float64, device=device.device()) * 1.0000001
    fetch = device.HostFetch(t.reshape(1, n), np.float32)
    busy = t * 2  # work queued in between
    got = fetch.result()
    assert got.shape == (1, n) and got.dtype == np.float32
    assert np.array_equal(got[0], t.to(torch.float32).cpu().numpy())
    assert torch.equal(busy, t * 2)


def test_host_fetch_of_a_strided_tensor():
    import torch
    from minkasi_amd import device
    t = torch.arange(3 * (1 << 20), dtype=torch.float64, device=device.device()).reshape(3, 1 << 20).T
    assert np.array_equal(device.HostFetch(t, np.float32).result(), t.to(torch.float32).cpu().numpy())


def test_host_fetch_keeps_no_memory():
    """More fetches than torch has side streams reserve no more device memory
    than a few pairs of 8 MiB buffers, in segments of 20 MiB: the buffers just
    given back may still wait for their event."""
    import torch
    from minkasi_amd import device
    t = torch.ones(2 * device.HostFetch.kChunk, dtype=torch.float64, device=device.device())
    device.HostFetch(t, np.float32).result()
    before = torch.cuda.memory_reserved()
    for _ in range(40):
        device.HostFetch(t, np.float32).result()
    assert torch.cuda.memory_reserved() - before <= 3 * (20 << 20)
