"""Device plumbing: torch owns device buffers and streams; libmkgpu computes.

Helpers here turn tensors into raw pointers for the C ABI, hand out the
current HIP stream, and keep per-device scratch (the FP64 reduction
workspace and a small scalar block) so entry points never allocate on the
hot path.
"""
import threading

import numpy as np
import torch

from .lib import mkgpu

_tls = threading.local()


def require_gpu():
    if not torch.cuda.is_available():
        raise RuntimeError("minkasi_amd needs a ROCm GPU (torch.cuda.is_available() is False)")


def device():
    require_gpu()
    return torch.device("cuda", torch.cuda.current_device())


def stream_ptr():
    """Current torch stream as a hipStream_t (void*)."""
    return torch.cuda.current_stream().cuda_stream


def ptr(t, dtype=None, name="tensor"):
    """Raw device pointer of a contiguous CUDA/HIP tensor (checked)."""
    if t is None:
        return None
    if not isinstance(t, torch.Tensor):
        raise TypeError("%s must be a torch tensor on the GPU, got %s" % (name, type(t)))
    if not t.is_cuda:
        raise ValueError("%s must live on the GPU" % name)
    if dtype is not None and t.dtype != dtype:
        raise TypeError("%s must be %s, got %s" % (name, dtype, t.dtype))
    if not t.is_contiguous():
        raise ValueError("%s must be contiguous" % name)
    return t.data_ptr()


def to_device(a, dtype=None):
    """numpy / tensor -> contiguous device tensor (no copy when already there)."""
    dev = device()
    if isinstance(a, torch.Tensor):
        t = a.to(dev)
        if dtype is not None:
            t = t.to(dtype)
        return t.contiguous()
    a = np.ascontiguousarray(a)
    t = torch.from_numpy(a).to(dev)
    if dtype is not None:
        t = t.to(dtype)
    return t.contiguous()


class HostFetch:
    """Copies a device tensor into a new numpy array of another data type.

    A copy into fresh pageable memory is bound by its page faults and by
    staging copies, and holds the stream meanwhile.  Here a side stream
    converts and copies kChunk elements at a time into two pinned buffers
    (torch's pool of pinned memory keeps them), so work queued between the
    construction and result() runs beside it, and result() moves the chunks on
    into memory that numpy asks for in huge pages.  19.4 million FP64 values to
    FP32: 6 ms against 19 for .to(float32).cpu().  Moving them with more
    threads, or on a thread of its own, measured no gain: the threads wait for
    each other's page faults."""

    kChunk = 1 << 21

    def __init__(self, t, dtype):
        self.src = t.reshape(-1)
        self.out = np.empty(tuple(t.shape), dtype=dtype)
        on_dev = torch.from_numpy(self.out).dtype
        size = min(self.kChunk, self.src.numel())
        # The device buffers come from the caller's stream: torch keeps memory
        # per stream and hands out 32 side streams in turn, so buffers of the
        # side streams' own would stay reserved 32 times over, out of reach of
        # everything else.
        buffers = [torch.empty(size, dtype=on_dev, device=t.device) for _ in range(2)]
        self.stream = torch.cuda.Stream(device=t.device)
        self.stream.wait_stream(torch.cuda.current_stream(t.device))
        for used in (self.src, *buffers):
            used.record_stream(self.stream)  # also where result() is never reached
        with torch.cuda.stream(self.stream):
            self.slots = [(b, torch.empty(size, dtype=on_dev, pin_memory=True), torch.cuda.Event()) for b in buffers]
            for i in range(2):
                self._issue(i)

    def _range(self, i):
        return i * self.kChunk, min((i + 1) * self.kChunk, self.src.numel())

    def _issue(self, i):
        a, b = self._range(i)
        if a < b:
            on_dev, pinned, done = self.slots[i % 2]
            on_dev[:b - a].copy_(self.src[a:b])
            pinned[:b - a].copy_(on_dev[:b - a], non_blocking=True)
            done.record()

    def result(self):
        """The array.  Every read of the tensor has finished then, so it may be
        freed on its own stream."""
        flat = self.out.reshape(-1)
        with torch.cuda.stream(self.stream):
            for i in range(-(-self.src.numel() // self.kChunk)):
                a, b = self._range(i)
                _, pinned, done = self.slots[i % 2]
                done.synchronize()
                np.copyto(flat[a:b], pinned[:b - a].numpy())
                self._issue(i + 2)
        self.src = self.slots = None
        return self.out


class Scratch:
    """Per-device reduction workspace + FP64 scalar block."""

    def __init__(self, dev):
        nbytes = int(mkgpu.lib.mk_reduce_workspace_bytes())
        self.work = torch.empty(nbytes // 8 + 32, dtype=torch.float64, device=dev)
        self.sc = torch.zeros(mkgpu.SC_COUNT, dtype=torch.float64, device=dev)


_scratch = {}


def scratch():
    dev = device()
    s = _scratch.get(dev.index)
    if s is None:
        s = Scratch(dev)
        _scratch[dev.index] = s
    return s


def torch_dtype(x):
    if isinstance(x, torch.Tensor):
        return x.dtype
    return {np.dtype(np.float32): torch.float32, np.dtype(np.float64): torch.float64}[np.asarray(x).dtype]
