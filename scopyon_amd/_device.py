"""Device plumbing on top of PyTorch-ROCm: current device/stream, uploads,
and a per-device scratch arena (so kernels never allocate on the hot path)."""
import numpy
import torch

from . import _lib


def require_gpu():
    """Load the HIP library and check that a GPU is visible (no CPU fallback)."""
    _lib.lib()
    if not torch.cuda.is_available():
        raise RuntimeError('scopyon_amd: no HIP device is visible; the GPU path has no CPU fallback')
    return torch.device('cuda', torch.cuda.current_device())


def stream():
    """Raw hipStream_t of torch's current stream (for the C-ABI)."""
    return torch.cuda.current_stream().cuda_stream


def ptr(t):
    return None if t is None else t.data_ptr()


def upload(a, dtype=torch.float64, device=None):
    """Device copy of a host array, complete on return: for what an object keeps,
    which may be used on other streams than the one it was made on."""
    device = device or require_gpu()
    return torch.from_numpy(numpy.ascontiguousarray(a)).to(device=device, dtype=dtype,
                                                           non_blocking=False)


UPLOAD_STAGED = 1 << 18   # bytes


def stage(a, dtype=torch.float64, device=None):
    """Device copy of a host array, ordered on the current stream: for what only the
    work that the caller queues on this stream reads.  Small arrays go through
    pinned memory: a copy from pageable memory would wait for the kernels before
    it on the stream (torch keeps the pinned block until it is read)."""
    device = device or require_gpu()
    a = numpy.ascontiguousarray(a)
    if not 0 < a.nbytes <= UPLOAD_STAGED:
        return upload(a, dtype, device)
    src = torch.from_numpy(a)
    staged = torch.empty(src.shape, dtype=dtype, pin_memory=True)
    return staged.copy_(src).to(device=device, non_blocking=True)


class Arena:
    """Grow-only named scratch buffers, one set per device."""

    def __init__(self):
        self._bufs = {}

    def get(self, name, nbytes, device):
        key = (name, device.index if hasattr(device, 'index') else device)
        buf = self._bufs.get(key)
        nbytes = max(int(nbytes), 1)
        if buf is None or buf.numel() < nbytes:
            buf = torch.empty(int(nbytes * 1.25) + 256, dtype=torch.uint8, device=device)
            self._bufs[key] = buf
        return buf

    def typed(self, name, n, dtype, device):
        itemsize = torch.empty((), dtype=dtype).element_size()
        raw = self.get(name, max(int(n), 1) * itemsize, device)
        return raw[: max(int(n), 1) * itemsize].view(dtype)[: int(n)]


ARENA = Arena()
