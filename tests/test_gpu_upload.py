"""GPU: the pinned buffers that uploads share, from several threads and streams."""
import threading

import numpy as np
import pytest
import torch

from torchquantum_amd import engine as E

gpu = pytest.mark.gpu
DEV = torch.device("cuda", 0)
TYPES = [np.complex64, np.float32, np.int64]


def _array(rng, dtype, size):
    raw = rng.integers(0, 256, size=size * np.dtype(dtype).itemsize, dtype=np.uint8)
    if dtype is not np.int64:
        raw = (rng.standard_normal(size * np.dtype(dtype).itemsize // 4).astype(np.float32)).view(np.uint8)
    return raw.view(dtype)


@gpu
def test_uploads_of_threads_and_streams():
    """Four threads with a stream each, 60 uploads of every type and of growing and shrinking sizes per thread through
    eight buffers, the streams kept busy so that copies are still queued when a buffer comes round again: every copy
    holds its own array."""
    wrong, failed = [], []

    def work(k):
        try:
            rng = np.random.default_rng(k)
            stream = torch.cuda.Stream(DEV)
            busy = torch.randn(1 << 22, device=DEV)
            torch.cuda.synchronize()
            kept = []
            with torch.cuda.stream(stream):
                for j in range(60):
                    busy.mul_(1.0001).sin_()
                    a = _array(rng, TYPES[j % 3], int(rng.integers(1, 1 + (1 << rng.integers(1, 17)))))
                    a = a.reshape(-1, 1) if j % 2 else a
                    kept.append((a.copy(), E.upload(a, DEV)))
                    a[...] = 0                  # the caller's array is its own again at once
            stream.synchronize()
            for a, t in kept:
                if t.cpu().numpy().tobytes() != a.tobytes() or tuple(t.shape) != a.shape:
                    wrong.append((k, a.dtype, a.size))
        except Exception as e:      # noqa: BLE001 -- reported by the main thread
            failed.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed and not wrong
    assert len(E._RINGS[DEV].slots) == E._PinnedRing.SLOTS
