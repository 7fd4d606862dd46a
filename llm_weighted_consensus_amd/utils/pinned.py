"""Uploads that the host does not wait for."""
from __future__ import annotations

from typing import List

import numpy as np
import torch

MOST_BYTES = 2 << 20   # of one pinned upload; beyond, the work behind it is long enough for the host to wait
_TORCH = {"uint8": torch.uint8, "int32": torch.int32, "int64": torch.int64, "float32": torch.float32}


def to_device(device, *arrays: np.ndarray) -> List[torch.Tensor]:
    """Host arrays on ``device`` by one copy, ordered on the current stream alone.  On a GPU a pageable copy waits for everything
    queued on the stream, which runs dry while the host goes on (the three arrays of a batch of 64 texts, then the first
    launches: 0.1 ms without a kernel); here the arrays are staged through a block of torch's pinned pool, which keeps it from
    other uses until the copy is over.  86 kB take the host 22 us, a pageable copy 31 and the wait; a ring of the caller's
    own with events of its own 45 to 75.  What is larger than ``MOST_BYTES`` goes the pageable way, and so does what is
    captured (which refuses it)."""
    dev = torch.device(device)
    at, arrays = [0], [np.ascontiguousarray(a) for a in arrays]
    for a in arrays:
        at.append(at[-1] + (a.nbytes + 15 & ~15))
    if dev.type != "cuda" or at[-1] > MOST_BYTES or torch.cuda.is_current_stream_capturing():
        return [torch.from_numpy(a).to(dev) for a in arrays]
    block = torch.empty(at[-1], dtype=torch.uint8, pin_memory=True)
    host = block.numpy()   # (numpy copies: torch's host copy of as much wakes its threads and takes 100 us)
    for a, o in zip(arrays, at):
        host[o:o + a.nbytes].view(a.dtype)[:] = a.ravel()
    held, out, views = block.to(dev, non_blocking=True), [], {}
    for a, o in zip(arrays, at):
        v = views.get(a.dtype)
        if v is None:
            v = views[a.dtype] = held.view(_TORCH[a.dtype.name])
        t = v[o // a.itemsize:o // a.itemsize + a.size]
        out.append(t if a.ndim == 1 else t.view(a.shape))
    return out
