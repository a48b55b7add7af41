"""Small host arrays on the device, several in one transfer."""
from __future__ import annotations

from typing import List, Sequence

import numpy as np
import torch


def upload(arrays: Sequence[np.ndarray], device: torch.device
           ) -> List[torch.Tensor]:
    """The arrays as tensors on ``device``, in order; on a GPU they share one
    buffer and one copy from pinned memory that the host does not wait for
    (a pageable copy waits for all work before it on the stream, and each costs
    10 to 20 us; torch keeps pinned memory until its copies are done)."""
    arrays = [np.ascontiguousarray(a) for a in arrays]
    if torch.device(device).type != "cuda":
        return [torch.from_numpy(a.copy()) for a in arrays]
    # every array begins at a multiple of 16 bytes, for kernels that read so
    begin, total = [], 0
    for a in arrays:
        begin.append(total)
        total += (a.nbytes + 15) // 16 * 16
    host = torch.empty(max(total, 16), dtype=torch.uint8, pin_memory=True)
    raw = host.numpy()
    for a, at in zip(arrays, begin):
        raw[at:at + a.nbytes] = a.reshape(-1).view(np.uint8)
    dev = host.to(device, non_blocking=True)
    return [dev[at:at + a.nbytes].view(_TORCH[a.dtype.type]).view(a.shape)
            for a, at in zip(arrays, begin)]


_TORCH = {np.int32: torch.int32, np.int64: torch.int64}
