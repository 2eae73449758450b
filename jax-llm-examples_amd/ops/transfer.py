"""Small arrays on their way to the device."""
from __future__ import annotations

import torch


def to_device(host: torch.Tensor, device) -> torch.Tensor:
    """A copy of ``host`` on ``device``, in the current stream's order: by way of pinned memory, so that nobody waits.  (From
    ordinary memory the copy returns only when everything launched before it has run: a prompt's step that brings four lists
    of work to the device that way has the device idle four times, until its next launches are there.)  The pinned memory is
    given back to its allocator, which keeps it until the copy is done."""
    device = torch.device(device)
    if device.type != "cuda":
        return host.to(device)
    return host.pin_memory().to(device, non_blocking=True)
