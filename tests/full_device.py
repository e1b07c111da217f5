"""A card whose memory is taken, for tests of what runs with little room."""
import contextlib

import torch


@contextlib.contextmanager
def full_device(left_mib):
    """Holds device memory so that less than left_mib + 12 MiB (left_mib a multiple of 64)
    can be allocated."""
    torch.cuda.empty_cache()
    most = 64 << 20
    held = [torch.empty(max(torch.cuda.mem_get_info()[0] - (2 << 30), most), dtype=torch.uint8, device="cuda")]
    for step in (most, 12 << 20):  # the driver gives more than it reports free
        if step < most and left_mib > 0:
            continue
        while True:
            try:
                held.append(torch.empty(step, dtype=torch.uint8, device="cuda"))
            except torch.OutOfMemoryError:
                break
    del held[len(held) - left_mib // 64:]
    torch.cuda.empty_cache()
    try:
        yield
    finally:
        held.clear()
        torch.cuda.empty_cache()
