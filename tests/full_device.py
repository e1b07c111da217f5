"""A card whose memory is taken, for tests of what runs with little room."""
import contextlib

import torch


@contextlib.contextmanager
def full_device(left_mib):
    """Holds device memory so that no more than left_mib MiB (a multiple of 64, to within
    the driver's granules) can be allocated."""
    torch.cuda.empty_cache()
    step = 64 << 20
    held = [torch.empty(max(torch.cuda.mem_get_info()[0] - (2 << 30), step), dtype=torch.uint8, device="cuda")]
    while True:  # the driver gives more than it reports free
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
