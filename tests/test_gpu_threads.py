"""Calls into the native module beside other Python threads."""
import threading
import time

import pytest
import torch

pytestmark = pytest.mark.gpu

GIB = 1 << 30


def test_other_threads_run_while_a_call_waits_for_the_device():
    """A result that fits only once the allocator has given cached memory back, while the device is busy: freeing waits for
    the device, and the other Python threads go on meanwhile."""
    import any_precision_ext as ext
    N, K = 16384, 49152                                                # 1.5 GiB of fp16
    q = torch.zeros((3, N, K // 32), dtype=torch.int32, device="cuda")
    lut = torch.zeros((N, 8), dtype=torch.float16, device="cuda")
    a = torch.zeros((8192, 8192), dtype=torch.float16, device="cuda")
    out = torch.empty_like(a)
    torch.mm(a, a, out=out)
    ext.dequant_kbit(q[:, :64].contiguous(), lut[:64].contiguous(), 3)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    torch.empty((GIB,), dtype=torch.uint8, device="cuda")              # stays in the cache, too small for the result
    limit = (torch.cuda.memory_reserved() + 0.8 * GIB) / torch.cuda.get_device_properties(0).total_memory
    ticks, stop = [], threading.Event()

    def tick():
        while not stop.is_set():
            ticks.append(time.perf_counter())
            time.sleep(0.001)

    thread = threading.Thread(target=tick)
    torch.cuda.set_per_process_memory_fraction(limit)
    try:
        thread.start()
        for _ in range(400):                                           # some 0.3 s of work
            torch.mm(a, a, out=out)
        start = time.perf_counter()
        ext.dequant_kbit(q, lut, 3)
        end = time.perf_counter()
    finally:
        stop.set()
        thread.join()
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert end - start > 0.05, "the call did not wait for the device"
    inside = [start] + [t for t in ticks if start < t < end] + [end]
    gap = max(b - a for a, b in zip(inside, inside[1:]))
    print(f"call {end - start:.3f} s, longest gap {gap:.4f} s", flush=True)
    assert gap < 0.5 * (end - start)
