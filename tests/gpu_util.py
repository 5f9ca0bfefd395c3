"""Helpers shared by the GPU parity tests."""
import sys

import numpy as np
import torch


def announce(*what):
    """Name the case before the GPU step, flushed: if the step takes the box down this line survives."""
    print('[gpu-case]', *what, flush=True)
    sys.stdout.flush()


def dev(x: np.ndarray, dtype=None) -> torch.Tensor:
    t = torch.from_numpy(np.ascontiguousarray(x))
    if dtype is not None:
        t = t.to(dtype)
    return t.cuda()


def host(t: torch.Tensor) -> np.ndarray:
    if t.dtype == torch.bfloat16:
        return t.float().cpu().numpy()
    return t.cpu().numpy()


def fastest_ms(call, tries=5):
    """Shortest time of a few calls, by events on the current stream."""
    call()
    best = float('inf')
    for _ in range(tries):
        begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        begin.record()
        call()
        end.record()
        end.synchronize()
        best = min(best, begin.elapsed_time(end))
    return best


def last_launch():
    """(mangled kernel name, workgroups, threads per workgroup) of this thread's latest launch by the library."""
    import ctypes

    from hidet_amd import ffi

    grid, threads = ctypes.c_int64(), ctypes.c_int64()
    name = ffi.load_library().hidet_qmm_last_launch(ctypes.byref(grid), ctypes.byref(threads)).decode()
    return name, grid.value, threads.value


def variant(kernel, *arguments):
    """What the mangled name of a kernel holds for these template arguments (truth values and integers)."""
    return kernel + 'I' + ''.join('L{}{:d}E'.format('b' if isinstance(a, bool) else 'i', a) for a in arguments) + 'E'
