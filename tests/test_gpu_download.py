"""Downloads into memory that the runtime knows (pinned, a device's): the plain
copy, without the staging buffer and the threads that copy it out (8 MB and more
into pageable memory)."""
import ctypes
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
N = 64 ** 3


def _threads():
    return len(os.listdir("/proc/self/task"))


def _open(sep, m):
    ctx = sep.Context(64, 64, 64, 0.7, 0.8, 0.9)
    a = np.random.default_rng(5).standard_normal((m, N))
    ctx.states_upload(a)
    return ctx, a


def _get(ctx, ptr, m):
    from semi_empirical_pseudopotentials_amd._lib import lib
    rc = lib().sep_states_download(ctx._h, ctypes.cast(ptr, ctypes.POINTER(ctypes.c_double)), m)
    assert rc == 0


@pytest.mark.parametrize("m", [3, 4, 5, 16, 33])  # 6.3, 8.4, 10.5, 34 and 69 MB
def test_destinations(sep, m):
    import torch
    print("case download", m, flush=True)
    ctx, a = _open(sep, m)
    with ctx:
        pinned = torch.zeros(m + 1, N, dtype=torch.float64, pin_memory=True)
        _get(ctx, pinned.data_ptr(), m)
        assert np.array_equal(pinned[:m].numpy(), a) and not pinned[m].any()
        dev = torch.zeros(m + 1, N, dtype=torch.float64, device="cuda:0")
        torch.cuda.synchronize()
        _get(ctx, dev.data_ptr(), m)
        assert np.array_equal(dev[:m].cpu().numpy(), a) and not dev[m].any()
        assert np.array_equal(ctx.states_download(m), a)


def test_pinned_needs_no_staging(sep):
    import torch
    m = 16
    pinned = torch.zeros(m, N, dtype=torch.float64, pin_memory=True)
    ctx, a = _open(sep, m)  # the runtime's own threads start here
    with ctx:
        _get(ctx, pinned.data_ptr(), m)
        ctx.states_download(m)
    ctx, a = _open(sep, m)
    with ctx:
        before = _threads()
        _get(ctx, pinned.data_ptr(), m)
        assert np.array_equal(pinned.numpy(), a)
        assert _threads() == before
        ctx.states_download(m)
        assert _threads() > before or len(os.sched_getaffinity(0)) == 1
    assert _threads() == before
