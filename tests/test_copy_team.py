"""The threads that copy large downloads out of the pinned staging buffer
(sep_copy_team_*, csrc/sep_host.c): every byte of lengths around their cuts,
copies in quick succession, teams side by side, no CPU time used once a team
rests (a caller's own work follows a download at once) and no thread left once
it is closed."""
import ctypes
import os
import threading
import time

import numpy as np
import pytest

P = 8 * 4096  # pieces are whole pages, an eighth of the copy each
LENGTHS = (1, 4095, 4096, 4097, P - 1, P, P + 1, 5 * P + 3, (1 << 20) + 7, (8 << 20) - 1, 8 << 20)


@pytest.fixture(scope="module")
def host(sep):
    from semi_empirical_pseudopotentials_amd._lib import LIB_PATH
    L = ctypes.CDLL(LIB_PATH)
    L.sep_copy_team_open.restype = ctypes.c_void_p
    for name, args in (("wake", 0), ("rest", 0), ("close", 0), ("run", 3)):
        fn = getattr(L, "sep_copy_team_" + name)
        fn.restype = None
        fn.argtypes = [ctypes.c_void_p] + [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t][:args]
    return L


@pytest.fixture
def team(host):
    t = host.sep_copy_team_open()
    assert t
    yield t
    host.sep_copy_team_close(t)


def _copies(host, team, lengths, seed):
    rng = np.random.default_rng(seed)
    for n in lengths:
        src = rng.integers(0, 256, n, dtype=np.uint8)
        dst = np.zeros(n + 64, np.uint8)
        host.sep_copy_team_run(team, dst.ctypes.data, src.ctypes.data, n)
        if not (np.array_equal(dst[:n], src) and not dst[n:].any()):
            return False
    return True


def test_every_byte(host, team):
    host.sep_copy_team_wake(team)
    assert _copies(host, team, LENGTHS, 0)
    host.sep_copy_team_rest(team)


def test_alone(host, team):
    """No team, and one that is not awake: the caller copies by itself."""
    assert _copies(host, None, LENGTHS, 1)
    assert _copies(host, team, LENGTHS, 2)


def test_many_copies(host, team):
    """Copies in quick succession, whose late threads meet the next one."""
    for k in range(60):
        host.sep_copy_team_wake(team)
        for j in range(5):
            assert _copies(host, team, ((64 << 10) * (1 + j) + k % 3,), k)
        host.sep_copy_team_rest(team)


def test_teams_side_by_side(host):
    ok = [False] * 4

    def work(i):
        for k in range(5):
            team = host.sep_copy_team_open()
            host.sep_copy_team_wake(team)
            ok[i] = _copies(host, team, LENGTHS[:-2], 10 * i + k)
            host.sep_copy_team_rest(team)
            host.sep_copy_team_close(team)
            if not ok[i]:
                return

    th = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert all(ok)


def test_nothing_left_running(host):
    before = len(os.listdir("/proc/self/task"))
    n = 8 << 20
    src, dst = np.ones(n, np.uint8), np.zeros(n, np.uint8)
    team = host.sep_copy_team_open()
    host.sep_copy_team_wake(team)
    host.sep_copy_team_run(team, dst.ctypes.data, src.ctypes.data, n)
    host.sep_copy_team_rest(team)
    t = time.process_time()
    time.sleep(0.15)
    assert time.process_time() - t < 0.05
    host.sep_copy_team_close(team)
    assert len(os.listdir("/proc/self/task")) <= before
