"""The host parts that run on several threads (Newton points and coefficients,
the double-double Cholesky) leave none of them running: the CPU time of the
process over a sleep right after them.  In a process of its own, so that other
libraries' threads do not count."""
import subprocess
import sys

from tests.conftest import ROOT

PROBE = """
import ctypes, time
import numpy as np
import semi_empirical_pseudopotentials_amd as sep
from semi_empirical_pseudopotentials_amd._lib import lib, _p

def burnt():
    t = time.process_time()
    time.sleep(0.15)
    return time.process_time() - t

zn, _ = sep.leja_points(256)
print(burnt())
sep.newton_coeffs(zn, np.linspace(-0.5, 0.5, 8), 12.0, -1.0, 4.0)
print(burnt())
n = 200
A = np.random.default_rng(0).standard_normal((n, 2 * n))
G, R = A @ A.T, np.zeros((n, n))
time.sleep(0.5)  # numpy's own threads
L = lib()
L.sep_la_chol_dd.argtypes = [ctypes.c_long, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_double,
                             ctypes.c_void_p]
assert L.sep_la_chol_dd(n, G.ctypes.data, None, 0.0, R.ctypes.data) == 0
print(burnt())
assert np.abs(R.T @ R - G).max() < 1e-12 * np.abs(G).max()
"""


def test_no_threads_left_running(sep):
    r = subprocess.run([sys.executable, "-c", PROBE], capture_output=True, text=True, cwd=ROOT,
                       timeout=120)
    assert r.returncode == 0, r.stderr
    burnt = [float(v) for v in r.stdout.split()]
    print(burnt)
    assert len(burnt) == 3 and max(burnt) < 0.05
