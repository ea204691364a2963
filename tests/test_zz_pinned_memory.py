"""Read-back of fields where the host has no pinned memory left (hip_budget.cpp):
the same values, below and above the size up to which one thread works alone."""
import ctypes as C
import os
import subprocess
import sys

import pytest

from test_zz_spare_memory import HERE, small_gpu  # noqa: F401


@pytest.mark.gpu
def test_read_back_without_pinned_memory(small_gpu):  # noqa: F811
    r = subprocess.run([sys.executable, os.path.abspath(__file__), small_gpu], capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0 and r.stdout.endswith("ok\n"), r.stdout + r.stderr


def _main(so):
    shim = C.CDLL(so, mode=C.RTLD_GLOBAL)  # before the library
    shim.budget_set.argtypes = [C.c_size_t]
    shim.budget_set(16 << 30)
    sys.path[:0] = [HERE, os.path.dirname(HERE)]
    import numpy as np
    from lbm_mirror_amd import abi
    from lbm_mirror_amd.lattice import Lattice
    for st, ext in ((abi.F32, (97, 31)), (abi.F64, (700, 500)), (abi.F32, (1023, 517)), (abi.F64, (2000, 1501))):
        s = Lattice(abi.D2Q9, st, ext)
        rng = np.random.default_rng(2)
        rho, u = rng.uniform(0.9, 1.1, s.N), rng.uniform(-0.1, 0.1, (2, s.N))
        shim.pinned_set(0)
        s.set_macros(rho, u)
        got = s.get_macros()
        shim.pinned_set(1)
        if st == abi.F32:
            rho, u = (a.astype(np.float32).astype(np.float64) for a in (rho, u))
        assert np.array_equal(got[0], rho) and np.array_equal(got[1], u), ext
        s.close()


if __name__ == "__main__":
    _main(*sys.argv[1:])
    print("ok")
