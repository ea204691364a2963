"""A launch shape set by hand runs every step on its own; the autotuner brings the
launches of several steps back, seen by the buffer they take on a GPU whose
memory hip_budget.cpp counts, with the same results."""
import ctypes as C
import os
import subprocess
import sys

import pytest

from test_zz_spare_memory import HERE, small_gpu  # noqa: F401


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["lattice", "batch"])
def test_autotune_after_a_shape_set_by_hand(small_gpu, kind):  # noqa: F811
    r = subprocess.run([sys.executable, os.path.abspath(__file__), small_gpu, kind], capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0 and r.stdout.endswith("ok\n"), r.stdout + r.stderr


def _main(so, kind):
    budget = C.CDLL(so, mode=C.RTLD_GLOBAL)  # before the library
    budget.budget_set.argtypes = [C.c_size_t]
    budget.budget_used.restype = C.c_size_t
    budget.budget_set(4 << 30)
    sys.path[:0] = [HERE, os.path.dirname(HERE)]
    import numpy as np
    from helpers import c1_ops, channel_flags_2d, parabolic_inlet
    from lbm_mirror_amd import abi
    from lbm_mirror_amd.lattice import Batch, Lattice
    ext = (300, 200)
    spare = 9 * 8 * ext[0] * ext[1]
    out = []
    for tuned in (False, True):
        b = Lattice(abi.D2Q9, abi.F64, ext) if kind == "lattice" else Batch(abi.D2Q9, abi.F64, [ext])
        m = b if kind == "lattice" else b.members[0]
        m.set_flags(channel_flags_2d(*ext))
        for fl, op in c1_ops(0.8, 0.05).items():
            m.set_operator(fl, op)
        m.set_boundary_velocity(parabolic_inlet(*ext, 0.05))
        m.init_equilibrium(1.0, (0.0, 0.0))
        if tuned:
            (b.set_step_tuning if kind == "lattice" else lambda w: b.set_tuning(w, 1, 0))(64)
        before = budget.budget_used()
        b.step(40)
        # (a batch takes its lists of tiles there too)
        assert (budget.budget_used() - before < spare // 2) == tuned
        b.autotune()
        before = budget.budget_used()
        b.step(40)
        if tuned:
            assert budget.budget_used() - before >= spare
        out.append((m.get_populations(), *m.get_macros()))
        b.close()
    for x, y in zip(*out):
        assert np.array_equal(x, y)


if __name__ == "__main__":
    _main(*sys.argv[1:])
    print("ok")
