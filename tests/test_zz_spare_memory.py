"""The second population buffer of D2Q9 lattices and batches is spare: it goes
when another lattice, batch or network needs the GPU's memory, and when no
step can use it any more; a call of too few steps for it does not take it.  The
lattices then run on, step by step, with the same results.  Each case runs in a process of its own, on a GPU that
hip_budget.cpp makes small."""
import ctypes as C
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CASES = ["lattice_lattice", "lattice_network", "batch_batch", "shape", "operator", "particles", "tiles",
         "short", "shortbatch"]
EXT = (1024, 500)
SPARE = 9 * 4 * EXT[0] * EXT[1]  # FP32
MB = 1 << 20


@pytest.fixture(scope="module")
def small_gpu(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("budget") / "hip_budget.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", os.path.join(HERE, "hip_budget.cpp"), "-o", so, "-L/opt/rocm/lib",
                    "-Wl,--no-as-needed", "-lamdhip64", "-Wl,-rpath,/opt/rocm/lib", "-ldl"], check=True)
    return so


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES)
def test_spare_buffer(small_gpu, case):
    r = subprocess.run([sys.executable, os.path.abspath(__file__), small_gpu, case], capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0 and r.stdout.endswith("ok\n"), r.stdout + r.stderr


def _main(so, case):
    budget = C.CDLL(so, mode=C.RTLD_GLOBAL)  # before the library
    budget.budget_set.argtypes = [C.c_size_t]
    budget.budget_used.restype = C.c_size_t
    budget.budget_set(4 << 30)
    sys.path[:0] = [HERE, os.path.dirname(HERE)]
    import numpy as np
    from helpers import c1_ops, channel_flags_2d, make_particle, parabolic_inlet
    from lbm_mirror_amd import abi
    from lbm_mirror_amd.lattice import Batch, Lattice
    from lbm_mirror_amd.warmstart import Net
    used = budget.budget_used

    def setup(s, ext):
        s.set_flags(channel_flags_2d(*ext))
        for fl, op in c1_ops(0.8, 0.05).items():
            s.set_operator(fl, op)
        s.set_boundary_velocity(parabolic_inlet(*ext, 0.05))
        s.init_equilibrium(1.0, (0.0, 0.0))

    def lattice():
        s = Lattice(abi.D2Q9, abi.F32, EXT)
        setup(s, EXT)
        return s

    def batch(count=4):
        ext = (EXT[0], EXT[1] // count)
        b = Batch(abi.D2Q9, abi.F32, [ext] * count)
        for m in b.members:
            setup(m, ext)
        return b

    has, _, needs = case.partition("_")
    if case.startswith("short"):
        a = lattice() if case == "short" else batch()
        before = used()
        for n in (1, 2, 4, 3):
            a.step(n)
            assert used() - before < SPARE // 2
        a.step(5)
        assert used() - before >= SPARE
        a.step(1)
        a.close()
        return
    if not needs:
        a = batch() if case == "tiles" else lattice()
        before = used()
        a.step(37)
        assert used() - before >= SPARE
        if case == "shape":
            a.set_step_tuning(64)
        elif case == "tiles":
            a.set_tuning(256, 1, 0)
        elif case == "operator":
            a.set_operator(9, abi.op_desc(collision=abi.COLL_PSM, tau=0.8))
        else:
            a.particles_set([make_particle([50.0, 50.0], 4.0, 1.5, 2, abi.F32, mass=50.0, inertia=400.0)],
                            abi.particle_params(max_radius=4.0))
        assert used() - before < SPARE // 2
        a.step(3)
        a.close()
        return
    out = []
    for pressed in (False, True):
        a = lattice() if has == "lattice" else batch()
        before = used()
        a.step(37)
        assert used() - before >= SPARE  # it has its spare buffer
        if pressed:
            # what is left is too little for what comes, by less than the spare buffer
            if needs == "lattice":
                budget.budget_set(used() + 12 * MB)
                b = Lattice(abi.D2Q9, abi.F32, (EXT[0], EXT[1] - 200))
            elif needs == "batch":
                budget.budget_set(used() + 12 * MB)
                b = Batch(abi.D2Q9, abi.F32, [(EXT[0], EXT[1] // 16)] * 8)
            else:
                budget.budget_set(used() + 2 * MB)
                b = Net(32, 32, (8, 16, 16, 24), batch=4, capacity=16)
            assert used() > before - SPARE // 2
            b.close()
            assert used() - before < SPARE // 2  # it is gone
            budget.budget_set(4 << 30)
        a.step(37)
        m = a if has == "lattice" else a.members[3]
        out.append((m.get_populations(), *m.get_macros()))
        a.close()
    for x, y in zip(*out):
        assert np.array_equal(x, y)


if __name__ == "__main__":
    _main(*sys.argv[1:])
    print("ok")
