"""Several D2Q9 steps per launch against one-step launches, bit for bit: every
tile shape (chosen by the lattice's size), tile edges and remainders, lattices
smaller than a tile, periodic axes, every storage, and every operator that
may run there; step counts that use the long launches, the short ones and
single steps.  A launch shape set by hand runs every step on its own."""
import numpy as np
import pytest

from lbm_mirror_amd import abi
from helpers import c4_member

pytestmark = pytest.mark.gpu

# 24 x 24 cells and their multiples are whole tiles of the smaller shapes
EXTENTS = [(1, 1), (7, 3), (24, 8), (25, 9), (130, 47),  # the shape for the fewest cells
           (337, 161),                                    # up to 100,000 cells
           (600, 330),                                    # up to 800,000
           (1125, 769)]                                   # above
STEPS = (1, 46, 3, 20)


def _mixture(rng, ext, cell_force):
    nx, ny = ext
    ops = {1: abi.op_desc(boundary=abi.BC_BOUNCE_BACK),
           2: abi.op_desc(collision=abi.COLL_BGK, tau=0.8),
           3: abi.op_desc(boundary=abi.BC_ZOUHE_VELOCITY_X, collision=abi.COLL_BGK, east=1, tau=0.8),
           4: abi.op_desc(boundary=abi.BC_ZOUHE_PRESSURE_X, collision=abi.COLL_BGK, east=0, tau=0.8,
                          ramp=(1.0, 1e-4, 1.003, 30)),
           5: abi.op_desc(collision=abi.COLL_BGK_GUO, tau=0.7, vec=(1e-5, -2e-5, 0.0),
                          flags=abi.OPF_GUO_CELL_FORCE if cell_force else 0),
           6: abi.op_desc(boundary=abi.BC_EQUILIBRIUM, rho_eq=1.001, vec=(0.01, 0.0, 0.0)),
           7: abi.op_desc(boundary=abi.BC_ANTI_BOUNCE_BACK),
           8: abi.op_desc(),
           9: abi.op_desc(boundary=abi.BC_BOUNCE_BACK, collision=abi.COLL_BGK, tau=0.9)}
    flags = np.full((ny, nx), 2, np.uint8)
    flags[:, : max(1, nx // 3)] = 5
    few = rng.random((ny, nx)) < 0.02
    flags[few] = rng.choice([1, 1, 6, 7, 8, 9, 40], size=int(few.sum()))
    flags[0, :] = flags[-1, :] = 1
    flags[1:-1, 0] = 3
    flags[1:-1, -1] = 4
    return flags.reshape(-1), ops


def _lattice(ext, st, periodic, cell_force, one_step):
    from lbm_mirror_amd.lattice import Lattice
    from oracle import oracle as orc
    rng = np.random.default_rng(5)
    N = ext[0] * ext[1]
    flags, ops = _mixture(rng, ext, cell_force)
    w = np.asarray(orc.lattice(abi.D2Q9)[3])
    s = Lattice(abi.D2Q9, st, ext)
    s.set_flags(flags)
    s.set_periodic(periodic)
    for k, o in ops.items():
        s.set_operator(k, o)
    s.set_boundary_velocity(0.02 * rng.uniform(-1, 1, size=(2, N)))
    s.set_force_field(1e-5 * rng.uniform(-1, 1, size=(2, N)))
    s.set_populations(np.outer(w, np.ones(N)) * (1 + 0.01 * rng.uniform(-1, 1, size=(9, N))))
    if one_step:
        s.set_step_tuning(64)
    return s


@pytest.mark.parametrize("ext", EXTENTS)
@pytest.mark.parametrize("st", [abi.F64, abi.F32, abi.F16S, abi.BF16S])
@pytest.mark.parametrize("periodic", [0, 1, 2, 3])
def test_multi_step_launches_are_bitwise_single_steps(hip, ext, st, periodic):
    a, b = (_lattice(ext, st, periodic, periodic == 1, one) for one in (False, True))
    for n in STEPS:
        for s in (a, b):
            s.step(n)
        fa, fb = a.get_populations(), b.get_populations()
        assert np.array_equal(fa, fb) and np.all(np.isfinite(fa))
        for x, y in zip(a.get_macros(), b.get_macros()):
            assert np.array_equal(x, y)
    for s in (a, b):
        s.close()


@pytest.mark.parametrize("graph", [0, 32, 50])
def test_residual_tracking_and_graphs(hip, graph):
    a, b = (_lattice((130, 47), abi.F32, 0, False, one) for one in (False, True))
    for s in (a, b):
        s.set_residual()
        s.set_step_graph(graph)
    for n in (40, 150, 2, 33, 101):
        for s in (a, b):
            s.step(n)
        assert a.residual() == b.residual()
        assert np.array_equal(a.get_populations(), b.get_populations())


@pytest.mark.parametrize("st", [abi.F64, abi.F32])
@pytest.mark.parametrize("count,side", [(3, 40), (12, 150), (6, 420)])
def test_batches(hip, st, count, side):
    from lbm_mirror_amd.lattice import Batch
    rng = np.random.default_rng(side)
    ms = [c4_member(rng, side // 2, side, r_range=(2.0, 8.0), tau_range=(0.6, 1.0)) for _ in range(count)]
    out = []
    for one in (False, True):
        b = Batch(abi.D2Q9, st, [m[0] for m in ms])
        for mem, (ext, flags, ops, bcu, _) in zip(b.members, ms):
            mem.set_flags(flags)
            for k, o in ops.items():
                mem.set_operator(k, o)
            mem.set_boundary_velocity(bcu)
            mem.init_equilibrium(1.0, (0.0, 0.0))
        if one:
            b.set_tuning(256, 1, 0)
        b.step(26)
        b.step(3)
        b.step(39)
        # members stop at different times: the work list shrinks
        steps, res = b.run(2e-3, 30, 120)
        out.append((steps, res, [m.get_populations() for m in b.members], [m.get_macros() for m in b.members]))
        b.close()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    for x, y in zip(out[0][2], out[1][2]):
        assert np.array_equal(x, y)
    for (r0, u0), (r1, u1) in zip(out[0][3], out[1][3]):
        assert np.array_equal(r0, r1) and np.array_equal(u0, u1)
