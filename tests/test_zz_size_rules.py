"""What the launches choose by size, pinned at sizes that reach each choice with
certainty: batches of more than 800,000 cells, in every storage and with
periodic members; one lattice of more than 2^20 cells, whose steps no graph
replays; and 16-bit populations beyond the last-level cache, where even rows
take two cells per thread.  Bit for bit what one-step launches in a shape set
by hand give."""
import numpy as np
import pytest

from helpers import c1_ops, c2_ops, channel_flags_2d, duct_flags_3d, parabolic_inlet
from lbm_mirror_amd import abi

pytestmark = pytest.mark.gpu


def _obstacles(flags, seed):
    flags = flags.copy()
    rng = np.random.default_rng(seed)
    flags[(flags == 2) & (rng.random(flags.size) < 0.02)] = 1
    return flags


def _equal(a, b):
    assert np.array_equal(a.get_populations(), b.get_populations())
    for x, y in zip(a.get_macros(), b.get_macros()):
        assert np.array_equal(x, y) and np.all(np.isfinite(x))


@pytest.mark.parametrize("st", [abi.F64, abi.F32, abi.F16S, abi.BF16S])
def test_batch_of_many_cells(hip, st):
    from lbm_mirror_amd.lattice import Batch
    exts = [(701, 403), (56, 1000), (1000, 60), (640, 480), (513, 517)]  # 970,924 cells
    out = []
    for one in (False, True):
        b = Batch(abi.D2Q9, st, exts)
        for i, (m, ext) in enumerate(zip(b.members, exts)):
            m.set_flags(_obstacles(channel_flags_2d(*ext), i))
            m.set_periodic(i % 4)
            ops = c1_ops(0.8, 0.05)
            if i % 2:  # a closed, driven channel
                ops[3] = ops[4] = ops[2] = abi.op_desc(collision=abi.COLL_BGK_GUO, tau=0.7, vec=(1e-5, 2e-6, 0.0))
            for fl, op in ops.items():
                m.set_operator(fl, op)
            m.set_boundary_velocity(parabolic_inlet(*ext, 0.05))
            m.init_equilibrium(1.0, (0.0, 0.0))
        if one:
            b.set_tuning(256, 1, 0)
        b.step(14)  # a pair of launches of 4 steps, one of 2 and two single steps
        b.step(27)
        out.append(b)
    for x, y in zip(out[0].members, out[1].members):
        _equal(x, y)
    for b in out:
        b.close()


@pytest.mark.parametrize("st", [abi.F32, abi.BF16S])
def test_lattice_without_a_step_graph(hip, st):
    from lbm_mirror_amd.lattice import Lattice
    ext = (1301, 907)  # 1,180,007 cells
    out = []
    for one in (False, True):
        s = Lattice(abi.D2Q9, st, ext)
        s.set_flags(_obstacles(channel_flags_2d(*ext), 7))
        for fl, op in c1_ops(0.8, 0.05).items():
            s.set_operator(fl, op)
        s.set_boundary_velocity(parabolic_inlet(*ext, 0.05))
        s.init_equilibrium(1.0, (0.0, 0.0))
        if one:
            s.set_step_tuning(64)
        s.step(39)
        s.step(40)
        out.append(s)
    _equal(*out)
    for s in out:
        s.close()


@pytest.mark.parametrize("periodic", [1, 0])
def test_16_bit_populations_beyond_the_cache(hip, periodic):
    from lbm_mirror_amd.lattice import Lattice
    ext = (256, 168, 170)  # 277.8 MB of populations
    out = []
    for one in (False, True):
        s = Lattice(abi.D3Q19, abi.F16S, ext)
        s.set_flags(_obstacles(duct_flags_3d(*ext), 9))
        s.set_periodic(periodic)
        for fl, op in c2_ops(0.6, 1e-4).items():
            s.set_operator(fl, op)
        s.init_equilibrium()
        if one:
            s.set_step_tuning(256, (1, 1))
        s.step(9)
        out.append(s)
    _equal(*out)
    for s in out:
        s.close()
