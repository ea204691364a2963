"""HLBM's porosity and its sums N and D kept without a per-cell reset: after full
steps, moves between them (the stamped box is then not the next gather's) and a
porosity set from outside, every cell holds what HlbmReset, the gathers and the
stamps give (hlbm.hpp:28-308), checked against the oracle, which resets every
cell.  Heavy discs: the fluid's force, whose sums differ in order, moves none."""
import numpy as np
import pytest

from helpers import channel_flags_2d, make_particle
from lbm_mirror_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("st,n", [(abi.F64, 1), (abi.F32, 1), (abi.F32, 9)])
def test_hlbm_sweep_matches_reset(hip, orc, st, n):
    from lbm_mirror_amd.lattice import Lattice
    rng = np.random.default_rng(40 + n)
    ext = (130, 70)
    N = ext[0] * ext[1]
    g, o = Lattice(abi.D2Q9, st, ext), orc.Sim(abi.D2Q9, st, ext)
    _, Q, _, w, _ = orc.lattice(abi.D2Q9)
    f0 = np.outer(w, np.ones(N)) * (1 + 0.01 * rng.uniform(-1, 1, size=(Q, N)))
    parts = []
    for _ in range(n):
        r = rng.uniform(2.5, 7.0)
        xy = [rng.uniform(20, ext[0] - 20), rng.uniform(20, ext[1] - 20)]
        parts.append(make_particle(xy, r, 1.5, 2, st, vel=list(rng.uniform(-0.1, 0.1, 2)), mass=1e12, inertia=1e12))
    prm = abi.particle_params(k_n=0.0, zeta_n=0.0, sub_steps=1, eps=1.5, max_radius=7.0, walls=False,
                              coupling=abi.COUPLING_HLBM)
    for s in (g, o):
        s.set_flags(channel_flags_2d(*ext))
        s.set_periodic(1)
        s.set_operator(1, abi.op_desc(boundary=abi.BC_BOUNCE_BACK))
        for fl in (2, 3, 4):
            s.set_operator(fl, abi.op_desc(collision=abi.COLL_HLBM, tau=0.8))
        s.set_populations(f0)
        s.particles_set(parts, prm)
    o.match_gpu_arithmetic()
    tol = 1e-11 if st == abi.F64 else 1e-5
    for rnd, steps in enumerate((1, 3, 34, 1, 2)):
        for s in (g, o):
            s.step(steps)
        assert np.array_equal(g.get_porosity(), o.get_porosity()), rnd
        (ng, dg), (no_, do) = g.get_hlbm_sums(), o.get_hlbm()
        assert np.array_equal(dg, np.asarray(do).reshape(-1)), rnd
        assert np.allclose(ng, np.asarray(no_).reshape(2, -1), rtol=tol, atol=tol * 0.1), rnd
        for s in (g, o):  # up to 2 cells away from what the last stamp wrote
            for _ in range(20):
                s.integrate()
            if rnd == 2:
                s.set_porosity(np.full(N, 0.25))
    g.close()
