"""Read-back of macroscopic fields and predictions: every value exactly, on both
sides of the size up to which the calling thread works alone, with slots used
once and several times over, with ragged last pieces, and from several threads."""
import threading

import numpy as np
import pytest

from lbm_mirror_amd import abi

pytestmark = pytest.mark.gpu


def _round_trip(lattice, storage, ext, seed):
    from lbm_mirror_amd.lattice import Lattice
    g = Lattice(lattice, storage, ext)
    rng = np.random.default_rng(seed)
    rho, u = rng.uniform(0.9, 1.1, g.N), rng.uniform(-0.1, 0.1, (g.D, g.N))
    g.set_macros(rho, u)
    r, v = g.get_macros()
    if storage != abi.F64:  # held in FP32
        rho, u = rho.astype(np.float32).astype(np.float64), u.astype(np.float32).astype(np.float64)
    g.close()
    return np.array_equal(r, rho) and np.array_equal(v, u)


@pytest.mark.parametrize("lattice,storage,ext", [
    (abi.D2Q9, abi.F32, (3, 3)), (abi.D2Q9, abi.F64, (97, 31)),
    (abi.D2Q9, abi.F32, (87381, 1)), (abi.D2Q9, abi.F32, (87382, 1)),  # 4 bytes to either side of 1 MiB
    (abi.D2Q9, abi.F32, (699050, 1)), (abi.D2Q9, abi.F32, (699051, 1)),  # and of 8 MiB
    (abi.D2Q9, abi.F32, (1023, 517)), (abi.D3Q19, abi.F64, (61, 67, 71)),
    (abi.D3Q19, abi.F16S, (257, 129, 131)), (abi.D3Q19, abi.F64, (129, 127, 131)),
])
def test_macros_round_trip(hip, lattice, storage, ext):
    assert _round_trip(lattice, storage, ext, 5)


def test_macros_from_several_threads(hip):
    ok = [False] * 4
    def run(i):
        ok[i] = all(_round_trip(abi.D2Q9, abi.F32, (700 + 37 * i, 500), 10 * i + k) for k in range(4))
    th = [threading.Thread(target=run, args=(i,)) for i in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert all(ok)


@pytest.mark.parametrize("H,W,batch,count", [(24, 40, 3, 7), (200, 248, 4, 5)])
def test_prediction_is_the_scaled_output(hip, H, W, batch, count):
    from lbm_mirror_amd.warmstart import Net
    net = Net(H, W, (8, 8, 8, 8), batch=batch, seed=3)
    rng = np.random.default_rng(6)
    flags = [rng.integers(1, 5, H * W).astype(np.uint8) for _ in range(count)]
    um, tau = rng.uniform(0.02, 0.08, count), rng.uniform(0.6, 1.0, count)
    rho, u = net.predict(flags, um, tau)
    mu, sd = (a.astype(np.float64) for a in net.output_scale())
    for k in range(count):
        y = net.forward_raw(net.features(flags[k].reshape(H, W), um[k], tau[k])[None]).reshape(-1, 3).astype(np.float64)
        v = y * sd + mu
        fluid = flags[k] >= 2
        assert np.array_equal(u[k, 0], np.where(fluid, v[:, 0] * um[k], 0.0))
        assert np.array_equal(u[k, 1], np.where(fluid, v[:, 1] * um[k], 0.0))
        assert np.array_equal(rho[k], np.where(fluid, 1.0 + v[:, 2] * (3.0 * um[k] * um[k]), 1.0))
