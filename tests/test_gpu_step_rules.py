"""The one-step kernels' default launch shapes, and the two-cells-per-thread
kernel at the ends of rows and wavefronts: bitwise what one cell per thread
through global addresses gives."""
import numpy as np
import pytest

from lbm_mirror_amd import abi
from test_gpu_tuning import _build, _state

pytestmark = pytest.mark.gpu

PAIR_WIDTHS = [2, 4, 126, 128, 130, 258]


@pytest.mark.parametrize("periodic", [0, 1, 7])
@pytest.mark.parametrize("nx", PAIR_WIDTHS)
@pytest.mark.parametrize("lat,st", [(abi.D2Q9, abi.F16S), (abi.D3Q19, abi.BF16S)])
def test_two_cells_per_thread(hip, lat, st, nx, periodic):
    from lbm_mirror_amd.lattice import Lattice
    ext = (nx, 3) if lat == abi.D2Q9 else (nx, 3, 3)
    a, b = _build([lambda l, s, e: Lattice(l, s, e)] * 2, lat, st, ext, 3 + nx)
    for s, form in ((a, (3, 3)), (b, (1, 1))):
        s.set_periodic(periodic)
        s.set_step_tuning(64, form)
        s.step(5)
    for p, q in zip(_state(a), _state(b)):
        assert np.array_equal(p, q, equal_nan=True)


@pytest.mark.parametrize("lat,st,ext", [
    (abi.D3Q19, abi.F16S, (64, 5, 4)), (abi.D3Q27, abi.BF16S, (71, 4, 3)),
    (abi.D3Q27, abi.F64, (64, 4, 3)), (abi.D3Q27, abi.F64, (65, 4, 3)), (abi.D3Q27, abi.F64, (300, 3, 3)),
    (abi.D3Q19, abi.F64, (97, 4, 3)), (abi.D3Q19, abi.F32, (256, 4, 3)), (abi.D3Q19, abi.F32, (257, 4, 3)),
    (abi.D3Q19, abi.F64, (341, 3, 3)), (abi.D3Q19, abi.F16S, (342, 3, 3))])
def test_default_shape(hip, lat, st, ext):
    from lbm_mirror_amd.lattice import Lattice
    a, b = _build([lambda l, s, e: Lattice(l, s, e)] * 2, lat, st, ext, 5)
    b.set_step_tuning(64, (1, 1))
    for s in (a, b):
        s.step(5)
    for p, q in zip(_state(a), _state(b)):
        assert np.array_equal(p, q)
