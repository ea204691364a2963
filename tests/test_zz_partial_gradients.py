"""The network's memory for partial weight gradients: taken by the first
gradient, not by a network that only predicts; and of one layer at a time where
there is too little for all, with the same gradients."""
import ctypes as C
import os
import subprocess
import sys

import pytest

from test_zz_spare_memory import HERE, small_gpu  # noqa: F401


@pytest.mark.gpu
def test_partial_gradients(small_gpu):  # noqa: F811
    r = subprocess.run([sys.executable, os.path.abspath(__file__), small_gpu], capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0 and r.stdout.endswith("ok\n"), r.stdout + r.stderr


def _main(so):
    budget = C.CDLL(so, mode=C.RTLD_GLOBAL)  # before the library
    budget.budget_set.argtypes = [C.c_size_t]
    budget.budget_used.restype = C.c_size_t
    budget.budget_set(8 << 30)
    sys.path[:0] = [HERE, os.path.dirname(HERE)]
    import numpy as np
    from lbm_mirror_amd.warmstart import Net
    H, W, widths, B = 32, 64, (16, 32, 48, 64), 4
    rng = np.random.default_rng(4)
    x = rng.uniform(-1, 1, (B, H, W, 8)).astype(np.float32)
    t = rng.uniform(-1, 1, (B, H, W, 3)).astype(np.float32)
    m = (rng.random((B, H, W)) < 0.7).astype(np.float32)
    out, most = [], 8 << 30
    for _ in range(2):
        budget.budget_set(most)
        net = Net(H, W, widths, batch=B, seed=5)
        n1 = budget.budget_used()
        net.forward_raw(x)
        assert budget.budget_used() == n1
        out.append([net.loss_grad_raw(x, t, m) for _ in range(2)])
        n2 = budget.budget_used()
        assert n2 > n1
        out[-1].append(n2 - n1)
        net.close()
        most = n1 + (n2 - n1) // 2  # too little for all layers
    assert out[1][2] < out[0][2] // 2
    for (l0, g0), (l1, g1) in zip(out[0][:2], out[1][:2]):
        assert l0 == l1 and np.array_equal(g0, g1)


if __name__ == "__main__":
    _main(*sys.argv[1:])
    print("ok")
