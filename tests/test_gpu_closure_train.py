"""GPU test of the training kernels (sdc_amd/csrc/rbc_closure.hip k_mlp_train, k_grad_finish) against
the FP64 oracle (oracle/closure.py) at the sizes where their split can go wrong: one point, around
one 32-point group, fewer groups than blocks, all blocks with a ragged last group, and several
groups per wave.

Tolerance: a hidden value carries the FP32 rounding of a 64-term dot product (64 * 2^-24 * |terms|,
terms below 0.3 on average) and 1e-7 of the hardware exponential, about 1e-6 together; two layers and
their derivatives give at most a few of those per point, and the mean over points adds none:
2e-5 of the largest gradient entry, and 1e-5 relative for the loss.
"""
import numpy as np
import pytest

from oracle import closure as C

pytestmark = pytest.mark.gpu


def _net(n):
    rng = np.random.default_rng(n)
    w = (rng.uniform(-1, 1, C.NW) * 0.3).astype(np.float32)
    norm = (rng.normal(size=8).astype(np.float32), rng.uniform(0.5, 2, 8).astype(np.float32),
            rng.uniform(0.5, 3, 3).astype(np.float32))
    return w, norm, rng.standard_normal((n, C.NIN)).astype(np.float32), rng.standard_normal((n, 3)).astype(np.float32)


@pytest.mark.parametrize("n", [1, 31, 32, 33, 4000, 65536 + 7, 150001])
def test_gradient_at_group_edges(n):
    print(f"case: closure gradient n={n}", flush=True)
    from sdc_amd import Closure, Stepper
    w, norm, X, Y = _net(n)
    with Stepper(32, 32, 4, 4.0, 4.0, 3e4, 0.7, 2e-4, precision="f32") as S:
        cl = Closure(S, capacity_points=0)
        cl.set_weights(w)
        cl.set_normalization(*norm)
        g, loss = cl.gradient(X, Y)
        cl.close()
    lr, gr = C.loss_and_grad(C.bf16_round(w).astype(np.float64), norm, X, Y)
    assert abs(loss - lr) < 1e-5 * lr
    assert np.abs(g - gr).max() < 2e-5 * np.abs(gr).max(), np.abs(g - gr).max() / np.abs(gr).max()
