"""GPU test of RBC_GENERIC_FFT=1 where the velocity grid, the penalization and the closure's features have register
transforms of their own: the switch changes the kernels (the rounding differs) and nothing else.

Tolerance: as the other group-against-generic test, 2e-5 of the largest entry in FP32, 1e-12 in FP64."""
import os

import numpy as np
import pytest

from sdc_amd.initial import kept_mask
from tests.helpers import random_state

pytestmark = pytest.mark.gpu


def _both(call):
    group = call()
    os.environ["RBC_GENERIC_FFT"] = "1"
    try:
        return group, call()
    finally:
        del os.environ["RBC_GENERIC_FFT"]


def _close(group, generic, tol):
    assert any(not np.array_equal(a, b) for a, b in zip(group, generic))
    for a, b in zip(group, generic):
        assert np.abs(a - b).max() <= tol * np.abs(b).max()


@pytest.mark.parametrize("M,N", [(16, 512), (64, 16), (512, 128), (1024, 32)])
def test_velocity_grid(M, N):
    print(f"case: generic switch, velocity grid {M}x{N}", flush=True)
    from sdc_amd import Stepper
    L = 4
    with Stepper(M, N, L, 4.0, 3.0, 1e4, 0.7, 1e-4, precision="f32") as S:
        S.set_state(*random_state(M, N, L, seed=M, amp=1e-2, decay=0.05))
        _close(*_both(lambda: S.velocity_grid([-0.3, 0.05, 0.4])), 2e-5)


@pytest.mark.parametrize("precision,M,N", [("f32", 32, 64), ("f32", 1024, 16), ("f64", 64, 32), ("f64", 512, 16)])
def test_penalized_nonlinear_term(precision, M, N):
    print(f"case: generic switch, penalization {precision} {M}x{N}", flush=True)
    from sdc_amd import Stepper
    L = 3
    keep = kept_mask(M, N)
    st = random_state(M, N, L, seed=M, amp=1e-2, decay=0.05)
    with Stepper(M, N, L, 4.0, 2.7, 1e4, 0.7, 1e-4, precision=precision) as S:
        S.set_penalization(0.05, "circle")
        group, generic = _both(lambda: [a[:, keep] if a.ndim == 3 else a for a in S.calculate_nonlinear(*st)])
    _close(group, generic, 1e-12 if precision == "f64" else 2e-5)


@pytest.mark.parametrize("M,N", [(64, 32), (128, 64), (32, 512)])
def test_closure_features(M, N):
    print(f"case: generic switch, closure features {M}x{N}", flush=True)
    from sdc_amd import Closure, Stepper
    L = 4
    with Stepper(M, N, L, 4.0, 4.0, 1e4, 0.7, 1e-4, precision="f32") as S, \
            Stepper(2 * M, 2 * N, L, 4.0, 4.0, 1e4, 0.7, 1e-4, precision="f32") as fine:
        fine.set_state(*random_state(2 * M, 2 * N, L, seed=M, amp=1e-2, decay=0.05))
        cl = Closure(S, nz=8, capacity_points=2 * M * N * 8)
        group, generic = _both(lambda: cl.points(fine)[:1])
        cl.close()
    _close(group, generic, 2e-5)
