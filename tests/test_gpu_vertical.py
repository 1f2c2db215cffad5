"""GPU test of the parity-folded vertical transforms (sdc_amd/csrc/rbc_vertical.hip): the nonlinear term
against the FP64 oracle at vertical resolutions around the kernels' edges (one k-step of 8 modes,
odd L, the 32-mode halves of the projection, the largest L), with the smallest exact rule and with an odd
number of levels (the middle level is its own mirror), on a grid whose mode count is not a multiple
of a wave's 16.

Tolerance: as the other nonlinear-term tests, 1e-11 of the largest entry in FP64 (sums of up to 200
levels at 1e-16 with the k^2 weights' cancellation) and 2e-5 in FP32.
"""
import numpy as np
import pytest

from oracle import oracle as O
from sdc_amd.initial import kept_mask
from tests.helpers import random_state, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("L,odd", [(1, 0), (2, 1), (7, 0), (8, 1), (9, 0), (16, 0), (17, 1), (32, 0), (33, 0), (40, 1)])
def test_nonlinear_vs_oracle(prec, L, odd):
    print(f"case: vertical {prec} L={L} odd={odd}", flush=True)
    import sdc_amd
    M, N = 32, 16
    cfg = (M, N, L, 3.3, 4.1, 2e4, 0.7, 2e-4)
    st = random_state(M, N, L, seed=L, amp=1e-2, decay=0.05)
    keep = kept_mask(M, N)
    nq = 0
    if odd:
        with sdc_amd.Stepper(*cfg, precision=prec) as G:
            nq = G.nq + 1
    with sdc_amd.Stepper(*cfg, precision=prec, nq=nq) as G:
        out = G.calculate_nonlinear(*st)
    ref = O.Stepper(*cfg, nthreads=8).nonlinear(*st)
    tol = 1e-11 if prec == "f64" else 2e-5
    for i, (a, b) in enumerate(zip(out, ref)):
        if L == 1 and i >= 3:
            continue  # <uw, S'_1> vanishes by symmetry: both sides hold rounding noise
        a, b = (x[:, keep] if x.ndim == 3 else x for x in (a, b))
        assert rel_err(a, b) < tol, (i, rel_err(a, b))
