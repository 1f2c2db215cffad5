"""GPU test of the penalization's transforms (sdc_amd/csrc/rbc_kernels.hip k_pen_fields, k_rows_mask_w,
k_rows_mask, k_pen_combine) against the oracle's pairwise summands at every row length, at L around the
kernels' runs of 16 modes and at mode counts that are no multiple of a block's 64.

Tolerance: as the other penalization tests, 1e-12 (FP64) and 2e-5 (FP32) of the largest entry.
"""
import numpy as np
import pytest

from oracle import oracle as O
from sdc_amd.initial import kept_mask
from tests.helpers import random_state, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,L", [(8, 8, 3), (16, 8, 17), (16, 16, 16), (32, 64, 33), (64, 16, 15), (128, 16, 5),
                                   (256, 32, 18), (512, 16, 2), (1024, 8, 3)])
def test_penalized_nonlinear_term_vs_oracle(M, N, L):
    from sdc_amd import Stepper
    cfg = (M, N, L, 4.0, 2.7, 2e4, 0.7, 2e-4)
    st = random_state(M, N, L, seed=M + L, amp=1e-2, decay=0.05)
    keep = kept_mask(M, N)
    o = O.Stepper(*cfg, nthreads=8)
    o.set_penalization(0.05, "circle")
    ref = o.nonlinear(*st)
    o.close()
    for precision, tol in (("f64", 1e-12), ("f32", 2e-5)):
        if precision == "f64" and M > 512:
            continue  # beyond the FP64 row limit
        print(f"case: penalization {precision} {M}x{N}x{L}", flush=True)
        with Stepper(*cfg, precision=precision) as S:
            S.set_penalization(0.05, "circle")
            out = S.calculate_nonlinear(*st)
        for i, (a, b) in enumerate(zip(out, ref)):
            a, b = (x[:, keep] if x.ndim == 3 else x for x in (a, b))
            if np.abs(b).max() > 0:
                assert rel_err(a, b) < tol, (i, rel_err(a, b))
