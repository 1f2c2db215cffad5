"""GPU test of the parity-folded vertical transforms (sdc_amd/csrc/rbc_vertical.hip) above 32 vertical modes on
grids that take their other launch shapes: the projection with two waves and with one wave per 16 modes
(tests on small grids take four), both 32-mode halves, and the evaluation with all parts in one wave.
Against the plain VALU sums (RBC_NO_MFMA=1 at creation), which the small-grid tests hold to the FP64 oracle.

Tolerance: as the other nonlinear-term tests, 1e-11 of the largest entry in FP64 and 2e-5 in FP32."""
import os

import numpy as np
import pytest

from sdc_amd.initial import kept_mask
from tests.helpers import random_state, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("M,N,L", [(256, 128, 33), (512, 256, 40), (512, 512, 34)])
def test_nonlinear_term_against_plain_sums(precision, M, N, L):
    print(f"case: large vertical {precision} {M}x{N}x{L}", flush=True)
    from sdc_amd import Stepper
    cfg = (M, N, L, 3.3, 4.1, 2e4, 0.7, 2e-4)
    st = random_state(M, N, L, seed=L, amp=1e-2, decay=0.05)
    with Stepper(*cfg, precision=precision) as S:
        out = S.calculate_nonlinear(*st)
    os.environ["RBC_NO_MFMA"] = "1"
    try:
        with Stepper(*cfg, precision=precision) as S:
            ref = S.calculate_nonlinear(*st)
    finally:
        del os.environ["RBC_NO_MFMA"]
    keep = kept_mask(M, N)
    assert any(not np.array_equal(a, b) for a, b in zip(out, ref))
    for i, (a, b) in enumerate(zip(out, ref)):
        a, b = (x[:, keep] if x.ndim == 3 else x for x in (a, b))
        assert rel_err(a, b) < (1e-11 if precision == "f64" else 2e-5), (i, rel_err(a, b))
