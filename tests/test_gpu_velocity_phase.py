"""GPU test of the sine and cosine of the spectral point velocity (sdc_amd/csrc/rbc_velocity.hip
sincos_turn): a state of one Fourier mode, on a box with L_x = 2 pi and at mid-height, whose other factors
are powers of two, so that w / k^2 is the cosine (or, for an imaginary coefficient, minus the sine) of the
phase and nothing else rounds.  Phases up to 1, 16 and 256 turns, the last as on a 1024-point grid.

Tolerance: a sine or cosine of size 1/2 to 1 rounds to within 2^-25 = 3.0e-8; the reduced argument, its square and
the polynomial's largest coefficient times it add at most 2^-25 of 0.3 each, 2.6e-8 together: 5.6e-8.
The root mean square of a rounding is its bound over sqrt(3), less where values are small: 1.6e-8.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

F = np.float32
TWO_PI = 2 * np.pi


@pytest.mark.parametrize("M,N,i", [(16, 16, 1), (64, 64, 16), (1024, 16, 256)])
def test_phase_of_one_mode(M, N, i):
    print(f"case: phase of mode {i}, {M}x{N}", flush=True)
    from sdc_amd import Stepper
    n = 1 << 18
    x = (np.random.default_rng(i).random(n) * TWO_PI).astype(F)
    q = x / F(TWO_PI)
    phase = F(i) * (q - np.floor(q))  # as the kernel forms it: exact or one rounding
    with Stepper(M, N, 1, TWO_PI, TWO_PI, 1e4, 0.7, 1e-4, precision="f32") as G:
        def w(c, at):
            st = [np.zeros((1, N, M // 2 + 1), complex) for _ in range(3)] + [np.zeros(1, complex) for _ in range(2)]
            st[1][0, 0, i] = c
            G.set_state(*st)
            z = np.zeros(len(at), F)
            return G.velocity_at(at, z, z)[2]

        origin = np.zeros(1, F)
        k2 = F(i * i)
        c = k2 / w(1.0, origin)[0]
        near = [c]
        for way in (F(0), F(np.inf)):
            d = c
            for _ in range(8):
                d = np.nextafter(d, way)
                near.append(d)
        exact = [d for d in near if w(float(d), origin)[0] == k2]  # amplitude k^2 at phase 0
        assert exact
        for part, ref in ((1.0, np.cos(TWO_PI * phase.astype(float))), (1j, -np.sin(TWO_PI * phase.astype(float)))):
            e = w(float(exact[0]) * part, x).astype(float) / float(k2) - ref
            print("largest", np.abs(e).max(), "rms", np.sqrt((e * e).mean()))
            assert np.abs(e).max() < 5.6e-8
            assert np.sqrt((e * e).mean()) < 1.6e-8
