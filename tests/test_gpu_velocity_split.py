"""GPU test of the vertical sums of the spectral point velocity (sdc_amd/csrc/rbc_velocity.hip
k_vel_points_mma), which run as products of BF16 parts: a state of the Fourier mode (1, 0) on a box with
L_x = 2 pi, read at x = 0 and at a quarter of the box, where the phase factors are 0 and 1 and the three
velocities are the real and imaginary parts of sum f C', sum f C and sum g S themselves.  Every L that takes
its own operand layout, odd ones and ones between the multiples of four and eight.

Tolerance, RBC_F32: no further from the exact sum of the FP32 operands than a chain of FP32 FMAs over the
same terms, in the root mean square over 20,000 heights; its sampling error is 1 / sqrt(40,000) = 0.5 %,
the bound ten of those.  RBC_BF16X3: two parts hold an operand to 2^-17 of it and leave a2 b2 < 2^-16 out, so
2^-15 of the sum of the terms' magnitudes.
"""
import numpy as np
import pytest

from oracle import velocity as V

pytestmark = pytest.mark.gpu

F = np.float32
M = N = 16
TWO_PI = 2 * np.pi
POINTS = 20000


def _sums(L, precision, seed):
    """The six sums as the GPU gives them, and per sum the FP32 coefficients and basis values."""
    from sdc_amd import Stepper
    r = np.random.default_rng(seed)
    z = r.uniform(-0.45, 0.45, POINTS).astype(F)
    f, g = ((r.standard_normal(L) + 1j * r.standard_normal(L)).astype(np.complex64) for _ in range(2))
    st = [np.zeros((L, N, M // 2 + 1), complex) for _ in range(3)] + [np.zeros(L, complex) for _ in range(2)]
    st[1][:, 0, 1], st[2][:, 0, 1] = f, g
    x0 = np.zeros(POINTS, F)
    with Stepper(M, N, L, TWO_PI, TWO_PI, 1e4, 0.7, 1e-4, precision=precision) as G:
        G.set_state(*st)
        at0 = G.velocity_at(x0, x0, z)
        at4 = G.velocity_at(x0 + F(TWO_PI) / F(4), x0, z)
    C, Cp, S = (b.astype(F) for b in V.basis(L, z.astype(np.float64)))
    out = [(-at0[0], f.imag, Cp), (at0[1], g.imag, S), (at0[2], f.real, C),
           (-at4[0], f.real, Cp), (at4[1], g.real, S), (-at4[2], f.imag, C)]
    return [(a.astype(float) / 2, c.astype(float), b.astype(float)) for a, c, b in out]  # kx != 0 counts twice


@pytest.mark.parametrize("L", [1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 15, 16, 17, 19, 22, 24, 25, 30, 31, 32])
def test_vertical_sums_no_further_off_than_fp32(L):
    print(f"case: vertical sums f32 L={L}", flush=True)
    worst = 0.0
    for seed in (1, 2):
        for got, c, b in _sums(L, "f32", 10 * L + seed):
            exact = c @ b
            chain = np.zeros(POINTS, F)
            for m in range(L):
                chain = (c[m] * b[m] + chain).astype(F)
            rms = [np.sqrt(np.mean((a - exact) ** 2)) for a in (got, chain.astype(float))]
            worst = max(worst, rms[0] / rms[1])
    print("largest ratio", worst)
    assert worst < 1.05


@pytest.mark.parametrize("L", [1, 2, 5, 7, 8, 11, 13, 16, 19, 23, 30])
def test_vertical_sums_bf16x3(L):
    print(f"case: vertical sums bf16x3 L={L}", flush=True)
    for got, c, b in _sums(L, "bf16x3", L):
        assert np.all(np.abs(got - c @ b) <= 2.0 ** -15 * (np.abs(c) @ np.abs(b)))


@pytest.mark.parametrize("k", [60, 84, 100, 112])
@pytest.mark.parametrize("L", [6, 11, 20, 31])
def test_velocity_of_a_state_times_a_power_of_two(L, k):
    """2^-k times a state of coefficients of size 1/2 to 2 has 2^-k times its velocity.  Products and sums scale
    exactly as long as they stay above 2^-126; a term of a sum that falls below is held to 2^-150, and at k = 112
    the 2 * 16 * 21 modes' terms, each below 2^-111 in a sum above 2^-109 in the root mean square, to 672 * 2^-150 < 2^-31 of it; the
    last steps round at 2^-24 again, three times: 2^-22 of the root mean square."""
    print(f"case: state times 2^-{k} L={L}", flush=True)
    from sdc_amd import Stepper
    from sdc_amd.initial import kept_mask
    m, n = 32, 64
    r = np.random.default_rng(L)
    keep = kept_mask(m, n)

    def field(shape):
        return r.uniform(0.5, 2, shape) * np.exp(2j * np.pi * r.random(shape))

    st = [field((L, n, m // 2 + 1)).astype(np.complex64).astype(complex) * keep for _ in range(3)]
    st += [r.uniform(0.5, 2, L).astype(np.float32).astype(complex) for _ in range(2)]
    x, y, z = ((r.random(1000) * s - o).astype(F) for s, o in ((4.0, 0.0), (3.0, 0.0), (0.9, 0.45)))
    with Stepper(m, n, L, 4.0, 3.0, 1e4, 0.7, 1e-4, precision="f32") as G:
        G.set_state(*st)
        one = [a.astype(float) for a in G.velocity_at(x, y, z)]
        G.set_state(*[a * 2.0 ** -k for a in st])
        small = [a.astype(float) * 2.0 ** k for a in G.velocity_at(x, y, z)]
    for a, b in zip(small, one):
        assert np.abs(a - b).max() <= 2.0 ** -22 * np.sqrt(np.mean(b * b)), np.abs(a - b).max()
