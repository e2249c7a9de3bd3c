"""The FP64 engines' reciprocals and quotients (Newton steps and a residual) have the division's bits, and its
limits: read out of Hamilton's equations, where they stand alone in a product or a sum.

* He-Ar with mu = 1: dTheta/dt = pTheta (1/mu) (1/R) (1/R), products only.
* CH4-CO2 at theta = pi/2, psi = 0, pphi = ptheta = 0: dpsi/dt = ppsi / I3 + ppsi cos^2(theta) / I2, whose second
  term is 4e-33 of the first."""
import numpy as np
import pytest

import hawaiihybrid_amd as H

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    e = H.Engine(0)
    yield e
    e.close()


def rhs(eng, system, y):
    import torch
    return eng.eval(system, H.EVAL_RHS, torch.from_numpy(np.ascontiguousarray(y)).cuda()).cpu().numpy()


def values(n, lo, hi, seed):
    """n numbers between 2^lo and 2^hi, a quarter of them within 2^-36 of a power of two, where rounding is
    hardest"""
    rng = np.random.default_rng(seed)
    m = rng.integers(0, 1 << 52, n)
    m[: n // 8] &= 0xffff
    m[n // 8: n // 4] |= 0xfffffffff0000
    return np.ldexp(1.0 + m * 2.0 ** -52, rng.integers(lo, hi, n))


def test_reciprocals_have_the_divisions_bits(eng):
    n = 1 << 20
    s = H.he_ar()
    s.mu = 1.0
    y = np.ones((6, n))
    y[4] = values(n, 0, 12, 1)
    got = rhs(eng, s, y)[2]
    inv = 1.0 / y[4]
    assert np.array_equal(got, inv * inv)


@pytest.mark.parametrize("i3", [2.3e5, np.nextafter(2.0, 1.0), np.nextafter(1.0, 2.0), 4.0 / 3.0, 1.0e-3])
def test_quotients_have_the_divisions_bits(eng, i3):
    n = 1 << 18
    s = H.ch4_co2()
    s.I_rotor[1] = s.I_rotor[2] = i3
    y = np.zeros((16, n))
    y[2], y[4], y[8], y[14] = 1.0, 12.0, np.pi / 2, 1.0
    y[11] = values(n, -20, 20, 2)
    assert np.array_equal(rhs(eng, s, y)[10], y[11] / i3)


def test_limits(eng):
    """A division by 0 and a quotient beyond the largest number are infinite."""
    y = np.ones((6, 2))
    y[2] = [0.0, 1.0]          # sin(Theta) = 0
    y[4] = 12.0
    got = rhs(eng, H.he_ar(), y)
    assert np.all(np.isposinf(got[[0, 5], 0])) and np.all(np.isfinite(got[:, 1]))
    s = H.ch4_co2()
    s.I_rotor[2] = 1e-3
    y = np.zeros((16, 1))
    y[2], y[4], y[8], y[14], y[11] = 1.0, 12.0, np.pi / 2, 1.0, 1e308
    assert np.isposinf(rhs(eng, s, y)[10, 0])


def test_a_missing_moment_of_inertia_is_not_a_rotor_at_rest(eng):
    """CO2-Ar with I = 0: the rates of the rotor's angles are infinite and its trajectories fail."""
    s = H.co2_ar()
    s.I = 0.0
    y = np.ones((10, 1))
    y[4] = 12.0
    assert np.all(np.isposinf(rhs(eng, s, y)[[6, 8], 0]))
    smp = H.Sampler(H.IC_R0_INJECT, H.PAIR_FREE, 200.0, 4.0, 40.0, H.PESMIN_CO2AR, 15.0)
    ic = H.sample_ics(H.co2_ar(), smp, 5, 5)[0]
    eng.cf_run(s, H.cf_params(64, Rcut=20.0), [eng.to_device_soa(ic)])
    assert np.all(eng.items(0, 5, 64)["status"] != 0)
