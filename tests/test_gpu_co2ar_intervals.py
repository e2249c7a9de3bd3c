"""The CO2-Ar surfaces at the edges of their radial intervals (the lookup at 4 R): exactly on every
breakpoint, one unit below it, below the first and beyond the last, against the oracle's chain of
comparisons.  Energies to 1e-11 relative and Hamilton's equations to 1e-9, the bounds of
test_batched_surfaces_match_oracle."""
import numpy as np
import pytest

import hawaiihybrid_amd as H
import oracle_lib as O

pytestmark = pytest.mark.gpu

BOUNDS = np.concatenate([np.arange(4.5, 10.01, 0.25), [11.0, 12.0, 14.0, 16.0, 18.0, 20.0, 25.0, 30.0]])


@pytest.mark.parametrize("where", ["on", "below", "outside"])
def test_surfaces_at_interval_edges(where):
    R = {"on": BOUNDS, "below": np.nextafter(BOUNDS, 0.0), "outside": np.array([4.2, 4.4, 30.5, 41.0, 300.0])}[where]
    n = len(R)
    rng = np.random.default_rng(n)
    y = np.zeros((n, 10))
    y[:, [0, 6]] = rng.uniform(0, 2 * np.pi, (n, 2))
    y[:, [2, 8]] = np.arccos(rng.uniform(-0.95, 0.95, (n, 2)))
    y[:, 1::2] = rng.standard_normal((n, 5)) * 20.0
    y[:, 4] = R
    eng = H.Engine(0)
    yd = eng.to_device_soa(y)
    V = eng.eval(H.co2_ar(), H.EVAL_PES, yd).cpu().numpy()[0]
    D = eng.eval(H.co2_ar(), H.EVAL_DIPOLE, yd).cpu().numpy()
    F = eng.eval(H.co2_ar(), H.EVAL_RHS, yd).cpu().numpy()
    L = O.lib()
    for i in range(n):
        q = np.ascontiguousarray(y[i, 0::2])
        v = L.orc_pes(O.co2ar(), O.ptr(q))
        assert abs(V[i] - v) <= 1e-11 * abs(v) + 1e-16
        mu, f = np.zeros(3), np.zeros(10)
        L.orc_dipole(O.co2ar(), O.ptr(q), O.ptr(mu))
        assert np.allclose(D[:, i], mu, rtol=1e-11, atol=1e-16)
        L.orc_rhs(O.co2ar(), O.ptr(np.ascontiguousarray(y[i])), O.ptr(f))
        assert np.allclose(F[:, i], f, rtol=1e-9, atol=1e-15)
    eng.close()
