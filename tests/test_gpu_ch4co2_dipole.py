"""The CH4-CO2 dipole pass (products X_x Y_y shared by the functions of an (l_a, l_b) block) at the
edges of its 64-sample workgroups and of its radial intervals.

* FP64, hh_eval at 1, 63, 64, 65 and 130 points that include every interval's bounds and the tail
  beyond 30 bohr, against the oracle's term-by-term expansion: 1e-10 of the largest value (the bound of
  test_ch4co2_surfaces_match_oracle: FP64 sums of 31802 terms in another order and form).
* FP32, CF rows of 1, 63, 64 and 65 samples against the FP64 rows of the same trajectories, far from
  the well where the two integrations agree: FP32 carries 6e-8 per operation and the expansion's
  terms cancel by up to two orders, so 99 % of the samples agree to 1e-5 of mu(0)^2."""
import ctypes as C

import numpy as np
import pytest

import hawaiihybrid_amd as H
import oracle_lib as O

pytestmark = pytest.mark.gpu

BOUNDS = [5.0, 5.25, 5.5, 5.75, 6.0, 6.25, 6.5, 6.75, 7.0, 7.25, 7.5, 7.75, 8.0, 8.25, 8.5, 8.75, 9.0, 9.25, 9.5, 10.0,
          10.5, 11.0, 12.0, 14.0, 16.0, 18.0, 20.0, 25.0, 30.0]


@pytest.fixture(scope="module")
def eng():
    e = H.Engine(0)
    yield e
    e.close()


@pytest.mark.parametrize("n", [1, 63, 64, 65, 130])
def test_dipole_at_workgroup_and_interval_edges(eng, n):
    import torch
    rng = np.random.default_rng(n)
    y = np.zeros((16, n))
    y[[0, 6, 10, 12]] = rng.uniform(0, 2 * np.pi, (4, n))
    y[[2, 8, 14]] = np.arccos(rng.uniform(-0.97, 0.97, (3, n)))
    R = np.array(BOUNDS + [np.nextafter(b, 0) for b in BOUNDS] + [4.9, 33.0, 41.0])
    y[4] = np.resize(rng.permutation(R), n)
    got = eng.eval(H.ch4_co2(), H.EVAL_DIPOLE, torch.from_numpy(y).cuda()).cpu().numpy()
    s, m, want = O.ch4co2(), np.zeros(3), np.zeros((3, n))
    for i in range(n):
        O.lib().orc_dipole(C.byref(s), O.ptr(np.ascontiguousarray(y[0::2, i])), O.ptr(m))
        want[:, i] = m
    print(f"ch4co2 dipole n {n}: {np.max(np.abs(got - want)) / np.abs(want).max():.2e}", flush=True)
    assert np.max(np.abs(got - want)) < 1e-10 * np.abs(want).max()


@pytest.mark.parametrize("L", [1, 63, 64, 65])
def test_fp32_rows_match_fp64_rows(eng, L):
    smp = H.Sampler(H.IC_R0_INJECT, H.PAIR_FREE, 300.0, 4.75, 40.0, H.PESMIN_CH4CO2, 25.0)
    x = eng.to_device_soa(H.sample_ics(H.ch4_co2(), smp, 3, 70)[0])
    rows = []
    for prec in (H.PREC_MIXED, H.PREC_FP64):
        eng.cf_run(H.ch4_co2(), H.cf_params(L, rtol=1e-12, Rcut=40.0, precision=prec), [x])
        rows.append(eng.items(0, 70, L, rows=True)["rows"])
    d = np.abs(rows[0] - rows[1]) / rows[1][:, :1]
    print(f"ch4co2 rows L {L}: p99 {np.quantile(d, 0.99):.2e} max {d.max():.2e}", flush=True)
    assert np.quantile(d, 0.99) < 1e-5
