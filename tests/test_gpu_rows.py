"""The row kernel (one trajectory per 16-lane row: small requests and the tail of large ones) against
the lane kernel (one trajectory per lane): the same bits.

A job alone runs on the row kernel from its first step; beside a filler of 9000 trajectories in
the same call it starts on the lane kernel and, depending on its items, ends on either.  Every
item's row, length, status, right-hand-side count and energy drift, and the job's CF, must be equal
bit for bit: both kernels run the same expressions in the same order.  Sizes: one row, less and more
than a wavefront's four rows, more rows than wavefronts.

Beside a queue of more than three fills of the lane slots the orbiting items of a mixed pool stay on the
FP64 lane kernel: the same bits again.

An engine with graph-captured slices stays on the lane kernel at every size; against it, exact special values
of the initial conditions, the dipole series (Zimmermann's and PR/mu's), trajectories that end at a failed
sample or at the step limit."""
import numpy as np
import pytest

import hawaiihybrid_amd as H

pytestmark = pytest.mark.gpu

SYSTEMS = {"hear": (H.he_ar, 300.0, H.PESMIN_HEAR, 4.0), "co2ar": (H.co2_ar, 200.0, H.PESMIN_CO2AR, 4.0),
           "ch4co2": (H.ch4_co2, 300.0, H.PESMIN_CH4CO2, 4.75)}


@pytest.fixture(scope="module")
def eng():
    e = H.Engine(0)
    yield e
    e.close()


@pytest.mark.parametrize("which", ["hear", "co2ar", "ch4co2"])
@pytest.mark.parametrize("prec", [H.PREC_FP64, H.PREC_MIXED])
@pytest.mark.parametrize("n", [1, 3, 17, 1500])
def test_row_kernel_gives_the_lane_kernel_bits(eng, which, prec, n):
    make, T, pesmin, rmin = SYSTEMS[which]
    L = 1024 if n < 100 else 600
    # injected close in, so that the trajectories collide within the series
    smp = H.Sampler(H.IC_R0_INJECT, H.PAIR_FREE, T, rmin, 40.0, pesmin, 15.0)
    ic = H.sample_ics(make(), smp, 5, n + 9000)[0]
    x, filler = eng.to_device_soa(ic[:n]), eng.to_device_soa(ic[n:])
    p = H.cf_params(L, rtol=1e-10 if prec == H.PREC_MIXED else 1e-12, Rcut=20.0, precision=prec)
    alone, _ = eng.cf_run(make(), p, [x])
    a = eng.items(0, n, L, rows=True)
    beside, _ = eng.cf_run(make(), p, [x, filler])
    b = eng.items(0, n, L, rows=True)
    print(f"rows {which} prec {prec} n {n}: {int(a['nrhs'].sum())} right-hand sides", flush=True)
    assert a["nrhs"].sum() > 0
    for key in ("len", "status", "nrhs", "e_drift", "rows"):
        assert np.array_equal(a[key], b[key]), key
    assert np.array_equal(alone[0].cpu().numpy(), beside[0].cpu().numpy())


@pytest.fixture(scope="module")
def lane_eng():
    mp = pytest.MonkeyPatch()
    mp.setenv("HH_GRAPHS", "1")   # read at creation
    e = H.Engine(0)
    mp.undo()
    yield e
    e.close()


@pytest.mark.parametrize("which", ["hear", "co2ar", "ch4co2"])
@pytest.mark.parametrize("prec", [H.PREC_FP64, H.PREC_MIXED])
def test_angles_of_exactly_zero(eng, lane_eng, which, prec):
    """Azimuths of exactly 0 or equal to each other, with and without azimuthal momentum (a planar or aligned
    geometry): their sines are 0, and no equation of motion divides by them."""
    make, T, pesmin, rmin = SYSTEMS[which]
    L = 512
    smp = H.Sampler(H.IC_R0_INJECT, H.PAIR_FREE, T, rmin, 40.0, pesmin, 15.0)
    ic = H.sample_ics(make(), smp, 7, 8)[0]
    azimuths = {"hear": [0], "co2ar": [0, 6], "ch4co2": [0, 6, 12]}[which]
    ic[0:2, 0] = 0.0                    # Phi
    ic[1, 1] = 0.0
    for k in azimuths[1:]:
        ic[2:4, k] = 0.0                # a monomer's azimuth
        ic[3, k + 1] = 0.0
        ic[4:6, k] = ic[4:6, 0]         # the same azimuth
        ic[5, k + 1] = ic[5, 1]
    ic[6:8, azimuths] = 0.0             # in a plane
    ic[7, [k + 1 for k in azimuths]] = 0.0
    p = H.cf_params(L, rtol=1e-10 if prec == H.PREC_MIXED else 1e-12, Rcut=20.0, precision=prec)
    got = []
    for e in (eng, lane_eng):
        e.cf_run(make(), p, [e.to_device_soa(ic)])
        got.append(e.items(0, 8, L, rows=True))
    print(f"zero angles {which} prec {prec}: status {got[0]['status']} {got[1]['status']}", flush=True)
    assert np.all(got[1]["status"] == 0)
    for key in ("len", "status", "nrhs", "e_drift", "rows"):
        assert np.array_equal(got[0][key], got[1][key]), key


@pytest.mark.parametrize("which", ["co2ar", "ch4co2"])
def test_orbiting_items_beside_a_deep_queue(eng, which):
    """The same trajectories in a call of their own (their orbiting ones in FP64 on rows) and in front of a queue
    of four fills (on the lane kernel while the queue is deep, then on rows)."""
    make, T, pesmin, rmin = SYSTEMS[which]
    n, L = 3000, 512
    smp = H.Sampler(H.IC_R0_INJECT, H.PAIR_FREE, 150.0, rmin, 40.0, pesmin, 15.0)
    ic = H.sample_ics(make(), smp, 9, n)[0]
    x = eng.to_device_soa(ic)
    fill = x.repeat(1, -(-4 * 65536 // n)).contiguous()
    p = H.cf_params(L, rtol=1e-10, Rcut=20.0, precision=H.PREC_MIXED)
    alone, st = eng.cf_run(make(), p, [x])
    a = eng.items(0, n, L, rows=True)
    beside, std = eng.cf_run(make(), p, [x, fill])
    b = eng.items(0, n, L, rows=True)
    print(f"deep {which}: {st.n_orbit} of {n} orbiting, {std.launches} slices", flush=True)
    assert st.n_orbit > 0
    for key in ("len", "status", "nrhs", "e_drift", "rows"):
        assert np.array_equal(a[key], b[key]), key
    assert np.array_equal(alone[0].cpu().numpy(), beside[0].cpu().numpy())


def check_same(a, b):
    for key in ("len", "status", "nrhs", "e_drift", "rows"):
        assert np.array_equal(a[key], b[key]), key


@pytest.mark.parametrize("which,prec", [("hear", H.PREC_FP64), ("hear", H.PREC_MIXED), ("co2ar", H.PREC_FP64),
                                        ("co2ar", H.PREC_MIXED)])
def test_zimmermann_series(eng, lane_eng, which, prec):
    """Both halves of bound pairs, three dipole components a sample."""
    make, T, pesmin, rmin = SYSTEMS[which]
    n, L = 70, 96
    smp = H.Sampler(H.IC_REJECTION, H.PAIR_BOUND, 60.0, rmin, 40.0, pesmin, 0.0)
    ic = H.sample_ics(make(), smp, 3, n)[0]
    p = H.cf_params(L, rtol=1e-10 if prec == H.PREC_MIXED else 1e-12, halves=H.HALVES_BOTH, zimmermann=True, precision=prec)
    got = []
    for e in (eng, lane_eng):
        cf, _ = e.cf_run(make(), p, [e.to_device_soa(ic)])
        got.append((cf[0].cpu().numpy(), e.items(0, 2 * n, L, rows=True, zimmermann=True)))
    check_same(got[0][1], got[1][1])
    assert np.array_equal(got[0][0], got[1][0]) and np.any(got[0][0] != 0.0)


@pytest.mark.parametrize("which", ["hear", "co2ar"])
@pytest.mark.parametrize("prec", [H.PREC_FP64, H.PREC_MIXED])
def test_prmu_series(eng, lane_eng, which, prec):
    make, T, pesmin, rmin = SYSTEMS[which]
    L, nfreq, R0 = 512, 200, 12.0
    smp = H.Sampler(H.IC_R0_INJECT, H.PAIR_FREE, T, rmin, 40.0, pesmin, R0)
    ic = H.sample_ics(make(), smp, 37, 65)[0]
    p = H.PrmuParams(1e-10, 1e-10, 200.0, R0, L, nfreq, prec, 0, 0)
    a, b = [e.prmu(make(), p, e.to_device_soa(ic)) for e in (eng, lane_eng)]
    assert np.array_equal(a[0].cpu().numpy(), b[0].cpu().numpy()) and a[2] == b[2] > 0
    assert np.array_equal(np.asarray(a[1]), np.asarray(b[1]))


@pytest.mark.parametrize("prec", [H.PREC_FP64, H.PREC_MIXED])
def test_failed_samples_and_step_limits(eng, lane_eng, prec):
    """He-Ar pairs that come from 300 bohr and are sampled near their turning point next: the CF jumps by more than
    1e10 (status 3).  A limit of 5 steps between samples (status 4)."""
    n, L = 64, 8
    s = H.he_ar()
    v = 5.0e-4 * (1.0 + 0.004 * (np.arange(n) - n / 2))
    ic = np.zeros((n, 6))
    ic[:, 0], ic[:, 2], ic[:, 4], ic[:, 5] = 0.3, 1.1, 300.0, -s.mu * v
    ic[:, 1], ic[:, 3] = 0.4, 0.3
    jump = H.cf_params(L, rtol=1e-10, dt=146.0 / 5.0e-4, Rcut=400.0, precision=prec)
    smp = H.Sampler(H.IC_R0_INJECT, H.PAIR_FREE, 300.0, 4.0, 40.0, H.PESMIN_HEAR, 15.0)
    steps = H.cf_params(64, rtol=1e-12, dt=2000.0, Rcut=20.0, max_steps=5, precision=prec)
    for p, y, status in ((jump, ic, 3), (steps, H.sample_ics(s, smp, 5, n)[0], 4)):
        got = []
        for e in (eng, lane_eng):
            cf, _ = e.cf_run(s, p, [e.to_device_soa(y)])
            got.append((cf[0].cpu().numpy(), e.items(0, n, p.L, rows=True)))
        print(f"endings: status {np.bincount(got[0][1]['status'])}", flush=True)
        assert np.any(got[0][1]["status"] == status)
        check_same(got[0][1], got[1][1])
        assert np.array_equal(got[0][0], got[1][0])


@pytest.mark.parametrize("which", ["hear", "co2ar", "ch4co2"])
@pytest.mark.parametrize("prec", [H.PREC_FP64, H.PREC_MIXED])
@pytest.mark.parametrize("n", [1, 17, 700])
def test_rows_equal_the_lane_kernel_alone(eng, lane_eng, which, prec, n):
    """The same call on an engine that stays on the lane kernel: every compared item ran on it."""
    make, T, pesmin, rmin = SYSTEMS[which]
    L = 600
    smp = H.Sampler(H.IC_R0_INJECT, H.PAIR_FREE, T, rmin, 40.0, pesmin, 15.0)
    ic = H.sample_ics(make(), smp, 6, n)[0]
    p = H.cf_params(L, rtol=1e-10 if prec == H.PREC_MIXED else 1e-12, Rcut=20.0, halves=H.HALVES_BOTH, precision=prec)
    got = []
    for e in (eng, lane_eng):
        cf, _ = e.cf_run(make(), p, [e.to_device_soa(ic)])
        got.append((cf[0].cpu().numpy(), e.items(0, 2 * n, L, rows=True)))
    check_same(got[0][1], got[1][1])
    assert np.array_equal(got[0][0], got[1][0])
