"""CF -> SF at the edges of the transform's dispatch: the direct sum (n = 2), one pass from its
smallest to its largest, with a last step of one, two and three stages, two passes at their smallest
and largest, three passes.  Against the cosine transform in long double.

A radix transform's error in the 2-norm is at most about (3 + 1) eps per doubling (a product with a
rounded root, an addition); the bound below adds the input's window and the scaling, 8 eps."""
import numpy as np
import pytest
import scipy.fft

import hawaiihybrid_amd as H

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    e = H.Engine(0)
    yield e
    e.close()


@pytest.mark.parametrize("logn", [1, 2, 3, 4, 5, 9, 10, 11, 12, 13, 16, 20, 21, 22])
def test_cf_to_sf_against_long_double(eng, logn):
    n, dt = 1 << logn, 200.0
    rng = np.random.default_rng(logn)
    cf = 1e-10 * rng.standard_normal(n)
    d = eng.torch.from_numpy(cf.copy()).cuda()
    nu, sf, _ = eng.cf_to_sf(d, dt)
    r = np.arange(n, dtype=np.longdouble) / n
    window = cf * (1 - r * r) ** 2
    atu, pi = 2.4188843265857e-17, np.pi
    tmax = n * dt
    scale = tmax / pi * atu * 8.4783536255e-30 ** 2 / (4.0 * pi * 8.8541878128e-12) / (2.0 * n)
    ref = scipy.fft.dct(window, type=3) * scale
    eps = np.finfo(float).eps / 2
    err = np.linalg.norm((sf.cpu().numpy() - ref).astype(float)) / np.linalg.norm(ref.astype(float))
    assert err < (4 * logn + 8) * eps
    assert np.max(np.abs(d.cpu().numpy() - window)) <= 8 * eps * np.abs(cf).max()
    nu_ref = np.arange(n) * pi / tmax / 2.99792458e10 / atu / 2.0 / pi
    assert np.allclose(nu.cpu().numpy(), nu_ref, rtol=8 * eps, atol=0)
