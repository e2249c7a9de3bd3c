"""N2-Ar PIP-NN surfaces on the device (hh_pipnn_*: BF16 matrix-core networks, FP32 features,
evaluated as deviations from the value at infinite separation) against the FP64 oracle on phase
points drawn by q_generator + p_generator at 100, 300 and 500 K (R in [4.51, 40] bohr).

Tolerances, from the errors measured on these (seeded, deterministic) points with a margin of
about 2: energy |dE| in cm^-1 over the set, dipole |dmu| relative to the largest |mu| of the set.
  split BF16 (3 products, the default and the mode for dynamics)
                           max |dE| <= 0.25,  median <= 1e-3;   max dmu <= 1e-3
  single BF16 product      median |dE| <= 1e-2, 99th percentile <= 4, |dE| / |E| <= 12% where
                           |E| > 100 cm^-1;   99th percentile of dmu <= 0.12
(Measured here: split median 2.4e-4, max 0.11 cm^-1, dipole 4.1e-4; single median 1.7e-3 cm^-1,
99th percentile 1.9 cm^-1, relative 6.2% above 100 cm^-1, dipole 99th percentile 0.062.
The single product's error has a heavy tail: its largest errors sit on the repulsive wall, where
the network's terms are large and cancel (38 cm^-1 on these 4200 points, 93 cm^-1 on 2000 of 2^20
points of the benchmark), and its dipole reaches ~10% of the largest |mu|, since the induced
dipole is a small difference of site charges times positions up to 40 bohr.  Its maximum grows
with the sample, so it is bounded by quantiles: a throughput mode, not a parity-grade surface.)
"""
import ctypes as C

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

HTOCM = 2.1947463136320e5


@pytest.fixture(scope="module")
def setup():
    import torch
    import hawaiihybrid_amd as H
    from hawaiihybrid_amd import n2ar
    eng = H.Engine(0)
    W = n2ar.load_weights()
    m, keep = O.n2ar_model(W, n2ar.PES_EN_INF)
    pts = np.concatenate([n2ar.phase_points(1400, T, seed=int(T)) for T in (100.0, 300.0, 500.0)])
    q = n2ar.lab_q(pts)                     # [5][n], n = 4200 (not a multiple of 64)
    ref_E = np.array([O.lib().orc_n2ar_pes(C.byref(m), O.ptr(np.ascontiguousarray(q[:, i]))) for i in range(q.shape[1])])
    ref_mu = np.zeros((3, q.shape[1]))
    mu = np.zeros(3)
    for i in range(q.shape[1]):
        O.lib().orc_n2ar_dipole(C.byref(m), O.ptr(np.ascontiguousarray(q[:, i])), O.ptr(mu))
        ref_mu[:, i] = mu
    qd = torch.from_numpy(q).to("cuda:0")
    return dict(eng=eng, W=W, q=q, qd=qd, ref_E=ref_E, ref_mu=ref_mu, n2ar=n2ar, keep=keep, m=m)


@pytest.mark.parametrize("prec", [0, 1])
def test_reference_surfaces_match_oracle(setup, prec):
    s = setup
    print(f"pipnn precision {prec}: {s['q'].shape[1]} points", flush=True)
    model = s["n2ar"].PipNN(s["eng"], precision=prec, weights=s["W"])
    E, mu, ms = model.eval(s["qd"])
    E = E.cpu().numpy()
    mu = mu.cpu().numpy()
    dE = np.abs(E - s["ref_E"]) * HTOCM
    scale = np.max(np.linalg.norm(s["ref_mu"], axis=0))
    dmu_pt = np.max(np.abs(mu - s["ref_mu"]), axis=0) / scale
    big = np.abs(s["ref_E"]) * HTOCM > 100.0
    rel_big = np.max(dE[big] / (np.abs(s["ref_E"][big]) * HTOCM))
    print(f"  |dE| cm^-1: median {np.median(dE):.3e}, p99 {np.quantile(dE, 0.99):.3e}, max {dE.max():.3e}, "
          f"max rel above 100 cm^-1 {rel_big:.3e}; |dmu|/max|mu| p99 {np.quantile(dmu_pt, 0.99):.3e}, "
          f"max {dmu_pt.max():.3e}; {ms:.3f} ms", flush=True)
    assert np.all(np.isfinite(E)) and np.all(np.isfinite(mu))
    if prec == 1:
        assert dE.max() < 0.25 and np.median(dE) < 1e-3
        assert dmu_pt.max() < 1e-3
    else:
        assert np.median(dE) < 1e-2 and np.quantile(dE, 0.99) < 4.0 and rel_big < 0.12
        assert np.quantile(dmu_pt, 0.99) < 0.12
    model.close()


@pytest.mark.parametrize("width", [64, 128])
@pytest.mark.parametrize("prec", [0, 1])
def test_synthetic_tanh_networks_match_oracle(setup, width, prec):
    """The benchmark's synthetic shape (17 -> 3 x width, tanh -> 1) on the same features."""
    s = setup
    n2ar = s["n2ar"]
    layers = n2ar.synthetic_pes(width)
    keep = []
    om = O.orc_mlp(layers, O.ACT_TANH, keep)
    layers_pes, xm, xs, _, _ = s["W"]["pes"]
    xm = np.ascontiguousarray(xm)
    xs = np.ascontiguousarray(xs)
    q = s["q"][:, :1000]
    ref = np.array([O.lib().orc_n2ar_mlp_on_pes_features(C.byref(om), O.ptr(xm), O.ptr(xs),
                                                          O.ptr(np.ascontiguousarray(q[:, i]))) for i in range(q.shape[1])])
    model = n2ar.PipNN(s["eng"], precision=prec, pes_layers=layers, pes_act=n2ar.ACT_TANH, with_dipole=False,
                       weights=s["W"])
    E, _, ms = model.eval(s["qd"][:, :1000].contiguous(), dipole=False)
    out = E.cpu().numpy() * HTOCM          # yscale = 1, ymean = en_inf = 0: E = out / HTOCM
    err = np.max(np.abs(out - ref)) / np.max(np.abs(ref))
    print(f"synthetic {width} prec {prec}: max rel err {err:.3e} ({ms:.3f} ms)", flush=True)
    assert err < (3e-2 if prec == 0 else 2e-4)
    model.close()


def test_rejects_unsupported_shape(setup):
    s = setup
    n2ar = s["n2ar"]
    import hawaiihybrid_amd as H
    with pytest.raises(H.HHError):
        n2ar.PipNN(s["eng"], pes_layers=n2ar.synthetic_pes(96), with_dipole=False, weights=s["W"])


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("n", [1, 31, 33, 63, 65])
def test_points_do_not_depend_on_their_neighbours(setup, prec, n):
    """Batches that end within a wavefront or one of its halves: the same bits as the same points of a
    large batch, at whatever lanes they fall there."""
    s = setup
    model = s["n2ar"].PipNN(s["eng"], precision=prec, weights=s["W"])
    E, mu, _ = model.eval(s["qd"])
    Ep, mup, _ = model.eval(s["qd"][:, 100:100 + n].contiguous())
    assert np.array_equal(Ep.cpu().numpy(), E[100:100 + n].cpu().numpy())
    assert np.array_equal(mup.cpu().numpy(), mu[:, 100:100 + n].cpu().numpy())


def _split(x):
    """x (float32) as a BF16 head and the BF16 of the rest, round to nearest even"""
    def bf16(v):
        u = v.astype(np.float32).view(np.uint32)
        return ((u + 0x7fff + ((u >> 16) & 1)) & np.uint32(0xffff0000)).view(np.float32)
    x = x.astype(np.float32)
    hi = bf16(x)
    return hi.astype(np.float64), bf16(x - hi).astype(np.float64)


def _split_product(start, x, W, dtype):
    """start + x W by the split mode's three products, summed in `dtype`"""
    xh, xl = (v.astype(dtype) for v in _split(x))
    Wh, Wl = (v.astype(dtype) for v in _split(W))
    return start.astype(dtype) + xh @ Wh + xh @ Wl + xl @ Wh


def _split_mode_dipole(W, q, dtype):
    """The split mode's dipoles: the operands of every product rounded to BF16 pairs; polynomials, the networks'
    sums and activations in `dtype`, the rest in 64 bits."""
    from hawaiihybrid_amd.data import gen_pip_n2ar as G
    Phi, Theta, R, p1, t1 = q
    u = np.array([np.sin(t1) * np.cos(p1), np.sin(t1) * np.sin(p1), np.cos(t1)])
    Rh = np.array([np.sin(Theta) * np.cos(Phi), np.sin(Theta) * np.sin(Phi), np.cos(Theta)])
    c = np.clip((u * Rh).sum(0), -1.0, 1.0)
    s = np.sqrt(np.maximum(1.0 - c * c, 0.0))
    ex = (u - c * Rh) * np.where(s > 1e-12, 1.0 / np.maximum(s, 1e-12), 0.0)
    a = 0.5 * 2.07856749
    o = np.zeros_like(R)
    site = [np.array(v) for v in ([a * s, a * c], [-a * s, -a * c], [a * c, -a * s], [-a * c, a * s], [o, R])]
    w = np.clip((R - 9.5) / 3.0, 0.0, 1.0)
    w = w ** 3 * (10.0 - 15.0 * w + 6.0 * w * w)
    mu = np.zeros((2, len(R)))
    for (subnets, xmean, xscale), a0, weight in zip(W["dip"], (2.0, 6.0), (1.0 - w, w)):
        y = [np.exp(-np.sqrt(((site[i] - site[j]) ** 2).sum(0)) / a0).astype(np.float32).astype(dtype)
             for i in range(5) for j in range(i + 1, 5)]
        off, charges = 0, []
        for layers, reps, gens in zip(subnets, G.DIP_REPS, G.DIP_GENS):
            (W1, b1), (W2, b2) = layers
            polys = G.expand(G.parse_reps(reps), 5, gens)
            p = np.array([sum((np.prod([y[k] for k in m], axis=0) for m in ms), o.astype(dtype)) for ms in polys]).T
            mean, scale = xmean[off:off + len(polys)], xscale[off:off + len(polys)]
            off += len(polys)
            silu = lambda z: z / (1.0 + np.exp(-z))
            z_ref = b1 - (mean / scale) @ W1
            x = p.astype(np.float32) * (1.0 / scale).astype(np.float32)
            h = silu(_split_product(z_ref, x, W1, dtype)) - silu(z_ref).astype(dtype)
            charges += list(_split_product(np.zeros(W2.shape[1]), h, W2, dtype).T)
        mu += weight * sum(qa * xz for qa, xz in zip(charges, site))
    return mu[1] * Rh + mu[0] * ex


def test_split_mode_rounds_the_standardised_features(setup):
    """The split mode's dipoles come from BF16 pairs of the network's own weights and of its standardised
    features p/scale.  Against the same operands with polynomials, sums and activations in 64 bits, in the 2-norm
    over the set.  The device computes those in FP32 (the charges cancel, so their last bits show), whose size
    numpy's FP32 gives, 1.9e-4: four times that, for another order of the sums and the hardware's exponential.
    Other operands (1/scale in the weights) are off by 2.6e-3."""
    s = setup
    model = s["n2ar"].PipNN(s["eng"], precision=1, weights=s["W"])
    mu = model.eval(s["qd"])[1].cpu().numpy()
    want = _split_mode_dipole(s["W"], s["q"], np.float64)
    err = np.linalg.norm(mu - want) / np.linalg.norm(want)
    fp32 = np.linalg.norm(_split_mode_dipole(s["W"], s["q"], np.float32) - want) / np.linalg.norm(want)
    print(f"split operands: {err:.2e}, FP32 sums {fp32:.2e}", flush=True)
    assert err < 4 * fp32
    model.close()
