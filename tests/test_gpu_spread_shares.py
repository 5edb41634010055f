"""Spreading in float64 with one launch (4 levels) and two (5 levels: 3 and 2, 8 levels: 4 and 4),
with the points of few blocks shared between wavefronts (radius 1.5) and without (30): every
pixel of every level against the float64 direct sum, within what the points' 32-bit offsets and
the float32 image allow.

Bound: an offset below 16 cells is off by at most 4.8e-7 cells, of at most pi / 2 of phase, in
each of the three axes: 2.3e-6 of the sum of the values' moduli, in which the kernel's 1e-9 is
lost; the image is returned in float32, 6.0e-8 of the pixel."""
import math

import numpy as np
import pytest

import bipp_amd
from bipp_amd import synthetic
from oracle import bipp_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("radius", [1.5, 30.0])
@pytest.mark.parametrize("levels", [4, 5, 8])
def test_spread_shares(ctx, levels, radius):
    r = np.random.default_rng(levels)
    n, n_s = 24, 30
    src, flux = synthetic.zenith_cap_sources(r, 12, 5.0)
    p0 = synthetic.disk_positions(r, n, 1.0) + np.array([0, 0, 0.3]) * r.normal(size=(n, 1))
    lmn = synthetic.make_lmn_grid(17, math.radians(40))
    samples = []
    for k in range(n_s):
        xyz = synthetic.rotate_x(p0 * radius, 0.02 * k)
        s = synthetic.visibilities(xyz, 1.0, src, flux, 0.1)
        samples.append(synthetic.Sample(0, 0, 1.0, xyz, s, np.ones(n, bool)))
    # level bounds between eigenvalues of the first sample, in the wider gaps
    d = np.sort(O.eigh_gram(1.0, samples[0].s, None, samples[0].xyz)[1])
    d = d[d > 0]
    gap = np.argsort(d[1:] / d[:-1])[::-1][:levels - 1]
    edge = [0.0] + [math.sqrt(d[g] * d[g + 1]) for g in np.sort(gap)] + [3e38]
    iv = np.array([[edge[i], edge[i + 1]] for i in range(levels)])
    syn = bipp_amd.NufftSynthesis(ctx, n, n, iv, lmn, compute="fp64", imager="nufft",
                                  tolerance=1e-9)
    syn.collect(np.ones(n_s), np.stack([s.s for s in samples]), np.stack([s.xyz for s in samples]))
    img = syn.images()
    ref = np.zeros((levels, lmn.shape[0]))
    moduli = np.zeros(levels)
    for smp in samples:
        v, dk, _, scale = O.eigh_gram(smp.wl, smp.s.astype(np.complex64), None, smp.xyz)
        wts = O.sample_level_weights(dk, float(scale), iv, "lsq")
        uvw = O.baselines_uvw(smp.xyz) * (2 * math.pi / smp.wl)
        for lvl in range(levels):
            vv = O.virtual_vis(1.0, wts[lvl], v.astype(np.complex128))
            ref[lvl] += O.nuft_sum(1.0, vv, uvw, lmn) / n_s
            moduli[lvl] += np.abs(vv).sum() / n_s
    ratio = [float((np.abs(img[k] - ref[k]) / (2.3e-6 * moduli[k] + 6.0e-8 * np.abs(ref[k]))).max())
             for k in range(levels)]
    print(f"grid {syn.nufft_grid()}: shares of the bound {ratio}", flush=True)
    assert np.all(moduli > 0) and max(ratio) <= 1
