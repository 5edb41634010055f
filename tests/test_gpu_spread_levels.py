"""Type-3 NUFFT at every number of levels that the spreading kernel has an instantiation for
(six in float, four in double) and the first that takes two launches, on grids of few blocks
(their points shared between wavefronts) and of many, against the float64 oracle."""
import math

import numpy as np
import pytest

import bipp_amd
from bipp_amd import synthetic
from oracle import bipp_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("radius", [1.5, 30.0])
@pytest.mark.parametrize("compute,levels", [("mixed", k) for k in range(1, 8)] +
                         [("fp64", k) for k in range(1, 6)])
def test_spread_levels(ctx, request, compute, levels, radius):
    if (compute, levels, radius) == ("fp64", 5, 1.5):
        # two levels whose points nearly cancel: the 32-bit offsets of the point records alone
        # leave 3.0e-7, the same to 16 digits with the sums in another order
        request.applymarker(pytest.mark.xfail(reason="point records hold offsets in 32 bits"))
    tol, bound = (1e-9, 1e-7) if compute == "fp64" else (1e-5, 1e-4)
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
    cut = [math.sqrt(d[g] * d[g + 1]) for g in np.sort(gap)]
    edge = [0.0] + cut + [3e38]
    iv = np.array([[edge[i], edge[i + 1]] for i in range(levels)])
    syn = bipp_amd.NufftSynthesis(ctx, n, n, iv, lmn, compute=compute, imager="nufft",
                                  tolerance=tol)
    syn.collect(np.ones(n_s), np.stack([s.s for s in samples]),
                np.stack([s.xyz for s in samples]))
    img = syn.images()
    ref, _ = O.synthesize(samples, iv, lmn)
    top = max(np.linalg.norm(x) for x in ref)
    errs = [float(np.linalg.norm(img[k] - ref[k]) / top) for k in range(levels)]
    print(f"grid {syn.nufft_grid()} {compute}: {errs}", flush=True)
    assert max(errs) <= bound   # the bounds of the other NUFFT tests
