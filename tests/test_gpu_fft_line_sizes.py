"""x lines of the type-3 NUFFT at lengths that a plan can have (twice an even 2^a 3^b 5^c), on both
sides of the lengths at which a workgroup takes 16, 8, 4 and 2 lines (256, 512, 1024, 2048) and of
the longest that the one-pass kernel takes (2048), small ones and ones with radices 10, 12 and
15, against the float64 oracle.  The array is stretched along x until the plan has the length."""
import math

import numpy as np
import pytest

import bipp_amd
from bipp_amd import synthetic
from oracle import bipp_oracle as O

pytestmark = pytest.mark.gpu

SIZES = [48, 60, 100, 180, 256, 288, 512, 540, 900, 1024, 1080, 1800, 2000, 2048, 2160, 3000]


@pytest.mark.parametrize("compute,length", [(c, n) for c in ("mixed", "fp64") for n in SIZES])
def test_line_sizes(ctx, compute, length):
    tol = 1e-5 if compute == "mixed" else 1e-9
    # mixed: the bound of the other NUFFT tests.  fp64: the points' offsets are held in 32 bits, half
    # a unit in the last place below 16 cells is 4.8e-7 cells of at most pi / 2 of phase: 7.5e-7
    bound = 1e-4 if compute == "mixed" else 7.5e-7
    r = np.random.default_rng(length)
    n = 9
    src, flux = synthetic.zenith_cap_sources(r, 5, 5.0)
    p0 = synthetic.disk_positions(r, n, 1.0) + np.array([0, 0, 0.3]) * r.normal(size=(n, 1))
    lmn = synthetic.make_lmn_grid(21, math.radians(20))
    # nf2 = smooth(2 smooth(4 / pi X S + w + 1)); X: half extent of 2 pi (p_a - p_b) over a > b
    w = math.ceil(math.log10(1 / tol)) + 1
    a, b = np.tril_indices(n)
    u = 2 * np.pi * (p0[a, 0] - p0[b, 0])
    xs = 0.5 * (u.max() - u.min()) * 0.5 * (lmn[:, 0].max() - lmn[:, 0].min())
    # a little below the wanted spread grid, which is the next even size up
    scale = (length / 2 - 0.25 - w - 1) / (4 / math.pi * xs)
    xyz = p0 * np.array([scale, 5.0, 2.0])
    s = synthetic.visibilities(xyz, 1.0, src, flux, 0.1)
    syn = bipp_amd.NufftSynthesis(ctx, n, n, [[0.0, 3e38]], lmn, compute=compute, imager="nufft",
                                  tolerance=tol)
    syn.collect(1.0, s, xyz)
    assert syn.nufft_grid()[0] == length
    ref, _ = O.synthesize([synthetic.Sample(0, 0, 1.0, xyz, s, np.ones(n, bool))],
                          np.array([[0.0, 3e38]]), lmn)
    err = O.rel_l2(syn.images()[0], ref[0])
    print(f"grid {syn.nufft_grid()} {compute}: rel L2 {err:.2e}", flush=True)
    assert err <= bound
