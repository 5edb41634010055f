"""Type-3 NUFFT on grids whose strided axes take the register passes of radices 10 and 12 (60,
100, 108, 120 points in one pass, 180 = 90 * 2, 200 = 100 * 2 and 240 = 120 * 2 in two), against
the float64 oracle.  The array is scaled until the plan has the wanted y length (twice an even
2^a 3^b 5^c)."""
import math

import numpy as np
import pytest

import bipp_amd
from bipp_amd import synthetic
from oracle import bipp_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("length", [48, 60, 100, 108, 120, 180, 200, 240])
def test_fft_lengths(ctx, length):
    compute, tol, bound = "mixed", 1e-5, 1e-4
    r = np.random.default_rng(length)
    n = 9
    src, flux = synthetic.zenith_cap_sources(r, 5, 5.0)
    p0 = synthetic.disk_positions(r, n, 1.0) + np.array([0, 0, 0.3]) * r.normal(size=(n, 1))
    lmn = synthetic.make_lmn_grid(21, math.radians(20))
    # nf2 = smooth(2 smooth(4 / pi X S + w + 1)); X: half extent of 2 pi (p_a - p_b) over a > b
    w = math.ceil(math.log10(1 / tol)) + 1
    a, b = np.tril_indices(n)
    u = 2 * np.pi * (p0[a, 1] - p0[b, 1])
    xs = 0.5 * (u.max() - u.min()) * 0.5 * (lmn[:, 1].max() - lmn[:, 1].min())
    for want in np.arange(length / 2, length / 2 - 12, -0.25):
        scale = (want - w - 1) / (4 / math.pi * xs)
        if scale <= 0:
            break
        xyz = p0 * scale
        s = synthetic.visibilities(xyz, 1.0, src, flux, 0.1)
        syn = bipp_amd.NufftSynthesis(ctx, n, n, [[0.0, 3e38]], lmn, compute=compute,
                                      imager="nufft", tolerance=tol)
        syn.collect(1.0, s, xyz)
        if syn.nufft_grid()[1] == length:
            break
    assert syn.nufft_grid()[1] == length
    ref, _ = O.synthesize([synthetic.Sample(0, 0, 1.0, xyz, s, np.ones(n, bool))],
                          np.array([[0.0, 3e38]]), lmn)
    err = O.rel_l2(syn.images()[0], ref[0])
    print(f"grid {syn.nufft_grid()} {compute}: rel L2 {err:.2e}", flush=True)
    assert err <= bound     # the bound of the other mixed NUFFT tests


@pytest.mark.parametrize("compute,length", [("mixed", 576), ("mixed", 600), ("mixed", 1152),
                                            ("mixed", 1200), ("mixed", 4800), ("mixed", 5000),
                                            ("mixed", 9600), ("mixed", 10000), ("fp64", 240),
                                            ("fp64", 288), ("fp64", 576), ("fp64", 600),
                                            ("fp64", 2400), ("fp64", 2500), ("fp64", 4800),
                                            ("fp64", 5000)])
def test_fft_axis_lengths(ctx, compute, length):
    """The y axis in one pass on both sides of the lengths at which its tile halves (16, 8, 4
    and 2 positions, then two passes), an array stretched along y."""
    tol = 1e-5 if compute == "mixed" else 1e-9
    # mixed: the bound of the other tests.  fp64: the points' offsets are held in 32 bits, half a
    # unit in the last place below 16 cells is 4.8e-7 cells of at most pi / 2 of phase: 7.5e-7
    bound = 1e-4 if compute == "mixed" else 7.5e-7
    r = np.random.default_rng(length)
    n = 9
    src, flux = synthetic.zenith_cap_sources(r, 5, 5.0)
    p0 = synthetic.disk_positions(r, n, 1.0) + np.array([0, 0, 0.3]) * r.normal(size=(n, 1))
    lmn = synthetic.make_lmn_grid(21, math.radians(20))
    w = math.ceil(math.log10(1 / tol)) + 1
    a, b = np.tril_indices(n)
    u = 2 * np.pi * (p0[a, 1] - p0[b, 1])
    xs = 0.5 * (u.max() - u.min()) * 0.5 * (lmn[:, 1].max() - lmn[:, 1].min())
    for want in np.arange(length / 2, length / 2 * 0.9 - 12, -length / 400):
        scale = (want - w - 1) / (4 / math.pi * xs)
        xyz = p0 * np.array([5.0, scale, 2.0])
        s = synthetic.visibilities(xyz, 1.0, src, flux, 0.1)
        syn = bipp_amd.NufftSynthesis(ctx, n, n, [[0.0, 3e38]], lmn, compute=compute,
                                      imager="nufft", tolerance=tol)
        syn.collect(1.0, s, xyz)
        if syn.nufft_grid()[1] == length:
            break
    assert syn.nufft_grid()[1] == length
    ref, _ = O.synthesize([synthetic.Sample(0, 0, 1.0, xyz, s, np.ones(n, bool))],
                          np.array([[0.0, 3e38]]), lmn)
    err = O.rel_l2(syn.images()[0], ref[0])
    print(f"grid {syn.nufft_grid()} {compute}: rel L2 {err:.2e}", flush=True)
    assert err <= bound


@pytest.mark.parametrize("compute,length", [(c, n) for c in ("mixed", "fp64")
                                            for n in (54, 250, 750, 1024, 1250, 2000, 2048, 2160)])
def test_fft_line_lengths(ctx, compute, length):
    """The x lines on both sides of the lengths at which their workgroups take 16, 8, 4, 2 lines,
    and of the longest that they take (2048), an array stretched along x."""
    tol = 1e-5 if compute == "mixed" else 1e-9
    bound = 1e-4 if compute == "mixed" else 7.5e-7   # as test_fft_axis_lengths
    r = np.random.default_rng(length)
    n = 9
    src, flux = synthetic.zenith_cap_sources(r, 5, 5.0)
    p0 = synthetic.disk_positions(r, n, 1.0) + np.array([0, 0, 0.3]) * r.normal(size=(n, 1))
    lmn = synthetic.make_lmn_grid(21, math.radians(20))
    w = math.ceil(math.log10(1 / tol)) + 1
    a, b = np.tril_indices(n)
    u = 2 * np.pi * (p0[a, 0] - p0[b, 0])
    xs = 0.5 * (u.max() - u.min()) * 0.5 * (lmn[:, 0].max() - lmn[:, 0].min())
    for want in np.arange(length / 2, length / 2 * 0.9 - 12, -max(length / 1000, 0.1)):
        scale = (want - w - 1) / (4 / math.pi * xs)
        if scale <= 0:
            break
        xyz = p0 * np.array([scale, 5.0, 2.0])
        s = synthetic.visibilities(xyz, 1.0, src, flux, 0.1)
        syn = bipp_amd.NufftSynthesis(ctx, n, n, [[0.0, 3e38]], lmn, compute=compute,
                                      imager="nufft", tolerance=tol)
        syn.collect(1.0, s, xyz)
        if syn.nufft_grid()[0] <= length:
            break
    ref, _ = O.synthesize([synthetic.Sample(0, 0, 1.0, xyz, s, np.ones(n, bool))],
                          np.array([[0.0, 3e38]]), lmn)
    err = O.rel_l2(syn.images()[0], ref[0])
    print(f"grid {syn.nufft_grid()} {compute}: rel L2 {err:.2e}", flush=True)
    assert err <= bound
