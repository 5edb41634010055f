"""The NUFFT tuner on a grid whose shape some of its candidates do not change: up to 2048 points
the x lines run in a form without a radix choice, and strided axes whose lengths have register
passes do not read the strided radix.  Candidates that launch the same kernels share one time, so
that the choice between them is not noise."""
import pytest

import bipp_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("compute,tol", [("mixed", 1e-5), ("fp64", 1e-9)])
def test_equal_candidates_share_a_time(ctx, golden, compute, tol):
    z = golden("cfg1_small.npz")
    s, xyz = z["s"].swapaxes(1, 2), z["xyz"].swapaxes(1, 2)
    bipp_amd.call("bipp_nufft_tuning_reset")
    try:
        syn = bipp_amd.NufftSynthesis(ctx, 37, 37, z["intervals"], z["lmn"], compute=compute,
                                      imager="nufft", tolerance=tol, autotune=True)
        syn.collect(z["wl"], s, xyz)
        grid = syn.nufft_grid()
        print("grid", grid, flush=True)
        assert grid[0] <= 2048 and all(n % 125 for n in grid)
        shape, rows = syn.nufft_tuning()
        assert len(rows) == 24
        times = {}
        for c, ms in rows:
            times.setdefault((c["pass_tw_shift"], c["spread_chunk"]), set()).add(ms)
        assert len(times) == 4 and all(len(t) == 1 for t in times.values())
        # among equals the first, which holds the default radices
        assert (shape["lines_radix"], shape["pass_radix"]) == (9, 4)
    finally:
        bipp_amd.call("bipp_nufft_tuning_reset")
