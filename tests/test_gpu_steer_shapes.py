"""Split-bf16 steering at the edges of its tiling: row tiles of 8 eigenvectors dealt over 8
wavefronts (1 to 4 per wavefront, then two passes above 256 eigenvectors), antenna chunks of
16, pixel tiles of 128, and several samples of different live counts in one launch, against
the float64 oracle."""
import numpy as np
import pytest

import bipp_amd
from bipp_amd import synthetic
from oracle import bipp_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,grid,n_lv", [(3, 5, 1), (16, 12, 8), (65, 9, 2), (129, 16, 3),
                                         (193, 11, 4), (256, 8, 4), (300, 13, 2)])
def test_steer_shapes(ctx, n, grid, n_lv):
    wl_ = synthetic.make_workload(2, n_timesteps=3, grid=grid, n_antenna=n)
    rng = np.random.default_rng(n)
    for k, smp in enumerate(wl_.samples):
        dead = rng.choice(n, size=(k * n) // 5, replace=False)   # 0, 20 and 40 % flagged
        smp.s[dead, :] = 0
        smp.s[:, dead] = 0
        smp.s = smp.s.astype(np.complex64).astype(np.complex128)
    d = np.sort(O.eigh_gram(wl_.samples[0].wl, wl_.samples[0].s, None, wl_.samples[0].xyz)[1])
    cut = [0.0] + [float(np.sqrt(d[n * i // n_lv - 1] * d[n * i // n_lv])) if n > n_lv else float(i)
                   for i in range(1, n_lv)] + [3e38]
    iv = np.array([[cut[i], cut[i + 1]] for i in range(n_lv)])
    ref, _ = O.synthesize(wl_.samples, iv, wl_.lmn)
    syn = bipp_amd.NufftSynthesis(ctx, n, n, iv, wl_.lmn, compute="mixed", imager="steering")
    syn.collect([s.wl for s in wl_.samples],
                np.stack([s.s for s in wl_.samples]).astype(np.complex64),
                np.stack([s.xyz for s in wl_.samples]))
    img = syn.images()
    for lvl in range(n_lv):
        if np.linalg.norm(ref[lvl]) == 0:
            assert np.all(img[lvl] == 0)
            continue
        err = O.rel_l2(img[lvl], ref[lvl])
        print(f"n={n} grid={grid} level {lvl}: rel L2 {err:.2e}", flush=True)
        assert err <= 1e-4      # the mixed form's bound of the other image tests
