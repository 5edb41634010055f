"""Replays of the captured per-timestep chain against eager collects of the same batch, bit for
bit in float64: below and above the 256 beams from which the eigensolve runs phase by phase,
samples of different live counts, and more samples than that form takes at a time (256).  The
levels take at most 32 eigenvectors of a sample: one wavefront of the float64 steering kernel,
which adds the sums of several in no fixed order."""
import math

import numpy as np
import pytest

import bipp_amd
from bipp_amd import synthetic
from bipp_amd.hip import D2H, DeviceArray, hip
from oracle import bipp_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ns", [(40, 3), (264, 1), (264, 5), (264, 270)])
def test_graph_bits(ctx, n, ns):
    r = np.random.default_rng(n + ns)
    p0 = synthetic.disk_positions(r, n, 400.0)
    src, flux = synthetic.zenith_cap_sources(r, 24, 5.0)
    kinds = []
    for k, live in enumerate([n, n - 3, n // 2, 1, 0]):
        act = np.zeros(n, bool)
        act[r.choice(n, size=live, replace=False)] = True
        wl = 2.0 + 0.05 * k
        s = synthetic.visibilities(p0, wl, src, flux, 0.1)
        s[~act] = 0
        s[:, ~act] = 0
        kinds.append(synthetic.Sample(0, k, wl, p0, s, act))
    samples = [kinds[k % 5] for k in range(ns)]
    s_d, x_d, wl_d = (DeviceArray.from_numpy(a)
                      for a in synthetic.stack_samples(samples, np.complex64))
    lmn = synthetic.make_lmn_grid(12, math.radians(5))
    # levels: the ten largest eigenvalues over all samples, and the next ones down to the least
    # bound that no sample has more than 32 above
    ev = [np.sort(O.eigh_gram(k.wl, k.s, None, k.xyz)[1])[::-1] for k in kinds[:4]]
    low = max(d[32] for d in ev if len(d) > 32) * 1.001 + 1e-12
    top = np.sort(np.concatenate(ev))[-10] * 0.999
    iv = [[low, top], [top, 3e38]]

    def images(collect):
        syn = bipp_amd.NufftSynthesis(ctx, n, n, iv, lmn, compute="fp64")
        out = []
        for _ in range(3):
            syn.reset()
            collect(syn)
            ctx.synchronize()
            ptr, prec = syn.image_device()
            assert prec == "double"
            img = np.empty((2, lmn.shape[0]))
            assert hip().hipMemcpy(img.ctypes.data, ptr, img.nbytes, D2H) == 0
            out.append(img)
        return out

    eager = images(lambda syn: syn.collect_device(ns, wl_d.ptr, s_d.ptr, False, x_d.ptr))
    replay = images(lambda syn: syn.collect_graph(ns, wl_d.ptr, s_d.ptr, False, x_d.ptr))
    assert np.all(np.isfinite(eager[0])) and np.abs(eager[0]).max() > 0
    print(n, ns, [int(np.count_nonzero(a != eager[0])) for a in eager + replay], flush=True)
    assert all(np.array_equal(a, eager[0]) for a in eager + replay)
