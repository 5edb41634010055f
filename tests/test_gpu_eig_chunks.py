"""A float64 batch above 256 beams of more samples than the phase-split form takes at a time
(256), of very different live counts: two chunks that share their scratch memory.  A sample's
eigenpairs against LAPACK through the oracle, and the same bits wherever in the batch it is."""
import numpy as np
import pytest

from oracle import bipp_oracle as O
from test_gpu_eig_split import make, rel, solve

pytestmark = pytest.mark.gpu


def test_two_chunks(ctx):
    n, live = 258, [258, 0, 257, 130, 1, 256, 64]
    kinds = make(n, live, 5)
    ns = 259
    d, v, nr = solve(ctx, [kinds[k % len(kinds)] for k in range(ns)], n)
    for k, smp in enumerate(kinds):
        assert nr[k] == live[k]
        for q in range(k + len(kinds), ns, len(kinds)):
            assert np.array_equal(d[q], d[k]) and np.array_equal(v[q], v[k]) and nr[q] == nr[k]
        if not live[k]:
            assert np.all(d[k] == 0) and np.all(v[k] == 0)
            continue
        vo, do, _, _ = O.eigh_gram(smp.wl, smp.s.astype(np.complex64), None, smp.xyz)
        # the bounds of the other float64 batches
        assert np.abs(d[k] - do).max() < 1e-10 * np.abs(do).max()
        assert rel((v[k] * d[k]) @ v[k].conj().T, (vo * do) @ vo.conj().T) < 1e-10
