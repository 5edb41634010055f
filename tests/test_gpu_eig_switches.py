"""The eigensolver's environment switches above 256 beams, where a batch is solved phase by
phase: BIPP_EIG_PROFILE prints the phases, BIPP_EIG_MAX_SLOTS caps the samples solved together."""
import numpy as np
import pytest

from test_gpu_eig_split import make, solve

pytestmark = pytest.mark.gpu


def test_switches(ctx, monkeypatch, capfd):
    n, live = 260, [260, 0, 100, 259, 17]
    samples = make(n, live, 3)
    monkeypatch.delenv("BIPP_EIG_PROFILE", raising=False)
    monkeypatch.delenv("BIPP_EIG_MAX_SLOTS", raising=False)
    d, v, nr = solve(ctx, samples, n)
    assert "eig profile" not in capfd.readouterr().err
    monkeypatch.setenv("BIPP_EIG_PROFILE", "1")
    solve(ctx, samples, n)
    err = capfd.readouterr().err
    assert "5 samples phase by phase, 5 at a time" in err
    for phase in ("load", "cholesky", "whiten", "tridiag columns", "tridiag tail", "tridiag_eig",
                  "backtransform", "unwhiten"):
        assert f" {phase} " in err
    monkeypatch.setenv("BIPP_EIG_MAX_SLOTS", "2")
    d2, v2, nr2 = solve(ctx, samples, n)
    assert "5 samples phase by phase, 2 at a time" in capfd.readouterr().err
    # the same sums in another order: the bounds of the other float64 batches
    assert np.array_equal(nr, nr2) and list(nr) == live
    for k in range(len(live)):
        assert np.abs(d2[k] - d[k]).max() <= 1e-10 * max(np.abs(d[k]).max(), 1e-300)
        a, b = ((x[k] * y[k]) @ x[k].conj().T for x, y in ((v, d), (v2, d2)))
        assert np.linalg.norm(a - b) <= 1e-10 * np.linalg.norm(a)
