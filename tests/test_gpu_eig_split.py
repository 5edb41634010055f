"""Phase-split eigensolve (float64, above 256 beams) against LAPACK zhegv through the oracle:
sizes at the edges of its tiles (64), row tiles (16) and reflector blocks (16), one sample and
several of very different live counts (1, 17, 64, ... beams) in one batch, a general beamforming
matrix and a Gram matrix that is not positive definite in one sample."""
import numpy as np
import pytest

import bipp_amd
from bipp_amd import synthetic
from bipp_amd.hip import DeviceArray
from oracle import bipp_oracle as O

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def make(n, live, seed):
    r = np.random.default_rng(seed)
    p0 = synthetic.disk_positions(r, n, 400.0)
    src, flux = synthetic.zenith_cap_sources(r, 24, 5.0)
    out = []
    for k, m in enumerate(live):
        act = np.zeros(n, bool)
        act[r.choice(n, size=m, replace=False)] = True
        wl = 2.0 + 0.05 * k
        s = synthetic.visibilities(p0, wl, src, flux, 0.1)
        s[~act] = 0
        s[:, ~act] = 0
        out.append(synthetic.Sample(0, k, wl, p0, s, act))
    return out


def solve(ctx, samples, n):
    ns = len(samples)
    s_cm, x_cm, wls = synthetic.stack_samples(samples, np.complex64)
    s_d, x_d, wl_d = (DeviceArray.from_numpy(a) for a in (s_cm, x_cm, wls))
    d_d = DeviceArray.zeros((ns, n), np.float64)
    v_d = DeviceArray.zeros((ns, n, n), np.complex128)
    nr_d = DeviceArray.zeros(ns, np.int32)
    sc_d = DeviceArray.zeros(ns, np.float64)
    bipp_amd.call("bipp_eigh_gram_batched", ctx.handle, ns, n, n, 0, 1, 1, wl_d.ptr, s_d.ptr, n,
                  n * n, None, 0, 0, x_d.ptr, n, 3 * n, d_d.ptr, n, v_d.ptr, n, n * n, nr_d.ptr,
                  sc_d.ptr)
    ctx.synchronize()
    return d_d.numpy(), v_d.numpy().transpose(0, 2, 1), nr_d.numpy()


@pytest.mark.parametrize("n,live", [(257, [257]), (272, [0, 1, 2, 17, 64, 65, 272]),
                                    (320, [320, 200, 319] * 12), (512, [512, 497])])
def test_split_sizes(ctx, n, live):
    samples = make(n, live, n + len(live))
    print(f"split eigensolve n={n} live={live[:8]} jobs={len(live)}", flush=True)
    d, v, nr = solve(ctx, samples, n)
    for k, smp in enumerate(samples[:8]):
        assert nr[k] == live[k]
        if not live[k]:
            assert np.all(d[k] == 0) and np.all(v[k] == 0)
            continue
        vo, do, _, _ = O.eigh_gram(smp.wl, smp.s.astype(np.complex64), None, smp.xyz)
        # the bounds of the other float64 batches (test_gpu_eigh.py)
        assert np.abs(d[k] - do).max() < 1e-10 * np.abs(do).max()
        assert rel((v[k] * d[k]) @ v[k].conj().T, (vo * do) @ vo.conj().T) < 1e-10
    # the samples of a batch do not depend on each other: repeats agree bit for bit
    for k in range(3, len(live)):
        if len(live) > 8 and live[k] == live[k - 3]:
            one_d, _, _ = solve(ctx, [samples[k]], n)
            assert np.abs(one_d[0] - d[k]).max() <= 1e-12 * np.abs(d[k]).max()
            break


@pytest.mark.parametrize("n,live", [(64, [2, 3, 4, 5, 15, 16, 17, 33, 63, 64]),
                                    (128, [1, 65, 66, 97, 127, 128]),
                                    (256, [129, 159, 160, 161, 191, 192, 193, 223, 255, 256])])
def test_resident_sizes(ctx, n, live):
    """The tridiagonalisation with the trailing matrix in registers (up to 256 beams): sizes on
    both sides of its row tiles, and of the columns kept in registers (160) and LDS (192)."""
    samples = make(n, live, n)
    print(f"resident eigensolve n={n} live={live}", flush=True)
    d, v, nr = solve(ctx, samples, n)
    for k, smp in enumerate(samples):
        vo, do, _, _ = O.eigh_gram(smp.wl, smp.s.astype(np.complex64), None, smp.xyz)
        assert nr[k] == live[k]
        assert np.abs(d[k] - do).max() < 1e-10 * np.abs(do).max()
        assert rel((v[k] * d[k]) @ v[k].conj().T, (vo * do) @ vo.conj().T) < 1e-10


def test_cholesky_tile_sizes(ctx):
    """The Cholesky inverse on tiles of all samples: sizes on both sides of its diagonal blocks
    (32), tiles (64) and pairs of blocks, and samples far below the batch's largest."""
    n, live = 400, [400, 385, 384, 383, 352, 353, 321, 320, 319, 289, 288, 65, 64, 33, 32, 31, 1]
    samples = make(n, live, 11)
    print(f"split eigensolve n={n} live={live}", flush=True)
    d, v, nr = solve(ctx, samples, n)
    for k, smp in enumerate(samples):
        vo, do, _, _ = O.eigh_gram(smp.wl, smp.s.astype(np.complex64), None, smp.xyz)
        assert nr[k] == live[k]
        assert np.abs(d[k] - do).max() < 1e-10 * np.abs(do).max()
        assert rel((v[k] * d[k]) @ v[k].conj().T, (vo * do) @ vo.conj().T) < 1e-10


def test_handover_sizes(ctx):
    """The tridiagonalisation hands the last 256 columns from the column launches to one workgroup
    per sample: with one and with two updates pending (odd and even counts of columns before
    it), and samples that have no column before it."""
    n, live = 259, [256, 257, 258, 259, 255, 3]
    samples = make(n, live, 7)
    print(f"split eigensolve n={n} live={live}", flush=True)
    d, v, nr = solve(ctx, samples, n)
    for k, smp in enumerate(samples):
        vo, do, _, _ = O.eigh_gram(smp.wl, smp.s.astype(np.complex64), None, smp.xyz)
        assert nr[k] == live[k]
        assert np.abs(d[k] - do).max() < 1e-10 * np.abs(do).max()
        assert rel((v[k] * d[k]) @ v[k].conj().T, (vo * do) @ vo.conj().T) < 1e-10


def test_split_general_w(ctx):
    r = np.random.default_rng(5)
    na, nb = 300, 260
    p0 = synthetic.disk_positions(r, na, 300.0)
    src, flux = synthetic.zenith_cap_sources(r, 20, 5.0)
    w = np.zeros((na, nb), np.complex128)
    w[np.arange(na), np.arange(na) % nb] = np.exp(2j * np.pi * r.uniform(size=na))
    s = w.conj().T @ synthetic.visibilities(p0, 2.0, src, flux, 0.1) @ w
    v, d, _ = bipp_amd.eigh_gram(2.0, s, w, p0)
    vo, do, _, _ = O.eigh_gram(2.0, s, w, p0)
    assert np.abs(d - do).max() < 1e-10 * np.abs(do).max()
    assert rel((v * d) @ v.conj().T, (vo * do) @ vo.conj().T) < 1e-10


def test_split_not_positive_definite(ctx):
    r = np.random.default_rng(3)
    n = 270
    xyz = r.normal(size=(n, 3)) * 50
    w = np.eye(n)
    w[:, 130] = 0
    s = np.eye(n, dtype=np.complex128) + 0.1
    with pytest.raises(bipp_amd.EigensolverError):
        bipp_amd.eigh_gram(2.0, s, w, xyz)
