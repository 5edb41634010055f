"""Host side of short-lived handles: staging that grows with the samples (sizes on both sides of
its first 16), buffers handed on between calls of different sizes and between threads with a
context each, and one beamforming matrix for all samples of a collect."""
import math
import threading

import numpy as np
import pytest

import bipp_amd
from bipp_amd import synthetic
from oracle import bipp_oracle as O

pytestmark = pytest.mark.gpu


def dataset(ns, n_ant, seed):
    r = np.random.default_rng(seed)
    ds = bipp_amd.InMemoryDataset.create("rand", n_ant, n_ant)
    for k in range(ns):
        v = (r.normal(size=(n_ant, n_ant)) + 1j * r.normal(size=(n_ant, n_ant))) / 3
        ds.write(float(k), 1.5 + 0.01 * k, 1.0 / 81, v, r.lognormal(size=n_ant),
                 O.baselines_uvw(r.normal(size=(n_ant, 3)) * 30))
    return ds


def image(ctx, ds, grid, imager, batch=None):
    lmn = synthetic.make_lmn_grid(grid, math.radians(20)).astype(np.float32)
    prop = bipp_amd.InMemoryImageProp.create(grid, grid, 20.0, lmn)
    opt = bipp_amd.NufftSynthesisOptions().set_precision("double").set_tolerance(1e-9)
    opt.set_sample_batch_size(batch)
    opt.imager = imager
    sel = {"a": {k: ds.eig_val(k) for k in range(ds.num_samples())}}
    img = bipp_amd.image_synthesis(ctx, opt, ds, sel, prop).get("a").reshape(-1, order="F")
    ref = np.zeros(lmn.shape[0])
    for k in range(ds.num_samples()):
        vv = O.virtual_vis(float(ds.scale(k)), ds.eig_val(k).astype(np.float64),
                           ds.eig_vec(k).astype(np.complex128))
        ref += O.nuft_sum(1.0, vv, ds.uvw(k).astype(np.float64) * (2 * np.pi / ds.wl(k)),
                          lmn.astype(np.float64))
    return float(np.linalg.norm(img - ref / ds.num_samples()) / np.linalg.norm(ref) * ds.num_samples())


@pytest.mark.parametrize("ns,batch", [(1, None), (16, None), (17, None), (40, None), (40, 18)])
def test_staging_growth(ctx, ns, batch):
    # float32 images of double sums (test_gpu_image_synthesis.py: 1e-7)
    for imager in ("nufft", "direct"):
        assert image(ctx, dataset(ns, 4, ns), 9, imager, batch) <= 1e-7


def test_threads_with_own_contexts():
    errs, failed = {}, []

    def work(t):
        try:
            c = bipp_amd.Context("GPU")
            errs[t] = [image(c, dataset(3 + 5 * ((k + t) % 3), 3 + t + k % 2, 10 * t + k), 7 + t,
                             "nufft" if k % 2 else "direct") for k in range(4)]
        except Exception as e:  # reported by the main thread
            failed.append(e)

    th = [threading.Thread(target=work, args=(t,)) for t in range(3)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not failed and sorted(errs) == [0, 1, 2]
    assert max(max(e) for e in errs.values()) <= 1e-7


def test_one_matrix_for_all_samples(ctx):
    r = np.random.default_rng(2)
    na, nb, ns = 12, 7, 5
    xyz = r.normal(size=(na, 3)) * 40
    a = r.normal(size=(ns, nb, 20)) + 1j * r.normal(size=(ns, nb, 20))
    s = (a @ a.conj().transpose(0, 2, 1)).astype(np.complex64)
    w = (r.normal(size=(na, nb)) + 1j * r.normal(size=(na, nb))).astype(np.complex64)
    lmn = synthetic.make_lmn_grid(10, math.radians(10))
    imgs = []
    for ww in (w, np.stack([w] * ns)):
        syn = bipp_amd.NufftSynthesis(ctx, na, nb, [[0.0, 3e38]], lmn, compute="fp64")
        syn.collect(2.0, s, xyz, ww)
        imgs.append(syn.images())
    assert np.array_equal(imgs[0], imgs[1])
