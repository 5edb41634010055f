"""The direct-sum imager on batches: antisymmetric and general uvw in one batch, one to ten
images (eight levels per launch), pixel counts off the workgroup size with the slots of few
pixels split over workgroups and those of many pixels not, against the float64 sum over every
baseline of the stored values."""
import math

import numpy as np
import pytest

import bipp_amd
from bipp_amd import synthetic
from oracle import bipp_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_ant,n_beam,ns,grid,n_img,precision", [
    (1, 1, 2, 3, 1, "single"), (2, 2, 3, 5, 2, "double"), (9, 7, 5, 17, 3, "single"),
    (23, 23, 4, 33, 10, "single"), (23, 11, 4, 33, 10, "double"), (5, 5, 2, 730, 1, "single")])
def test_direct_sum_shapes(ctx, n_ant, n_beam, ns, grid, n_img, precision):
    r = np.random.default_rng(n_ant + ns + grid)
    ds = bipp_amd.InMemoryDataset.create("rand", n_ant, n_beam)
    for k in range(ns):
        v = (r.normal(size=(n_ant, n_beam)) + 1j * r.normal(size=(n_ant, n_beam))) / 3
        if k % 2 == 0:
            uvw = O.baselines_uvw(r.normal(size=(n_ant, 3)) * 30)
        else:
            uvw = r.normal(size=(n_ant * n_ant, 3)) * 30
        ds.write(float(k), 1.5 + 0.1 * k, 1.0 / 81, v, r.lognormal(size=n_beam), uvw)
    lmn = synthetic.make_lmn_grid(grid, math.radians(30)).astype(np.float32)
    prop = bipp_amd.InMemoryImageProp.create(grid, grid, 30.0, lmn)
    sel = {f"i{i}": {k: np.where(np.arange(n_beam) % n_img == i % n_beam, ds.eig_val(k), 0)
                     for k in range(ns)} for i in range(n_img)}
    opt = bipp_amd.NufftSynthesisOptions().set_precision(precision)
    opt.imager = "direct"
    data = bipp_amd.image_synthesis(ctx, opt, ds, sel, prop)
    sub = np.arange(0, grid * grid, max(1, grid * grid // 997))
    for name, samples in sel.items():
        ref = np.zeros(sub.size)
        for k, dsc in samples.items():
            vv = O.virtual_vis(float(ds.scale(k)), np.asarray(dsc, np.float64),
                               ds.eig_vec(k).astype(np.complex128))
            ref += O.nuft_sum(1.0, vv, ds.uvw(k).astype(np.float64) * (2 * np.pi / ds.wl(k)),
                              lmn[sub].astype(np.float64))
        ref /= ns
        img = data.get(name).reshape(-1, order="F")[sub]
        err = float(np.linalg.norm(img - ref) / max(np.linalg.norm(ref), 1e-300))
        print(f"{n_ant} antennas, {name}: rel L2 {err:.2e}", flush=True)
        # the bounds of the direct imager's other tests
        assert err <= (1e-5 if precision == "single" else 1e-7) or np.linalg.norm(ref) == 0
