"""Box counts of the uvw partition on both sides of the bound up to which a workgroup counts
its points in LDS (512 boxes), and a batch whose slots are no multiple of a workgroup's share:
the image is that of the direct form (the transform is linear in its points)."""
import numpy as np
import pytest

import bipp_amd
from oracle import bipp_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(1, 1, 2), (8, 8, 8), (9, 19, 3)])
def test_box_counts(ctx, golden, dims):
    z = golden("cfg1_small.npz")
    s, xyz = np.swapaxes(z["s"], 1, 2), np.swapaxes(z["xyz"], 1, 2)
    syn = bipp_amd.NufftSynthesis(ctx, 37, 37, z["intervals"], z["lmn"], compute="fp64",
                                  imager="nufft", tolerance=1e-9,
                                  partition=bipp_amd.Partition.grid(dims))
    syn.collect(z["wl"], s, xyz)
    print(f"boxes {syn.nufft_partition()}", flush=True)
    img = syn.images()
    # the tolerance of the transform and the float32 image, as the one-plan test's
    for lvl in range(img.shape[0]):
        assert O.rel_l2(img[lvl], z["img_steering"][lvl]) < 1e-7
