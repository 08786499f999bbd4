"""The network's convolutions take voxels in tiles over row ends, four tiles a wave for batches
of 2^18 voxels and more and one below.  Grids narrower than a tile, one voxel past it and with
one-voxel axes against the NumPy network; a batch of equal samples that takes the wide form
against its single sample in the narrow one: the mean over samples scales every gradient by a
power of two, so only the order of the FP32 sums over voxels differs (relative 1e-4 of the
layer's norm with at most 2^19 addends of either sign)."""
import os
import sys

import numpy as np
import pytest

from topoptspline3d_amd import learned

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))

pytestmark = pytest.mark.gpu


def batch(B, X, Y, Z, seed):
    rng = np.random.default_rng(seed)
    mask = (rng.random((B, Z, Y, X)) < 0.85)
    feat = rng.normal(size=(B, Z, Y, X, 4)).astype(np.float32) * mask[..., None]
    target = rng.normal(size=(B, Z, Y, X, 3)).astype(np.float32) * mask[..., None]
    return feat, target, mask.astype(np.uint8)


def net():
    from topoptspline3d_amd.backend import gpu_available, hip_api
    if not gpu_available():
        pytest.skip("no GPU")
    return learned.UNet(hip_api(), seed=5)


@pytest.mark.parametrize("dims,B", [((5, 3, 2), 3), ((17, 4, 1), 2), ((1, 9, 16), 1), ((33, 5, 3), 2)])
def test_small_grids_match_reference(dims, B):
    import unet_ref as U
    X, Y, Z = dims
    n = net()
    feat, target, mask = batch(B, X, Y, Z, X)
    loss, grad = n.loss_grad(feat, target, mask)
    params = U.unpack(n.params().astype(np.float64))
    ref_loss, ref = U.loss_and_grad(params, feat.astype(np.float64), target.astype(np.float64), mask, bf=True)[:2]
    ref_grad = U.pack(ref)
    print(f"[unet tiles] {dims} x {B}: loss {loss:.6f} reference {ref_loss:.6f}", flush=True)
    assert abs(loss - ref_loss) <= 1e-2 * abs(ref_loss)  # BF16 activations
    d = np.linalg.norm(grad - ref_grad) / np.linalg.norm(ref_grad)
    assert d <= 3e-2, d


def test_wide_tiles_match_narrow():
    n = net()
    feat, target, mask = batch(1, 33, 33, 33, 1)
    l1, g1 = n.loss_grad(feat, target, mask)
    l8, g8 = n.loss_grad(*(np.repeat(a, 8, axis=0) for a in (feat, target, mask)))
    assert abs(l8 - l1) <= 1e-6 * abs(l1)
    d = np.linalg.norm(g8 - g1) / np.linalg.norm(g1)
    print(f"[unet tiles] wide against narrow {d:.2e}", flush=True)
    assert d <= 1e-4
