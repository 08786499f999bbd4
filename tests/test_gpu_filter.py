"""tos_filter against the weighted mean in 64 bits, over the radii of each kernel (0.4 and 4.6:
the per-element one) and boxes that are smaller than a tile, end inside one and take one or
several z chunks.  Inputs have one sign, so a result is off by its rounding to float (2^-24)
and the rounding of FP64 sums of at most 500 terms."""
import math

import numpy as np
import pytest

from topoptspline3d_amd.context import Context

pytestmark = pytest.mark.gpu


def mean64(s, on, radius):
    H = int(radius + 0.5)
    nz, ny, nx = s.shape
    num, den = np.zeros(s.shape), np.zeros(s.shape)
    v = np.where(on, s.astype(np.float64), 0.0)
    for dz in range(-H, H + 1):
        for dy in range(-H, H + 1):
            for dx in range(-H, H + 1):
                r2 = dx * dx + dy * dy + dz * dz
                if r2 > radius * radius or abs(dz) >= nz or abs(dy) >= ny or abs(dx) >= nx:
                    continue
                r = math.sqrt(r2) / radius
                w = 1 - 6 * r ** 2 + 8 * r ** 3 - 3 * r ** 4
                a = tuple(slice(max(0, -d), min(n, n - d)) for d, n in ((dz, nz), (dy, ny), (dx, nx)))
                b = tuple(slice(max(0, d), min(n, n + d)) for d, n in ((dz, nz), (dy, ny), (dx, nx)))
                num[a] += w * v[b]
                den[a] += w * on[b]
    return np.where(on, num / np.where(on, den, 1.0), 0.0)


@pytest.mark.parametrize("dims", [(5, 4, 3), (64, 8, 2), (65, 17, 33), (130, 9, 70), (71, 43, 37)])
def test_filter_matches_64bit_mean(dims):
    from topoptspline3d_amd.backend import gpu_available, hip_api
    if not gpu_available():
        pytest.skip("no GPU")
    nx, ny, nz = dims
    rng = np.random.default_rng(nx)
    solid = (rng.random((nz, ny, nx)) > 0.2).astype(np.uint8)
    solid[:, :, 0] = 1
    solid[nz // 2, : (ny + 1) // 2, 1:] = 0  # stretches without an active element
    support = np.zeros((nz + 1, ny + 1, nx + 1), np.uint8)
    support[:, :, 0] = 1
    c = Context(hip_api(), solid, support)
    c.set_material(1e6, 0.4, 3.0, 1e-3)
    f = -np.exp(rng.normal(0, 2, solid.shape)).astype(np.float32)
    for radius in (0.4, 1.0, 1.49, 2.0, 2.6, 3.49, 3.6, 4.45, 4.6):
        print(f"[filter] {dims} radius {radius}", flush=True)
        c.set_sensitivity(f.ravel())
        c.filter(radius, 0)
        ref = mean64(f, solid > 0, radius)
        np.testing.assert_allclose(c.get_sensitivity(0), ref.ravel(), rtol=6.1e-8, atol=0)
    c.close()
