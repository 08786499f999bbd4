"""tos_filter against the weighted mean in 64 bits, over the radii of each kernel (0.4 and 4.6:
the per-element one, which also takes 3.6 and 4.45 on the narrow tall box) and boxes that are
smaller than a tile, end inside one and take one or several z chunks.  Inputs have one sign, so a result is off by its rounding to float (2^-24)
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


@pytest.mark.parametrize("dims", [(5, 4, 3), (64, 8, 2), (65, 17, 33), (130, 9, 70), (71, 43, 37), (8, 9, 900)])
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


@pytest.mark.parametrize("dims", [(8, 100, 1500), (8, 260, 400)])
def test_narrow_boxes_keep_the_per_element_kernel(dims):
    """Radii 4.4 and 4.6 on boxes that fill 8 of a column's 64 lanes: the smaller radius, within the
    ring kernel's range, has fewer taps and must not take longer than 1.4 times the larger one (the
    ring kernel takes 2.5 to 3 times as long there)."""
    import time
    from topoptspline3d_amd.backend import gpu_available, hip_api
    if not gpu_available():
        pytest.skip("no GPU")
    nx, ny, nz = dims
    support = np.zeros((nz + 1, ny + 1, nx + 1), np.uint8)
    support[0] = 1
    c = Context(hip_api(), np.ones((nz, ny, nx), np.uint8), support, n_levels=1)
    c.set_material(1e6, 0.4, 3.0, 1e-3)
    c.set_sensitivity(-np.random.default_rng(0).random(nx * ny * nz).astype(np.float32))
    t = {}
    for radius in (4.4, 4.6):
        best = 1e9
        for _ in range(20):
            t0 = time.perf_counter()
            c.filter(radius, 0)
            best = min(best, time.perf_counter() - t0)
        t[radius] = best * 1e3
    print(f"\n[filter] {dims}: {t[4.4]:.3f} ms at 4.4, {t[4.6]:.3f} ms at 4.6", flush=True)
    assert t[4.4] <= 1.4 * t[4.6]
    c.close()
