"""Grouping of the surface points by knot cell and its gradient sums, against the oracle, at
the sizes where they can go wrong: cells of more points than a wavefront has lanes, spline
orders whose k^3 block is smaller and larger than a wavefront, boxes without any point, and
buffers reused after a larger and a smaller lattice.

Both sides sum the same FP64 products, in another order; the results are FP32.  A gradient
sums at most a few thousand terms of one sign pattern, so 1e-5 of the largest entry (100
FP32 roundings) bounds the difference."""
import numpy as np
import pytest

from test_gpu_surface import coeffs_for, hip, pair  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode,order,param,cells", [(1, 4, 8, (90, 24, 90)), (1, 2, 4, (40,)), (1, 5, 5, (60,)),
                                                    (0, 3, 5, (70, 12)), (1, 3, 16, (64,))])
def test_gradients_match_oracle(hip, mode, order, param, cells):  # noqa: F811
    nx, ny, nz = 28, 20, 24
    (o, g), n = pair(hip, nx, ny, nz, mode, order, param)
    cf = coeffs_for(o, nx, ny, nz, mode, order, param)
    for c in (o, g):
        c.set_coeffs(cf)
    for m in cells:
        so, sg = (c.surface_constraints(cells=m, beta=8.0, ss_mode=4, drip_mode=7, drip_beta=4.0, drip_mu=2.0,
                                        drip_beta_scale=1.0) for c in (o, g))
        print(mode, order, param, m, sg, flush=True)
        assert so["n_points"] == sg["n_points"]
        for which in (2, 3):
            go, gg = o.coeff_sens(which), g.coeff_sens(which)
            assert np.abs(gg - go).max() <= 1e-5 * max(np.abs(go).max(), 1e-30), (m, which)


def test_a_box_without_surface_points(hip):  # noqa: F811
    (o, g), n = pair(hip, 12, 9, 10, 1, 4, 4)
    cf = np.linspace(0.05, 0.3, n, dtype=np.float32)  # below the level everywhere
    for c in (o, g):
        c.set_coeffs(cf)
        s = c.surface_constraints(cells=20, beta=8.0)
        assert s["n_points"] == 0
        assert not np.any(c.coeff_sens(2)) and not np.any(c.coeff_sens(3))


def plane(nx, ny, nz, param):
    """coefficients of a tilted plane surface, uniform lattice"""
    ncx, ncy, ncz = (nx + param - 1) // param + 1, (ny + param - 1) // param + 1, (nz + param - 1) // param + 1
    k, j, i = np.meshgrid(np.arange(ncz), np.arange(ncy), np.arange(ncx), indexing="ij")
    return np.clip(0.5 + 0.9 * (k / ncz + 0.25 * i / ncx - 0.6), 0.01, 1).astype(np.float32).ravel()


@pytest.mark.parametrize("param,cells", [(16, (8, 9, 12, 48)), (6, (40, 64))])
def test_cells_of_more_points_than_a_slot(hip, param, cells):  # noqa: F811
    """Knot cells of less than one, one and a few, and up to some thirty slots of 128 points: the
    point order within a cell and the sums over a cell's slots."""
    nx, ny, nz = 24, 16, 20
    (o, g), n = pair(hip, nx, ny, nz, 1, 4, param)
    cf = np.random.default_rng(param).uniform(0.05, 1.0, n).astype(np.float32)
    for c in (o, g):
        c.set_coeffs(cf)
    for m in cells:
        so, sg = (c.surface_constraints(cells=m, beta=8.0, ss_mode=4, drip_mode=7, drip_beta=4.0, drip_mu=2.0,
                                        drip_beta_scale=1.0) for c in (o, g))
        print(param, m, sg, flush=True)
        assert so["n_points"] == sg["n_points"] > 0
        first = [g.coeff_sens(w).copy() for w in (2, 3)]
        for which in (2, 3):
            go = o.coeff_sens(which)
            assert np.abs(first[which - 2] - go).max() <= 1e-5 * max(np.abs(go).max(), 1e-30), (m, which)
        g.surface_constraints(cells=m, beta=8.0, ss_mode=4, drip_mode=7, drip_beta=4.0, drip_mu=2.0,
                              drip_beta_scale=1.0)
        assert all(np.array_equal(g.coeff_sens(w), first[w - 2]) for w in (2, 3)), m


def test_a_lattice_much_finer_than_the_knots_takes_no_serial_chain(hip):  # noqa: F811
    """2e5 points in a few knot cells: some milliseconds; a chain over a cell's points, or over
    their pairs in one wavefront, takes seconds."""
    import time
    solid, support, _ = cantilever_box(32, 20, 20)
    from topoptspline3d_amd.context import Context
    c = Context(hip, solid, support)
    c.set_material(1e6, 0.4, 3.0, 1e-3)
    n = c.spline_init(1, 4, 16)
    c.set_coeffs(np.random.default_rng(3).uniform(0.05, 1.0, n).astype(np.float32))
    c.surface_constraints(cells=256, beta=8.0)
    t = time.perf_counter()
    s = c.surface_constraints(cells=256, beta=8.0)
    t = time.perf_counter() - t
    print(f"\n[surface] {s['n_points']} points, {t * 1e3:.1f} ms", flush=True)
    assert s["n_points"] > 100000 and t < 1.0


def cantilever_box(*dims):
    from topoptspline3d_amd.domains import cantilever
    return cantilever(*dims)


def test_memory_follows_the_occupied_cells(hip):  # noqa: F811
    """Order 8 (8 KB of sums per occupied cell), a plane through 45 x 33 x 33 coefficients: two
    thousand occupied cells of 5e4, 1e4 points.  Lattice and points need 400 MB at 84 cells; sums
    for as many cells as points would add 160 MB.  Other lattice sizes replace the buffers."""
    import torch
    from topoptspline3d_amd.context import Context
    solid, support, _ = cantilever_box(88, 64, 64)
    c = Context(hip, solid, support)
    c.set_material(1e6, 0.4, 3.0, 1e-3)
    c.spline_init(1, 8, 2)
    c.set_coeffs(plane(88, 64, 64, 2))
    used = []
    free0 = torch.cuda.mem_get_info()[0]
    for cells in (84, 40, 84, 40, 84):
        s = c.surface_constraints(cells=cells, beta=8.0)
        used.append((free0 - torch.cuda.mem_get_info()[0]) >> 20)
        print(f"\n[surface] cells {cells}: {s['n_points']} points, {used[-1]} MB", flush=True)
    nl = 86 ** 3
    assert used[0] <= (592 * nl + 2400 * s["n_points"] >> 20) + 60
    assert used[4] <= used[0] + 40 and used[3] < used[0]
