"""V-cycles whose stencil levels take several waves per row: against the FP64 oracle, and against
the one-wave kernels at the same precision.  Rows of one pair, of the longest single segment (125
free nodes: 250 elements on the fine level) and of two segments (from 252 elements on, where the
level keeps the one-wave kernels), odd sizes, voids that break rows, supports that start rows at
x = 0 and at x = 1 (the long boxes stand on z = 0: as cantilevers their coarsest solve alone, of
condition 1e7, differs from the oracle's by 3e-9).  Against the oracle FP64 cycles agree to rounding
(relative 1e-11 over a few thousand operations of condition up to 1e4), FP32 ones to 2e-4 and FP16
stencils to 1e-2 as in the general V-cycle test: these bound the precision, and the comparison at
equal precision the kernels."""
import numpy as np
import pytest

from oracle_api import oracle_api
from topoptspline3d_amd.context import Context
from topoptspline3d_amd.domains import cantilever

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,void,zsup", [((9, 9, 40), 0.0, False), ((10, 24, 11), 0.3, True),
                                            ((252, 10, 9), 0.1, True), ((256, 9, 10), 0.1, True),
                                            ((37, 41, 23), 0.25, False), ((64, 50, 33), 0.0, True)])
def test_vcycles_match_oracle(dims, void, zsup):
    from topoptspline3d_amd.backend import gpu_available, hip_api
    if not gpu_available():
        pytest.skip("no GPU")
    nx, ny, nz = dims
    print(f"\n[split] {dims} void {void} zsup {zsup}", flush=True)
    rng = np.random.default_rng(nx)
    solid, support, f = cantilever(nx, ny, nz)
    if zsup:
        support = np.zeros_like(support)
        support.reshape(nz + 1, ny + 1, nx + 1)[0] = 1
    solid = (rng.random(solid.shape) >= void).astype(np.uint8)
    solid[:, :, 0] = 1
    solid[0] = 1
    rho = rng.uniform(0.3, 1.0, solid.size).astype(np.float32)
    r = rng.normal(size=3 * (nx + 1) * (ny + 1) * (nz + 1))
    z = []
    for api in (oracle_api(), hip_api()):
        c = Context(api, solid, support)
        c.set_material(1e6, 0.4, 3.0, 1e-3)
        c.set_loads(f)
        c.set_density(rho)
        c.update_operator()
        z.append(c.vcycle(r) if api is oracle_api() else [c.vcycle(r, precision=p) for p in (0, 1, 2)])
        c.close()
    zo = z[0]
    for zp, tol in zip(z[1], (1e-11, 2e-4, 1e-2)):
        d = np.linalg.norm(zp - zo) / np.linalg.norm(zo)
        print(f"[split] relative difference {d:.2e}", flush=True)
        assert d <= tol


@pytest.mark.parametrize("nx", [12, 67, 250])
def test_several_waves_per_row_match_one_wave_at_the_same_precision(nx):
    """A small body alone in its box, and beside a second one that takes the levels' row and chunk
    counts past the limits of the kernels with several waves per row.  A gap of a coarsest element
    keeps the bodies' equations apart on every level, so a residual on the first one gives the
    same correction there, formed by the other kernels from the same stencils (also the FP16
    ones).  The sums differ in order only: of a row's 243 products 243 FP32 roundings, 1.5e-5, at
    the very most (3e-14 in FP64, which the levels may add up), where a block missed or read from
    another node would change them by some 1e-2."""
    from topoptspline3d_amd.backend import gpu_available, hip_api
    if not gpu_available():
        pytest.skip("no GPU")
    ny, nz = 64, 160
    rng = np.random.default_rng(nx)
    both, support, f = cantilever(nx, ny, nz)
    both = (rng.random(both.shape) >= 0.05).astype(np.uint8)
    both[:, :, 0] = 1
    both[16:32] = 0
    one = both.copy()
    one[:, 32:] = 0
    one[32:] = 0
    both[:32] = one[:32]
    rho = rng.uniform(0.3, 1.0, one.shape).astype(np.float32)
    r = np.zeros((3, nz + 1, ny + 1, nx + 1))
    r[:, :17, :33] = rng.normal(size=(3, 17, 33, nx + 1))
    z, info = [], []
    for solid in (one, both):
        c = Context(hip_api(), solid, support, n_levels=5)
        c.set_material(1e6, 0.4, 3.0, 1e-3)
        c.set_density(rho.ravel())
        c.update_operator()
        info.append(c.info()["n_free_nodes"])
        z.append([c.vcycle(r.ravel(), precision=p).reshape(r.shape)[:, :17, :33] for p in (0, 1, 2)])
        c.close()
    print(f"\n[split] {nx}: free nodes {info}", flush=True)
    for p, tol in ((0, 1e-12), (1, 1.5e-5), (2, 1.5e-5)):
        d = np.linalg.norm(z[1][p] - z[0][p]) / np.linalg.norm(z[0][p])
        print(f"[split] precision {p}: relative difference {d:.2e}", flush=True)
        assert d <= tol
