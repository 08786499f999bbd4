"""V-cycles whose stencil levels take several waves per row, against the FP64 oracle: rows of
one pair and of the largest single segment (126 free nodes, 252 elements on the fine level;
with 256 the level's rows are two segments and it keeps the one-wave kernels), odd sizes, voids
that break rows, supports that start rows at x = 0 and at x = 1 (the long boxes stand on z = 0:
as cantilevers their coarsest solve alone, of condition 1e7, differs from the oracle's by 3e-9).  FP64 cycles agree to rounding
(relative 1e-11 over a few thousand operations of condition up to 1e4); FP32 ones to 2e-4 and
FP16 stencils to 1e-2 as in the general V-cycle test."""
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
