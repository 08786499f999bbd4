"""MMA updates for every constraint count and vector lengths around a workgroup, against the
FP64 oracle over a few outer iterations of a problem with curved objective and constraints.
The subproblem is solved to a KKT residual of about 1e-5 by the same Newton steps, so the points
agree to the effect of rounding on sums of n terms (1e-9 of the unit box).  Constraints of ordinary
scale accept a step within three halvings; the line search tries four together, so steep ones
follow, which take up to fourteen."""
import numpy as np
import pytest

from oracle_api import oracle_api
from topoptspline3d_amd.context import MMA

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 2, 3, 4])
@pytest.mark.parametrize("n", [1, 7, 256, 1000])
def test_updates_match_oracle(n, m):
    from topoptspline3d_amd.backend import gpu_available, hip_api
    if not gpu_available():
        pytest.skip("no GPU")
    rng = np.random.default_rng(10 * n + m)
    a, t = rng.uniform(0.5, 2, n), rng.uniform(0.1, 0.9, n)
    B, cap = rng.uniform(0.2, 1.0, (m, n)) / n, 0.45
    xs = []
    for api in (oracle_api(), hip_api()):
        opt = MMA(api, n, m, 0.0, 1.0, move=0.2)
        x = np.full(n, 0.6)
        opt.set_x(x)
        path = []
        for it in range(6):
            df = 2 * a * (x - t) / n
            g = B @ (x * x) - cap * B.sum(axis=1)
            opt.update(df, 2 * B * x, g)
            x = opt.x()
            path.append(x)
        xs.append(np.array(path))
        opt.close()
    d = np.abs(xs[1] - xs[0]).max()
    print(f"[mma] n {n} m {m}: largest difference {d:.2e}", flush=True)
    assert d <= 1e-9


@pytest.mark.parametrize("m", [1, 2, 3, 4])
@pytest.mark.parametrize("n", [7, 1000])
@pytest.mark.parametrize("steep", [100.0, 1e4])
def test_updates_with_long_line_searches_match_oracle(n, m, steep):
    """Constraints `steep` times steeper than the objective: of the oracle's accepted Newton steps
    in these three updates 69 to 206 come after four halvings or more, the longest after 5 (n = 7,
    m = 3, 100) to 14 (n = 7, m = 4, 1e4) of them (counted in its line search).  Inputs changed by
    2e-15 of themselves move the points by at most 4e-15, so 1e-12 leaves room for sums in another
    order and for nothing else."""
    from topoptspline3d_amd.backend import gpu_available, hip_api
    if not gpu_available():
        pytest.skip("no GPU")
    rng = np.random.default_rng(n + m)
    a, t = rng.uniform(0.5, 2, n), rng.uniform(0.1, 0.9, n)
    B = rng.uniform(0.2, 1.0, (m, n)) / n * steep
    opts = [MMA(api, n, m, 0.0, 1.0, move=0.2) for api in (oracle_api(), hip_api())]
    x = np.full(n, 0.6)
    for opt in opts:
        opt.set_x(x)
    for it in range(3):
        for opt in opts:
            opt.update(2 * a * (x - t) / n, 2 * B * x, B @ (x * x) - 0.45 * B.sum(axis=1))
        x, y = opts[0].x(), opts[1].x()
        d = np.abs(y - x).max()
        print(f"[mma] n {n} m {m} steep {steep} update {it}: largest difference {d:.2e}", flush=True)
        assert d <= 1e-12
    for opt in opts:
        opt.close()
