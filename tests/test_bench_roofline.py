"""The work that bench.py's roofline counts per Gauss-Seidel launch follows the schedule that the
library runs: one colour a launch, or two in sweep mode 3 (FP64 fine sweeps only where every row
is one segment)."""
import numpy as np
import pytest

import bench
from oracle_api import oracle_api
from topoptspline3d_amd.context import Context
from topoptspline3d_amd.domains import cantilever

INFO = {"n_active_elements": [1000], "n_free_nodes": [1100, 200], "n_levels": 2}


@pytest.mark.parametrize("nx,one", [(24, True), (125, True), (126, False), (250, False)])
def test_rows_of_one_segment(nx, one):
    """125 free nodes behind a fixed one are the longest row that fits one wave from either parity"""
    solid, support, _ = cantilever(nx, 5, 6)
    c = Context(oracle_api(), solid, support)
    assert bench.rows_of_one_segment(c.node_flags(0), c.info()["level_dims"][0]) == one


def test_a_hole_does_not_shorten_a_row():
    flags = np.zeros((3, 3, 201), np.uint8)
    flags[1, 1, 10:20] = 4
    assert bench.rows_of_one_segment(flags.ravel(), (200, 2, 2))
    flags[1, 1, 150] = 4
    assert not bench.rows_of_one_segment(flags.ravel(), (200, 2, 2))


@pytest.mark.parametrize("cls,colours", [("fine_gs_f32", (1, 2, 2)), ("fine_gs_f64", (1, 1, 2)),
                                         ("st_gs_f32_l1", (1, 2, 2))])
def test_work_per_launch(cls, colours):
    sweep = {"fine_gs_f32": 4 * 1000 + 40 * 1100, "fine_gs_f64": 4 * 1000 + 76 * 1100,
             "st_gs_f32_l1": (243 * 4 + 36) * 200}[cls]
    flops = 504 * 200 if cls == "st_gs_f32_l1" else 1170 * 1100
    for (mode, pairs), n in zip(((0, True), (3, False), (3, True)), colours):
        r = bench.roofline({cls: (2e-4, 10)}, INFO, 1100, 1, None, 1, mode, pairs)
        assert r["kernel"] == cls
        assert r["bytes_per_launch"] == pytest.approx(sweep / 8.0 * n)
        assert r["achieved_tflops"] == pytest.approx(flops / 8.0 * n / 2e-8 / 1e12, abs=6e-3)
