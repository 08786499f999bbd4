"""How many passes a Gauss-Seidel sweep takes, counted by the library's kernel timers: which
schedule runs is a rule on the level's rows, the cycle's precision and the sweep mode, and the
results are the same bit for bit, so only the passes show that the rule holds."""
import ctypes

import numpy as np
import pytest

from topoptspline3d_amd import _abi
from topoptspline3d_amd.context import Context
from topoptspline3d_amd.domains import cantilever

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    from topoptspline3d_amd.backend import gpu_available, hip_api
    if not gpu_available():
        pytest.skip("no GPU")
    return hip_api()


def context(hip, dims, n_levels=0):
    solid, support, f = cantilever(*dims)
    c = Context(hip, solid, support, n_levels=n_levels)
    c.set_material(1e6, 0.4, 3.0, 1e-3)
    c.set_loads(f)
    c.set_density(np.full(solid.size, 0.5, np.float32))
    c.update_operator()
    return c


def passes(hip, c, precision, which):
    """launches of the timed classes `which` in one V(1,1) cycle"""
    r = np.random.default_rng(0).normal(size=3 * c.nn)
    c.vcycle(r, precision=precision)
    ks = _abi.KernelStats()
    hip.profile(c.h, 1, ctypes.byref(ks))
    c.vcycle(r, precision=precision)
    hip.profile(c.h, 0, ctypes.byref(ks))
    return sum(ks.launches[i] for i in range(ks.n_classes) if ks.names[i].value.decode() in which)


@pytest.mark.parametrize("dims,paired", [((24, 12, 12), True), ((125, 6, 7), True), ((126, 6, 7), False),
                                         ((250, 9, 10), False), ((9, 130, 130), True)])
def test_fp64_fine_sweeps_pair_colours_on_rows_of_one_segment(hip, dims, paired):
    """125 free nodes after a fixed one are the longest row that is one segment for either first
    colour; (9, 130, 130) has 4225 rows a class.  Two sweeps a cycle, of four or eight passes."""
    c = context(hip, dims)
    n = {m: None for m in (0, 3)}
    for m in n:
        c.set_sweep_mode(m)
        n[m] = passes(hip, c, 0, ("fine_gs_f64",))
    print(f"\n[passes] {dims}: mode 0 {n[0]}, mode 3 {n[3]}", flush=True)
    assert n[0] == 16
    assert n[3] == (8 if paired else 16)


@pytest.mark.parametrize("precision", [0, 1, 2])
def test_stencil_levels_with_few_rows_take_one_colour_a_pass_but_in_mode_3(hip, precision):
    """Three levels, the second one a stored-stencil level of few rows, the third the coarsest
    solve: two sweeps a cycle on the second, of eight passes in modes 0 to 2 and four in mode 3."""
    c = context(hip, (40, 20, 24), n_levels=3)
    n = []
    for m in (0, 1, 2, 3):
        c.set_sweep_mode(m)
        n.append(passes(hip, c, precision, ("st_gs_f64", "st_gs_f32", "st_gs_f32_l1")))
    print(f"\n[passes] precision {precision}: {n}", flush=True)
    assert n == [16, 16, 16, 8]
