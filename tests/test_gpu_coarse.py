"""Factorisation of the coarsest system (blocked symmetric sweep, 32-wide blocks, out of
place) at the sizes where it can go wrong: fewer unknowns than one block, remainders of
every kind, an even and an odd number of block steps, and a singular system.

The V-cycle of a two-level hierarchy applies the factor once between two FP64 sweeps, so
its difference from the oracle's (Cholesky) is bounded by a few n eps cond: with n <= 1400,
a coarsest system of condition below 1e6 (a box of at most 25 elements' length at contrast
125) and eps 1.1e-16 that is 1e-7; 1e-9 leaves no room for a wrong entry."""
import numpy as np
import pytest

from topoptspline3d_amd.context import Context, TosError
from topoptspline3d_amd.domains import cantilever

from oracle_api import oracle_api

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    from topoptspline3d_amd.backend import gpu_available, hip_api
    if not gpu_available():
        pytest.skip("no GPU")
    return hip_api()


def build(api, dims, prec=0, support=True):
    solid, sup, f = cantilever(*dims)
    ctx = Context(api, solid, sup if support else None, n_levels=2)
    ctx.set_material(1e6, 0.4, 3.0, 1e-3)
    ctx.set_loads(f)
    rng = np.random.default_rng(sum(dims))
    ctx.set_density(rng.uniform(0.2, 1.0, solid.size).astype(np.float32))
    ctx.set_galerkin_precision(prec) if prec else None
    ctx.update_operator()
    return ctx, f


# coarsest unknowns 24 (one partial block), 36, 96 (three whole blocks), 192, 210, 225, 1344
@pytest.mark.parametrize("dims", [(2, 2, 2), (4, 2, 2), (6, 6, 2), (6, 6, 6), (8, 12, 2), (9, 8, 4), (25, 12, 7)])
def test_two_level_cycle_matches_oracle(hip, dims):
    g, f = build(hip, dims)
    o, _ = build(oracle_api(), dims)
    assert g.info()["coarse_dofs"] == o.info()["coarse_dofs"]
    print("coarsest unknowns", g.info()["coarse_dofs"], flush=True)
    r = np.random.default_rng(3).standard_normal(f.size) * (np.tile(g.node_flags(0), 3) & 4 > 0)
    zg, zo = g.vcycle(r), o.vcycle(r)
    assert np.linalg.norm(zg - zo) <= 1e-9 * np.linalg.norm(zo)
    # a second update starts from the swept matrix's memory again
    g.update_operator()
    assert np.array_equal(g.vcycle(r), zg)


def test_singular_coarsest_system_is_reported(hip):
    """all nodes of one end fixed but a detached block floating: the pivot test sees it"""
    solid, sup, f = cantilever(24, 4, 4)
    solid[:, :, 10:14] = 0
    ctx = Context(hip, solid, sup, n_levels=2)
    ctx.set_density(np.full(solid.size, 0.5, np.float32))
    with pytest.raises(TosError) as e:
        ctx.update_operator()
    assert e.value.code == -5
