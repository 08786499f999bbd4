"""The trials of tos_oc_update_noalloc over element arrays in whole, ragged and single chunks,
aligned and not, with and without masks, for targets inside, below and above the reach of the
move limit, and inputs that a 32-bit estimate cannot place (zeros, infinities, NaN, values at
the ends of the float range).  Reference: the same bisection with the update in 64 bits; pow
may differ by an ulp there, which moves a rounded float by at most one ulp (1.2e-7)."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def reference(act, shell, rho, sens, vgoal, move, damp, rmin):
    def trial(g):
        with np.errstate(all="ignore"):
            gg = np.where(sens > 0, 0.0, -sens.astype(np.float64))
            r = rho.astype(np.float64) * np.power(gg / g, damp)
        r = np.fmin(np.fmax(r, rho.astype(np.float64) - move), rho.astype(np.float64) + move)
        r = np.fmin(np.fmax(r, rmin), 1.0)
        return np.where(shell, 1.0, r).astype(np.float32)

    with np.errstate(all="ignore"):
        hi = float(np.fmax.reduce(np.abs(sens[act].astype(np.float64)), initial=0.0))
    lo, g, steps = 0.0, 0.5 * hi, 0
    while True:
        v = trial(g)[act].astype(np.float64).sum() / act.sum()
        steps += 1
        if v > vgoal:
            lo = g
        elif v < vgoal:
            hi = g
        if abs(v - vgoal) <= 1e-4 or steps >= 31:
            break
        g = 0.5 * (lo + hi)
    return np.where(act, trial(g), rho), g, steps


@pytest.mark.parametrize("n", [1, 3, 1023, 8192, 8195, 3 * 8192 + 777])
@pytest.mark.parametrize("odd", [False, True])
def test_trials_match_64bit_bisection(n, odd):
    import torch
    from topoptspline3d_amd.backend import gpu_available, hip_api
    if not gpu_available():
        pytest.skip("no GPU")
    rng = np.random.default_rng(n)
    act, shell = rng.random(n) < 0.8, rng.random(n) < 0.05
    act[0] = True
    shell[0] = False
    rho = rng.uniform(0.05, 0.95, n).astype(np.float32)
    sens = (-np.exp(1.2 * rng.normal(size=n))).astype(np.float32)
    special = np.array([0.0, -0.0, 2.0, np.nan, -1e-38, -1e-44, -3e-30, 1e30], np.float32)
    if n > 1000:
        sens[rng.integers(1, n, 64)] = np.tile(special, 8)
        rho[rng.integers(1, n, 8)] = np.array([0.0, 1e-44, 1e-31, 1.0, 1.5, -0.25, 1e-3, 0.999], np.float32)
    k = 1 if odd else 0  # odd: every array starts off a 16-byte (4-byte) boundary

    def dev(a):
        t = torch.zeros(n + k, dtype=torch.from_numpy(a[:1].copy()).dtype, device="cuda")
        t[k:] = torch.from_numpy(a)
        return t

    da, ds, dr, dg = dev(act.astype(np.uint8)), dev(shell.astype(np.uint8)), dev(rho), dev(sens)
    ptr = lambda t: t.data_ptr() + k * t.element_size()
    for masks in (True, False):
        for vgoal, move, damp, rmin in ((0.45, 0.05, 0.5, 1e-3), (0.1, 0.03, 0.5, 1e-3), (0.95, 0.03, 0.3, 1e-3),
                                        (0.5, 0.2, 1.0, 0.0), (0.5, 0.1, 4.5, 1e-9), (0.5, 0.1, 0.01, 1e-3)):
            print(f"[oc flat] n {n} odd {odd} masks {masks} goal {vgoal} damp {damp}", flush=True)
            out = torch.full((n + k,), -7.0, device="cuda")
            torch.cuda.synchronize()
            g, steps = ctypes.c_double(), ctypes.c_int()
            rc = hip_api().oc_update_noalloc(n, ptr(da) if masks else None, ptr(ds) if masks else None, ptr(dr),
                                             ptr(dg), ptr(out), vgoal, move, damp, rmin, None, ctypes.byref(g),
                                             ctypes.byref(steps))
            assert rc == 0
            a = act if masks else np.ones(n, bool)
            ref, g_ref, st_ref = reference(a, shell if masks else np.zeros(n, bool), rho, sens, vgoal, move, damp, rmin)
            assert steps.value == st_ref and g.value == g_ref
            np.testing.assert_allclose(out.cpu().numpy()[k:], ref, rtol=1.2e-7, atol=0)
        if n <= 1000:
            break
    # in place
    rc = hip_api().oc_update_noalloc(n, ptr(da), ptr(ds), ptr(dr), ptr(dg), ptr(dr), 0.45, 0.05, 0.5, 1e-3, None,
                                     ctypes.byref(g), ctypes.byref(steps))
    assert rc == 0
    ref, g_ref, st_ref = reference(act, shell, rho, sens, 0.45, 0.05, 0.5, 1e-3)
    assert steps.value == st_ref and g.value == g_ref
    np.testing.assert_allclose(dr.cpu().numpy()[k:], ref, rtol=1.2e-7, atol=0)
