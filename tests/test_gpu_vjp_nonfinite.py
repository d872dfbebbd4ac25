"""A value of rbar that is not finite reaches, in the adjoint of the right-hand side, the entries that depend
on it and no others: terms of weight zero (the QUICK cell on the other side of the upwind direction, the
one-sided differences next to a wall) are left out, not multiplied by zero.  The adjoint is linear in rbar, so
the entries that depend on rbar[p] are those where its answer to a unit rbar[p] is not zero: every metric is
moved off zero, also on the planar boundary faces."""
import numpy as np
import pytest

from tosca_amd import case as C
from tests.test_gpu_vjp_tiles import _setup, _vjp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("scheme,les", [(C.DIV_CENTRAL, 1), (C.DIV_QUICK, 1), (C.DIV_QUICK, 0)])
@pytest.mark.parametrize("periodic", [(0, 0, 0), (1, 2, 1), (2, 0, 2)])
def test_nonfinite_reaches_its_stencil_only(periodic, scheme, les, mixed):
    lay, mesh, params, x, tau, rbar, rng = _setup((9, 8, 7), periodic, scheme, les)
    mesh = {k: v + 0.01 * rng.standard_normal(v.shape) if v.ndim == 4 else v for k, v in mesh.items()}
    x = {k: v if k == "cs" else v.astype(np.float32).astype(np.float64) for k, v in x.items()}
    for k, j, i, q in ((4, 5, 5, 0), (3, 4, 4, 1), (4, 4, 3, 2), (1, 4, 4, 1), (4, 1, 4, 0), (4, 4, lay.mx - 2, 2), (lay.mz - 2, 3, 4, 2)):
        unit = np.zeros_like(rbar)
        unit[k, j, i, q] = 1.0
        reach = _vjp(lay, mesh, params, x, tau, unit, mixed)
        for bad in (np.nan, np.inf):
            r = rbar.copy()
            r[k, j, i, q] = bad
            for name, got in _vjp(lay, mesh, params, x, tau, r, mixed).items():
                lost = ~np.isfinite(got)
                assert not (lost & (reach[name] == 0.0)).any(), f"{name} {bad} at {(k, j, i, q)}: {np.argwhere(lost & (reach[name] == 0.0))[:3]}"
                assert lost.any() or name == "cs" or name == "theta", f"{name} {bad} at {(k, j, i, q)}"


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("periodic", [(0, 0, 0), (1, 2, 1), (2, 0, 2)])
def test_nonfinite_velocity_reaches_its_stencil_only(periodic, mixed):
    """The same for the velocity at and next to the boundaries, which ucat_bar and Cs_bar take through nu_t and
    |S|: the entries that depend on it are those that move by more than the rounding when it moves by 1/2, in FP64."""
    lay, mesh, params, x, tau, rbar, rng = _setup((9, 8, 7), periodic, C.DIV_CENTRAL, 1)
    mesh = {k: v + 0.01 * rng.standard_normal(v.shape) if v.ndim == 4 else v for k, v in mesh.items()}
    x = {k: v if k == "cs" else v.astype(np.float32).astype(np.float64) for k, v in x.items()}
    base = _vjp(lay, mesh, params, x, tau, rbar)
    for k, j, i in ((0, 4, 5), (4, 0, 5), (4, 4, 0), (4, 4, lay.mx - 1), (1, 4, 4), (4, 1, lay.mx - 2), (4, 4, 5)):
        at = (k + 3, j + 3, i + 3)
        moved = {n: v.copy() for n, v in x.items()}
        moved["ucat"][at] += 0.5
        moved = _vjp(lay, mesh, params, moved, tau, rbar)
        bad = {n: v.copy() for n, v in x.items()}
        bad["ucat"][at] = np.nan
        for name, got in _vjp(lay, mesh, params, bad, tau, rbar, mixed).items():
            still = np.abs(moved[name] - base[name]) <= 1e-13 * np.abs(base[name]).max()
            lost = ~np.isfinite(got)
            assert not (lost & still).any(), f"{name} at {(k, j, i)}: {np.argwhere(lost & still)[:3]}"
            assert lost.any() or name != "ucat", f"{name} at {(k, j, i)}"
