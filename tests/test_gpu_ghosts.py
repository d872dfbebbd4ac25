"""Ghost fills that one launch composes from the operations along the axes: UpdateNutBCs and the wraps of
nu_t and k_sgs, the periodic resets and wraps of Cs, ucont and ucat, bTheta and the farm AXPY outside the
interior cells; smallest and odd sizes, both periodic types, against the oracle on whole arrays that are
filled with the same values before (so what a routine must leave alone is compared too).
Ghosts are copies of values that carry up to about 200 roundings: 200 * 1e-16 * sqrt(200) < 1e-12 relative L2."""
import numpy as np
import pytest
import torch

from tosca_amd import case as C
from oracle import oracle as O
from tests._util import np_mesh, out_arrays, random_case, relerr, to_dev, to_np

pytestmark = pytest.mark.gpu

TOL = 1e-12
SIZES = [(2, 2, 2), (2, 3, 7), (6, 6, 6), (7, 9, 3), (64, 3, 2), (3, 14, 23)]      # cells along i, j, k
PERS = [(0, 0, 0), (1, 1, 1), (2, 2, 2), (2, 0, 1), (0, 1, 2), (1, 2, 0)]


def _setup(n, periodic, seed, model):
    lay, mesh, f, params = random_case(n=(n[2], n[0], n[1]), periodic=periodic, seed=seed, les_model=model,
                                       bcu_nonper=(C.BCU_GENERIC, C.BCU_SLIP, C.BCU_WALLFUNCTION),
                                       bcnut_nonper=(C.BCNUT_ZEROGRADIENT, C.BCNUT_FIXEDVALUE))
    assert (lay.mx, lay.my, lay.mz) == tuple(c + 2 for c in n)
    from tosca_amd.rhs import RhsContext
    nm = np_mesh(mesh)
    tau = (to_np(f["tau_i"]), to_np(f["tau_j"]))
    dt = tuple(to_dev(t) for t in tau)
    po = dict(params, tau_wall_i=tau[0].ctypes.data, tau_wall_j=tau[1].ctypes.data)
    pg = dict(params, tau_wall_i=dt[0].data_ptr(), tau_wall_j=dt[1].data_ptr())
    return lay, nm, {k: to_dev(v) for k, v in nm.items()}, {k: to_np(v) for k, v in f.items()}, po, pg, RhsContext(lay.info()), (tau, dt)


@pytest.mark.parametrize("periodic", PERS)
@pytest.mark.parametrize("n", SIZES)
def test_update_nut_ghosts(n, periodic):
    lay, nm, dm, f, po, pg, ctx, keep = _setup(n, periodic, 3, C.LES_DSM)
    out = out_arrays(lay)
    cs = np.random.default_rng(4).uniform(0.0, 0.1, lay.gshape)
    nut, ksgs = out["nut"].copy(), out["ksgs"].copy()
    O.update_nut(lay.info(), nm, po, f["ucat"], cs, nut, ksgs)
    gn, gk = to_dev(out["nut"]), to_dev(out["ksgs"])
    ctx.UpdateNut(dm, pg, to_dev(f["ucat"]), to_dev(cs), gn, gk)
    assert relerr(to_np(gn), nut) <= TOL and relerr(to_np(gk), ksgs) <= TOL
    ctx.close()


@pytest.mark.parametrize("farm", [False, True])
@pytest.mark.parametrize("periodic", PERS)
@pytest.mark.parametrize("n", SIZES)
def test_step_ghosts(n, periodic, farm):
    lay, nm, dm, f, po, pg, ctx, keep = _setup(n, periodic, 5, C.LES_SMAGORINSKY)
    names = ("rhs", "cs", "nut", "btheta")
    o = {k: v for k, v in out_arrays(lay).items() if k in names}
    g = {k: to_dev(v) for k, v in o.items()}
    src = np.random.default_rng(6).standard_normal(o["rhs"].shape)
    flow, flow_g = [f[k] for k in ("ucont", "ucat", "theta")], [to_dev(f[k]) for k in ("ucont", "ucat", "theta")]
    tail = lambda a: (a["rhs"], 0.8, a["cs"], a["nut"], a["btheta"], 1.1)
    if farm:
        O.rhs_les_step_farm(lay.info(), nm, po, *flow, src, *tail(o))
        ctx.rhs_les_step_farm(dm, pg, *flow_g, to_dev(src), *tail(g))
    else:
        O.rhs_les_step(lay.info(), nm, po, *flow, *tail(o))
        ctx.rhs_les_step(dm, pg, *flow_g, *tail(g))
    for k in names:
        assert relerr(to_np(g[k]), o[k]) <= TOL, k
    ctx.close()


@pytest.mark.parametrize("periodic", PERS)
@pytest.mark.parametrize("n", SIZES)
def test_predictor_ghosts(n, periodic):
    lay, nm, dm, f, po, pg, ctx, keep = _setup(n, periodic, 7, C.LES_DSM)
    rng = np.random.default_rng(8)
    dp, bt, uo = (rng.standard_normal((lay.mz, lay.my, lay.mx, 3)) for _ in range(3))
    rhs, utmp = np.full_like(dp, 7.0), np.full_like(dp, 7.0)
    uc, ua = f["ucont"].copy(), f["ucat"].copy()
    g = [to_dev(a) for a in (uc, ua, rhs, utmp)]
    O.ueqn_rk4(lay.info(), nm, po, uc, ua, f["nut"], dp, bt, None, 0, None, uo, 1e-4, rhs, utmp)
    ctx.UeqnRK4(dm, pg, g[0], g[1], to_dev(f["nut"]), to_dev(dp), to_dev(bt), None, 0, None, to_dev(uo), 1e-4, g[2], g[3])
    for name, a, b in zip(("ucont", "ucat", "rhs", "utmp"), g, (uc, ua, rhs, utmp)):
        assert relerr(to_np(a), b) <= TOL, name
    ctx.close()


@pytest.mark.parametrize("periodic", PERS)
@pytest.mark.parametrize("n", SIZES)
def test_predictor_ghosts_transposed(n, periodic):
    """<xbar, J d> = <J^T xbar, d> of two RK3W stages against the tangent oracle: the transposed copies of
    the smallest axes, on which every point has several.  About 100 roundings a product against the sum of
    the sizes of at most 1e4 terms, with a wrong value among them showing as 1e-4: bound 1e-10."""
    lay, nm, dm, f, po, pg, ctx, keep = _setup(n, periodic, 9, C.LES_DSM)
    rng = np.random.default_rng(10)
    shape = (lay.mz, lay.my, lay.mx, 3)
    dp, bt, xbar, du = (rng.standard_normal(shape) for _ in range(4))
    dn, dt = rng.standard_normal(lay.gshape), 0.02
    work = [torch.zeros(shape, dtype=torch.float64, device="cuda") for _ in range(3)]
    ub, nb = to_dev(xbar), torch.zeros(lay.gshape, dtype=torch.float64, device="cuda")
    ctx.UeqnRK3W_adjoint(dm, pg, to_dev(f["ucont"]), to_dev(f["ucat"]), to_dev(f["nut"]), to_dev(dp), to_dev(bt), None, 0, None,
                         dt, 2, *work, ub, nb)
    for d, bar in ((dict(d_ucont=du), np.sum(to_np(ub) * du)), (dict(d_nut=dn), np.sum(to_np(nb) * dn))):
        _, dF = O.rk3w_jvp(lay.info(), nm, po, f["ucont"], f["ucat"], f["nut"], dp, bt, None, 0, None, dt, 2, **d)
        err = abs(np.sum(xbar * dF) - bar) / (np.sum(np.abs(xbar * dF)) + 1e-300)
        assert err <= 1e-10, (d.keys(), err)
    ctx.close()
