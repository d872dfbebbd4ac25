"""UpdateCs on the FP64 test-filter kernels at the edges of their tiles: 30 x 14 (3-point filter) and
28 x 12 (5-point filter) cells of (i, j), chunks of a few k planes, against the oracle.

Tolerances (relative L2 of Cs): a filtered sum carries about 10 roundings, the Leonard terms
L = <U u> - <U><u> lose the factor |U u| / |L| ~ 1 / 0.05^2 to 1e4 of a 5 % turbulence over a mean flow,
so LM / MM is good to 1e-16 * 10 * 1e4 = 1e-11; the plane means of DPASD's QN cancel by up to another
factor of 10 over a few hundred cells: 1e-10."""
import numpy as np
import pytest
import torch

from tosca_amd import case as C

pytestmark = pytest.mark.gpu

SIZES = [  # (cells along i, j, k)
    (2, 2, 2), (28, 12, 5), (29, 13, 3), (30, 14, 2), (31, 15, 4), (57, 25, 6), (61, 29, 9), (13, 43, 33),
]


@pytest.mark.parametrize("model,tol", [(C.LES_DSM, 1e-11), (C.LES_DPASD, 1e-10)])
@pytest.mark.parametrize("ptype", [C.PERIODIC_COPY, C.PERIODIC_WRAP])
@pytest.mark.parametrize("ni,nj,nk", SIZES)
def test_update_cs_tile_edges(ni, nj, nk, ptype, model, tol):
    from oracle import oracle as O
    from tosca_amd.rhs import RhsContext
    case = C.abl_case(nx=nk, ny=ni, nz=nj, lx=15.0 * nk, ly=15.0 * ni, les_model=model, turbulence="noise")
    lay = case.lay
    params = dict(case.params, periodic=(ptype, C.PERIODIC_NONE, ptype))
    mesh = {k: v.numpy().copy() for k, v in case.mesh.items() if k != "cent"}
    start = np.random.default_rng(3).standard_normal(lay.gshape)
    want = start.copy()
    O.update_cs(lay.info(), mesh, params, case.ucat.numpy().copy(), want)
    dev = {k: torch.as_tensor(v).cuda() for k, v in mesh.items()}
    cs = torch.as_tensor(start).cuda()
    ctx = RhsContext(lay.info())
    ctx.UpdateCs(dev, params, case.ucat.cuda(), cs)
    got = cs.cpu().numpy()
    ctx.close()
    assert np.isfinite(got).all()
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert err <= tol, f"{ni} x {nj} x {nk}: {err:.2e}"
