"""resetNoPenetrationFluxes sets the normal flux of a wall to 0.0, also where it was -0.0, in place and in the
periodic copies: the fluxes ExplicitRhsU leaves, bit for bit against the oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.test_gpu_ghosts import _setup
from tests._util import to_dev, to_np
from tosca_amd import case as C

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("periodic", [(0, 0, 0), (1, 0, 2), (2, 2, 0)])
def test_negative_zero_flux(periodic):
    lay, nm, dm, f, po, pg, ctx, keep = _setup((9, 7, 8), periodic, 21, C.LES_DSM)
    wall = tuple(C.BCU_PERIODIC if periodic[a // 2] else C.BCU_NOSLIP for a in range(6))
    po, pg = dict(po, bc_u=wall), dict(pg, bc_u=wall)
    rng = np.random.default_rng(22)
    uc, ua = f["ucont"].copy(), f["ucat"].copy()
    uc[rng.uniform(size=uc.shape) < 0.5] = -0.0
    dp, bt, uo = (rng.standard_normal((lay.mz, lay.my, lay.mx, 3)) for _ in range(3))
    rhs = np.zeros_like(dp)
    g = [to_dev(a) for a in (uc, ua, rhs)]
    O.explicit_rhs_u(lay.info(), nm, po, uc, ua, f["nut"], dp, bt, None, 0, None, uo, rhs, 0)
    ctx.ExplicitRhsU(dm, pg, g[0], g[1], to_dev(f["nut"]), to_dev(dp), to_dev(bt), None, 0, None, to_dev(uo), g[2])
    assert np.array_equal(to_np(g[0]).view(np.int64), uc.view(np.int64))
    ctx.close()
