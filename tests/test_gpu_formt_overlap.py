"""FormT into an rhs that lies in the memory of one of its inputs gives what it gives into an array of its own,
bit for bit: the inputs are read before they are overwritten.  Several workgroups along every axis, chunks of
one plane (each workgroup's neighbours are other workgroups)."""
import pytest
import torch

from tests._util import to_dev
from tests.test_gpu_formt import _case
from tosca_amd import case as C

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("offset", [0, 37])
@pytest.mark.parametrize("name", ["theta", "kt", "nut", "ucont"])
@pytest.mark.parametrize("model", [C.LES_SMAGORINSKY, C.LES_DSM])
def test_rhs_in_an_input(model, name, offset):
    from tosca_amd.rhs import RhsContext
    lay, mesh, params, f, tp = _case((24, 70, 23), (2, 0, 1), 51, 1, model, walls=True)
    ctx = RhsContext(lay.info())
    dm = {k: to_dev(v) for k, v in mesh.items()}
    tp = dict(tp, q_wall_i=to_dev(tp["q_wall_i"]), q_wall_j=to_dev(tp["q_wall_j"]))
    x = {k: to_dev(f[k]) for k in ("ucont", "theta", "nut", "kt")}
    shape = (lay.mz, lay.my, lay.mx)
    inside = x[name].view(-1)[offset:offset + lay.mz * lay.my * lay.mx].view(shape)
    apart = inside.clone()
    ctx.FormT(dm, params, tp, x["ucont"], x["theta"], x["nut"], x["kt"], apart)
    ctx.FormT(dm, params, tp, x["ucont"], x["theta"], x["nut"], x["kt"], inside)
    assert torch.equal(inside, apart)
    ctx.close()
