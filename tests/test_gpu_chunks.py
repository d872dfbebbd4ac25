"""The k-marching kernels over chunks of several planes, as on the grids they are made for: on the small meshes of
the other tests a chunk is one plane, so what these kernels carry from plane to plane (registers, the slots in
LDS) never reaches a compared value there.  Tall meshes of few columns here: chunks of 2 to 24 planes, the last one
shorter, several tiles along i or j, against the oracle."""
import numpy as np
import pytest
import torch

import tests.test_gpu_formt as formt
import tests.test_gpu_mixed as mixed
import tests.test_gpu_vjp_tiles as vjp
from oracle import oracle as O
from tests._util import np_mesh, out_arrays, random_case, relerr, to_dev, to_np
from tests.test_chunks import RULES, plane_chunk
from tosca_amd import case as C

pytestmark = pytest.mark.gpu

# column tiles of the kernels (cells or points along i, j) and the planes they march over
TILES = dict(FORMU=(62, 7), FILTER3=(30, 14), FILTER5=(28, 12), BOX=(64, 8), DPASD_IJ=(60, 12), DPASD_K=(64, 4), FORMT=(60, 7))
SIZES = [(5, 9, 700), (4, 9, 1001), (61, 13, 331), (5, 15, 2003)]       # cells along i, j, k
PERS = [(0, 0, 0), (1, 2, 1), (2, 0, 2)]


def chunk(rule, n):
    """planes per chunk, and of the last chunk, on n cells"""
    up = lambda a, b: -(-a // b)
    ni, nj, nk = n
    if rule == "VJP_MARCH":
        nk, tiles = nk + 2, up(ni + 2, 60) * up(nj, 4)
    elif rule == "VJP_FINISH":
        nk, tiles = nk + 2, up(ni + 2, 62) * up(nj + 2, 6)
    elif rule == "FILTER_F32":                             # pieces of chunks of nk // 8 planes
        t = up(ni, 62) * up(nj, 6)
        full = up(nk, max(1, min(up(2048, t), nk // 8)))
        nk, tiles = full, t * up(nk, full)
    else:
        tiles = up(ni, TILES[rule][0]) * up(nj, TILES[rule][1])
    k = plane_chunk(nk, tiles, rule)
    return k, (nk - 1) % k + 1


def test_chunks_of_several_planes():
    for rule in RULES:
        got = [chunk(rule, n) for n in SIZES]
        assert max(k for k, _ in got) >= (8 if rule != "FILTER_F32" else 2), (rule, got)
        assert any(k > 1 and last < k for k, last in got) or rule == "FILTER_F32", (rule, got)
    # the FP32 DPASD k pass takes four planes a step: its chunks end in steps of every length
    assert {x % 4 for n in MIXED for x in chunk("DPASD_K", n)} == {0, 1, 2, 3}


def _case(n, periodic, model, scheme=C.DIV_QUICK, **kw):
    lay, mesh, f, params = random_case(n=(n[2], n[0], n[1]), periodic=periodic, seed=31, les_model=model, div_scheme=scheme, amp=0.1, **kw)
    assert (lay.mx, lay.my, lay.mz) == tuple(c + 2 for c in n)
    from tosca_amd.rhs import RhsContext
    nm = np_mesh(mesh)
    return lay, nm, {k: to_dev(v) for k, v in nm.items()}, {k: to_np(v) for k, v in f.items()}, params, RhsContext(lay.info())


@pytest.mark.parametrize("scheme", [C.DIV_CENTRAL, C.DIV_QUICK])
@pytest.mark.parametrize("periodic", PERS)
@pytest.mark.parametrize("n", SIZES)
def test_formu(n, periodic, scheme):
    """The fluxes of a cell cancel by 10 to 100, each of about 100 roundings: 1e-12 relative L2."""
    lay, nm, dm, f, params, ctx = _case(n, periodic, C.LES_SMAGORINSKY, scheme)
    out = out_arrays(lay)
    want, got = out["rhs"].copy(), to_dev(out["rhs"])
    O.formu(lay.info(), nm, params, f["ucont"], f["ucat"], f["nut"], want, 0.7, 0)
    ctx.FormU(dm, params, to_dev(f["ucont"]), to_dev(f["ucat"]), to_dev(f["nut"]), got, 0.7, 0)
    assert relerr(to_np(got), want) <= 1e-12
    ctx.close()


@pytest.mark.parametrize("model,tol", [(C.LES_DSM, 1e-12), (C.LES_DPASD, 1e-11)])
@pytest.mark.parametrize("periodic", PERS)
@pytest.mark.parametrize("n", SIZES + [(2, 2, 2), (29, 13, 3), (28, 12, 5), (31, 15, 4)])
def test_update_cs(n, periodic, model, tol):
    """The computed cells by their own norm, the entries left alone bit for bit, the periodic copies as the cells.
    Velocities without a mean: L = <U u> - <U><u> loses a digit, the box average or the plane mean of LM two to
    three, each value carries about 10 roundings: 1e-12 (DSM), and the quotient of DPASD's four means 1e-11.
    max_cs above every value, so that cells are not clipped from above; those below 0 are."""
    lay, nm, dm, f, params, ctx = _case(n, periodic, model, max_cs=1e6)
    start = out_arrays(lay)["cs"]
    u, want = f["ucat"], start.copy()
    O.update_cs(lay.info(), nm, params, u, want)
    cells = want[4:-4, 4:-4, 4:-4]
    assert np.count_nonzero(cells) >= cells.size // 4 and cells.max() < 1e6
    g = to_dev(start)
    ctx.UpdateCs(dm, params, to_dev(u), g)
    got = to_np(g)
    assert relerr(got[4:-4, 4:-4, 4:-4], cells) <= tol
    inside = np.zeros(want.shape, bool)
    inside[4:-4, 4:-4, 4:-4] = True
    kept = (want == start) & ~inside
    assert np.array_equal(got[kept], start[kept])
    copies = ~kept & ~inside
    assert np.abs(got[copies] - want[copies]).max(initial=0.0) <= tol * np.linalg.norm(cells)
    ctx.close()


@pytest.mark.parametrize("model", [C.LES_SMAGORINSKY, C.LES_DSM])
@pytest.mark.parametrize("n", SIZES[1:])
def test_step(n, model):
    """The step, with nu_t from the box average's kernel and bTheta from FormU's: as test_formu and test_update_cs,
    nu_t and Rhs with the error of Cs (one more digit)."""
    lay, nm, dm, f, params, ctx = _case(n, (2, 0, 2), model)
    o = {k: v for k, v in out_arrays(lay).items() if k in ("rhs", "cs", "nut", "btheta")}
    g = {k: to_dev(v) for k, v in o.items()}
    O.rhs_les_step(lay.info(), nm, params, f["ucont"], f["ucat"], f["theta"], o["rhs"], 0.7, o["cs"], o["nut"], o["btheta"], 1.3)
    ctx.rhs_les_step(dm, params, to_dev(f["ucont"]), to_dev(f["ucat"]), to_dev(f["theta"]), g["rhs"], 0.7, g["cs"], g["nut"], g["btheta"], 1.3)
    for k in o:
        cut = (slice(4, -4),) * 3 if k in ("cs", "nut") else ...
        assert relerr(to_np(g[k])[cut], o[k][cut]) <= (1e-12 if model == C.LES_SMAGORINSKY else 1e-11), k
    ctx.close()


MIXED = [(5, 9, 700), (4, 9, 1001), (29, 13, 1100), (5, 15, 2003)]


@pytest.mark.parametrize("model", [C.LES_DSM, C.LES_DPASD])
@pytest.mark.parametrize("n", MIXED)
def test_mixed_step(n, model):
    from tosca_amd import rhs
    mixed.test_mixed_step(rhs, f"{n} {model}", lambda: C.abl_case(nx=n[2], ny=n[0], nz=n[1], lx=15.0 * n[2], ly=15.0 * n[0],
                                                                 les_model=model, turbulence="noise"))


@pytest.mark.parametrize("scheme,les", [(C.DIV_CENTRAL, 1), (C.DIV_QUICK, 1), (C.DIV_QUICK, 0)])
@pytest.mark.parametrize("periodic", PERS)
@pytest.mark.parametrize("n", SIZES)
def test_vjp(n, periodic, scheme, les):
    """As the tile tests of the adjoint: at most 1e6 terms, 30 * 1e-16 * sqrt(1e6) = 3e-12, one wrong value 1e-6."""
    vjp.test_vjp_tile_edges(n, periodic, scheme, les)


@pytest.mark.parametrize("scheme", [C.DIV_CENTRAL, C.DIV_QUICK])
@pytest.mark.parametrize("periodic", PERS)
@pytest.mark.parametrize("n", SIZES[:3])
def test_vjp_mixed(n, periodic, scheme):
    vjp.test_vjp_mixed_tile_edges(n, periodic, scheme)


@pytest.mark.parametrize("scheme", [C.DIV_CENTRAL, C.DIV_QUICK])
@pytest.mark.parametrize("periodic", PERS)
@pytest.mark.parametrize("n", [(2, 2, 2), (3, 2, 4), (61, 9, 2)])
def test_vjp_mixed_smallest(n, periodic, scheme):
    """Axes of two cells: a handful of values, whose sums of 40 terms may all cancel to a hundredth: 6e-8 * sqrt(40)
    * 100 = 4e-5: relative L2 1e-4; one wrong value shows as 1e-2 or more."""
    lay, mesh, params, x, tau, rbar, _ = vjp._setup(n, periodic, scheme, 1)
    x = {k: v if k == "cs" else v.astype(np.float32).astype(np.float64) for k, v in x.items()}
    want, got = vjp._vjp(lay, mesh, params, x, tau, rbar), vjp._vjp(lay, mesh, params, x, tau, rbar, mixed=True)
    for name in x:
        assert relerr(got[name], want[name]) <= 1e-4, name


@pytest.mark.parametrize("les,model", [(0, C.LES_DSM), (1, C.LES_SMAGORINSKY), (1, C.LES_DSM)])
@pytest.mark.parametrize("periodic", PERS)
@pytest.mark.parametrize("n", SIZES)
def test_formt(n, periodic, les, model):
    """As the tile tests of FormT: the cube roots differ in the last ulps, the fluxes of a cell cancel by 1e3: 1e-12."""
    from tosca_amd import rhs
    lay, mesh, params, f, tp = formt._case((n[2], n[0], n[1]), periodic, 61, les, model, walls=True)
    assert formt._compare(rhs, lay, mesh, params, f, tp, 1.0, 0, f"{n}") <= 1e-12
