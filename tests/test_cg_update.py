"""CG update of meshes without a 3-D box structure: up to 786432 nodes it
assembles A p from the group lists, above from a DSS pass.  10 iterations on
each side of that line, at the smallest order and grid, and with a ragged last
workgroup, against the oracle."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
import geoflow_amd as ga
import oracle

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]

# 10 iterations of FP64 CG in two summation orders: the parity tests' bound
TOL = 1e-11


@pytest.mark.parametrize("bdy", [ga.GF_BDY_DIRICHLET, ga.GF_BDY_PERIODIC])
@pytest.mark.parametrize("p,ne", [(1, [3, 2]), (6, [9, 7]), (11, [70, 78]), (11, [71, 78])])
def test_cg_update_2d(p, ne, bdy):
    from geoflow_amd.device import Context, Mesh
    print("cg update", p, ne, bdy, flush=True)
    bg, og = ga.BoxGrid(2, p, ne, bdy=[bdy] * 4), oracle.Grid.box(2, p, ne, bdy=[bdy] * 4)
    m = Mesh(Context(0), bg)
    rng = np.random.default_rng(p)
    f = og.dss(rng.standard_normal(bg.ndof), "smooth")
    b = og.mass_apply(f)
    xb = np.zeros(bg.ndof) if bdy == ga.GF_BDY_DIRICHLET else None
    its = 10 if p > 1 else 1  # the smallest grid has two free nodes
    kw = dict(xb=xb, p=0.1, maxit=its, tol=1e-300, normtype=0)
    dev = {k: torch.from_numpy(v).cuda() if isinstance(v, np.ndarray) else v for k, v in kw.items()}
    xg, info = m.cg_solve(torch.from_numpy(b).cuda(), q=1.0, **dev)
    xo, _, it, res = og.cg_solve(b, q=np.ones(bg.ndof), **kw)
    assert info["iters"] == it == its
    assert np.abs(xg.cpu().numpy() - xo).max() <= TOL * np.abs(xo).max()
    assert np.abs(np.array(info["resid"][:its]) - res[:its]).max() <= TOL * np.abs(res[:its]).max()
