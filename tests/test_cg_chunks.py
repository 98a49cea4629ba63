"""Box CG (k_cg_apply3p, k_cg_update_halo) at every order: a small ragged box
against the oracle, and a periodic box of more than two chunks of elements to
every workgroup, the last one partly filled, against the same box without its
structure (group lists or DSS passes); then a box whose vectors exceed the
256 MB cache, where the apply bypasses it."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
import geoflow_amd as ga
import oracle
from geoflow_amd.ensemble import _UnionGrid
from geoflow_amd import workloads

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _rel(a, b):
    return float((a - b).abs().max() / b.abs().max())


@pytest.mark.parametrize("bdy", [ga.GF_BDY_DIRICHLET, ga.GF_BDY_PERIODIC])
@pytest.mark.parametrize("p", range(1, 10))
def test_small_ragged_box(p, bdy):
    from geoflow_amd.device import Context, Mesh
    print("cg small", p, bdy, flush=True)
    ne = [3, 2, 3] if p > 2 else [5, 4, 3]
    bg, og = ga.BoxGrid(3, p, ne, bdy=[bdy] * 6), oracle.Grid.box(3, p, ne, bdy=[bdy] * 6)
    m = Mesh(Context(0), bg)
    assert m.flags & 1
    b = og.mass_apply(workloads.unique_normal(bg, seed=p))
    xb = np.zeros(bg.ndof) if bdy == ga.GF_BDY_DIRICHLET else None
    dxb = None if xb is None else _dev(xb)
    for precond in (0, 1):
        # 10 iterations in another summation order: the parity tests' bounds
        xg, info = m.cg_solve(_dev(b), xb=dxb, p=0.1, q=1.0, maxit=10, tol=1e-300, precond=precond)
        xo, _, it, res = og.cg_solve(b, xb=xb, p=0.1, q=np.ones(bg.ndof), maxit=10, tol=1e-300,
                                     normtype=0, precond=precond)
        assert info["iters"] == it == 10
        assert np.abs(xg.cpu().numpy() - xo).max() <= 1e-11 * np.abs(xo).max()
        assert np.abs(info["resid"][:10] - res[:10]).max() <= 1e-10 * np.abs(res[:10]).max()
        # FP32 recurrences end at the FP64 residual's tolerance
        sol = [m.cg_solve(_dev(b), xb=dxb, p=0.1, q=1.0, maxit=4000, tol=1e-11, normtype=4,
                          precond=precond, precision=q) for q in (0, 1)]
        assert sol[0][1]["status"] == sol[1][1]["status"] == 0
        assert _rel(sol[1][0], sol[0][0]) <= 1e-8


def _pair(p, ne):
    from geoflow_amd.device import Context, Mesh
    ctx = Context(0)
    box = ga.BoxGrid(3, p, ne, device_maps=True)
    m, lists = Mesh(ctx, box), Mesh(ctx, _UnionGrid([box], device_maps=True), structured=False)
    assert m.flags & 1 and not lists.flags & 1
    g = torch.Generator(device="cuda").manual_seed(p)
    f = torch.randn(m.ndof, generator=g, device="cuda", dtype=torch.float64)
    return m, lists, m.mass_apply(m.dss(f, "smooth"))


# elements of a workgroup times the largest grids (512 in FP64, 1024 in FP32)
@pytest.mark.parametrize("p,ne", [(1, [41, 41, 40]), (2, [31, 31, 30]), (3, [26, 26, 25]),
                                  (4, [22, 22, 22]), (5, [20, 19, 19]), (6, [17, 17, 15]),
                                  (7, [17, 17, 15]), (8, [15, 15, 14]), (9, [13, 13, 13])])
def test_several_chunks_a_workgroup(p, ne):
    print("cg chunks", p, ne, flush=True)
    m, lists, b = _pair(p, ne)
    kw = dict(p=0.1, q=1.0, precond=1)
    x, info = m.cg_solve(b, maxit=20, tol=1e-300, **kw)
    y, ref = lists.cg_solve(b, maxit=20, tol=1e-300, **kw)
    assert info["iters"] == ref["iters"] == 20
    assert _rel(x, y) <= 1e-12
    for op in ("max", "min"):  # all copies of a node the same
        assert torch.equal(m.dss(x.clone(), op), x)
    kw.update(maxit=4000, tol=1e-11, normtype=4, precision=1)
    x, info = m.cg_solve(b, **kw)
    y, ref = lists.cg_solve(b, **kw)
    assert info["status"] == ref["status"] == 0
    # residuals of 1e-11, and a condition of 1e4 between them and the solutions
    assert _rel(x, y) <= 1e-7
    r = b - m.helmholtz(x, p=0.1, q=1.0)
    nrm = [float((m.dss(v.clone(), "sum") ** 2 * m.imult()).sum().sqrt()) for v in (r, b)]
    assert nrm[0] <= 1.01e-11 * nrm[1]


def test_vectors_beyond_the_cache():
    print("cg beyond the cache", flush=True)
    m, lists, b = _pair(7, [33, 32, 32])
    for precision, its in ((0, 6), (1, 12)):
        assert 4 * m.ndof * (4 if precision else 8) > 256 << 20
        kw = dict(p=0.1, q=1.0, precond=1, precision=precision, normtype=4)
        if precision:
            kw.update(maxit=its, tol=1e-30, inner_tol=1e-30)
        else:
            kw.update(maxit=its, tol=1e-300)
        x, info = m.cg_solve(b, **kw)
        y, ref = lists.cg_solve(b, **kw)
        assert info["iters"] == ref["iters"] == its
        # FP32: 12 iterations of roundings of 6e-8
        assert _rel(x, y) <= (1e-5 if precision else 1e-12)
