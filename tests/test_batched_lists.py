"""Batched CG on members that are not the boxes the mesh was made of (two boxes
joined to one member), and on a mesh that was not told of its boxes: q is
assembled from the group lists, or, on more than 786432 nodes, by DSS passes.
Members that converge at different iterations, FP64 and mixed, against the same
members each solved alone."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
import geoflow_amd as ga
from geoflow_amd.ensemble import _UnionGrid
from geoflow_amd import workloads

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("big", [False, True])
@pytest.mark.parametrize("joined", [False, True])
def test_members_without_boxes(joined, big, precision):
    from geoflow_amd.device import Context, Mesh
    print("batched lists", joined, big, precision, flush=True)
    ctx = Context(0)
    p = 4
    nes = [2, 4, 3] + ([19] if big else [])  # 19^3 elements: 857375 nodes
    grids = [ga.BoxGrid(3, p, [n] * 3, device_maps=True) for n in nes]
    ug = _UnionGrid(grids, device_maps=True)
    m = Mesh(ctx, ug, structured=False)
    assert (m.ndof > 3 << 18) == big
    off = np.cumsum([0] + [g.nelems for g in grids])
    if joined:
        eoff = [0] + list(off[2:])  # the first two boxes are one member
    else:
        # the boxes' groups in host lists, and no box named
        og, mg = [np.zeros(1, np.int64)], []
        for g, e in zip(grids, off):
            from geoflow_amd.device import box_ggfx_device
            o, q = box_ggfx_device(ctx, p + 1, g.ne, g.periodic)
            og.append(o[1:] + og[-1][-1])
            mg.append(q + e * (p + 1) ** 3)
        ug.ggfx_offs, ug.ggfx_members = np.concatenate(og), np.concatenate(mg)
        ug.device_maps, ug.box_list = False, None
        m = Mesh(ctx, ug, structured=False)
        eoff = list(off)
    m.set_segments(eoff)
    rng = np.random.default_rng(7)
    # a smooth, a rough and a mixed right-hand side: different iteration counts
    f = torch.from_numpy(np.concatenate(
        [rng.standard_normal(g.ndof) * 10.0 ** k for k, g in enumerate(grids)])).cuda()
    b = m.mass_apply(m.dss(f, "smooth"))
    kw = dict(p=0.02, q=1.0, maxit=4000, normtype=4, precond=1, precision=precision)
    x, info = m.cg_solve(b, tol=1e-11, **kw)
    assert info["status"] == 0
    its = m.member_results()[0]
    assert len(set(int(i) for i in its)) > 1  # members end at different iterations
    nn = (p + 1) ** 3
    for k in range(len(eoff) - 1):
        sub = [g for g, e in zip(grids, off) if eoff[k] <= e < eoff[k + 1]]
        alone = Mesh(ctx, _UnionGrid(sub, device_maps=True), structured=False)
        sl = slice(int(eoff[k]) * nn, int(eoff[k + 1]) * nn)
        y, one = alone.cg_solve(b[sl].clone(), tol=1e-11, **kw)
        assert one["status"] == 0
        # the same recurrence with other partial sums: the count may move by
        # what the last digits of a residual move
        assert abs(int(its[k]) - one["iters"]) <= 2 + one["iters"] // (10 if precision else 50)
        assert float((x[sl] - y).abs().max() / y.abs().max()) <= 1e-9
