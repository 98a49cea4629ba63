"""Rounding of a pure-advection RK step on the sphere: the error of the result
against extended precision (rms over the nodes, ten states) is no larger than
that of the oracle, which does step_b's operations one by one in FP64.  The step
is so short that its value is u + dt S(F(u)) (dt^2 |F'F| is below 1e-3 of an
ulp), formed in extended precision from the device's right-hand side."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
import geoflow_amd as ga
import oracle

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


@pytest.mark.parametrize("order", [1, 2, 3, 4])
@pytest.mark.parametrize("p,lev", [(3, 2), (5, 2), (6, 1)])
def test_step_rounds_no_more_than_step_b(p, lev, order):
    from geoflow_amd.device import Context, Mesh
    print("sphere rounding", p, lev, order, flush=True)
    g, og = ga.IcosGrid(p, lev, radius=1.0), oracle.Grid.icos(p, lev, radius=1.0)
    m = Mesh(Context(0), g)
    x, y, z = g.xyz
    offs, mem = np.asarray(g.ggfx_offs), np.asarray(g.ggfx_members)
    cnt = np.diff(offs)
    vel = [np.ascontiguousarray(a) for a in (-y, x, 0.0 * z)]
    nu, dt = 1e-3, 1e-12
    dev = ora = 0.0
    for seed in range(10):
        a = np.random.default_rng(seed).standard_normal(6)
        h = a[0] * x * y + a[1] * z + a[2] * np.sin(3 * x + a[3]) + a[4] * np.cos(4 * y * z + a[5])
        h = h[mem[offs[:-1]]]  # the same at every copy of a node
        d = [torch.from_numpy(q.copy()).cuda() for q in [h] + vel]
        K = m.burgers_rhs(d, nu, mode=1)[0].cpu().numpy().astype(np.longdouble)
        ref = h + np.longdouble(dt) * (np.add.reduceat(K[mem], offs[:-1]) / cnt)
        o = [h.copy()] + [v.copy() for v in vel]
        m.burgers_steps(d, nu, dt, 1, mode=1, order=order)
        og.burgers_step(o, nu, dt, mode=1, order=order)
        dev += float(((d[0].cpu().numpy() - ref) ** 2).sum())
        ora += float(((o[0] - ref) ** 2).sum())
    print((dev / ora) ** 0.5, flush=True)
    assert dev <= ora
