"""Box RK stages with a third of the workgroup to each component (few elements)
and with all components in a thread: a periodic box of few elements, checked
against the oracle, and copies of it stacked in z to more elements than the
first form takes, whose fields are the copies of the small box's."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
import geoflow_amd as ga
import oracle

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]

# the parity tests' bound for RK steps
TOL = 1e-12
# elements up to which a stage is split, by nodes per direction
LIMIT = {2: 3072, 3: 3072, 4: 3072, 5: 3072, 6: 8192, 7: 3072, 8: 1024, 9: 3072, 10: 512}


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _rel(a, b):
    return float(np.abs(a.cpu().numpy() - b).max() / np.abs(b).max())


@pytest.mark.parametrize("p", range(1, 10))
def test_split_and_whole_stages(p):
    from geoflow_amd.device import Context, Mesh
    print("stage split", p, flush=True)
    per = [ga.GF_BDY_PERIODIC] * 6
    ne = [3, 2, 2]  # the last workgroup of N <= 5 and of N = 6, 9 partly empty
    k = LIMIT[p + 1] // 12 + 1
    kw = dict(P1=[3.0, 2.0, 2.0], bdy=per)
    small, og = ga.BoxGrid(3, p, ne, **kw), oracle.Grid.box(3, p, ne, **kw)
    big = ga.BoxGrid(3, p, [3, 2, 2 * k], P1=[3.0, 2.0, 2.0 * k], bdy=per, device_maps=True)
    ms, mb = Mesh(Context(0), small), Mesh(Context(0), big)
    assert small.nelems <= LIMIT[p + 1] < big.nelems
    rng = np.random.default_rng(p)
    u0 = [rng.standard_normal(small.ndof) for _ in range(3)]  # discontinuous
    nu, dt = 0.02, 1e-4
    for order in (2, 3, 4):
        us, ub = [_dev(u) for u in u0], [_dev(np.tile(u, k)) for u in u0]
        uo = [u.copy() for u in u0]
        ms.burgers_steps(us, nu, dt, 2, order=order)
        mb.burgers_steps(ub, nu, dt, 2, order=order)
        for _ in range(2):
            og.burgers_step(uo, nu, dt, order=order)
        for a, b, c in zip(us, ub, uo):
            assert _rel(a, c) <= TOL, order
            assert _rel(b, np.tile(c, k)) <= TOL, order
    lam = [rng.standard_normal(small.ndof) for _ in range(3)]
    ls, lb = [_dev(v) for v in lam], [_dev(np.tile(v, k)) for v in lam]
    ms.burgers_adjoint([_dev(u) for u in u0], ls, nu, dt, 2)
    mb.burgers_adjoint([_dev(np.tile(u, k)) for u in u0], lb, nu, dt, 2)
    for a, b in zip(ls, lb):
        assert _rel(b, np.tile(a.cpu().numpy(), k)) <= TOL
