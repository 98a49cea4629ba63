"""Fused right-hand side, advection and gradient kernels of regular meshes
against the oracle, at every element order and at element counts that leave
the last workgroup partly empty."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
import geoflow_amd as ga
import oracle

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]

# FP64 sums of at most 3 (p + 1) products per node and their transposes: the
# parity tests' 1e-12 of the largest value
TOL = 1e-12


def _rel(a, b):
    return float(np.abs(a.cpu().numpy() - b).max() / np.abs(b).max())


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("dim,p,ne", [(3, 1, [3, 2, 1]), (3, 2, [5, 1, 3]), (3, 3, [2, 3, 2]),
                                      (3, 4, [3, 1, 1]), (3, 5, [1, 1, 1]), (3, 6, [3, 2, 1]),
                                      (3, 7, [2, 1, 3]), (3, 8, [2, 2, 1]), (3, 9, [1, 3, 1]),
                                      (2, 3, [5, 3]), (2, 11, [2, 1])])
def test_fused_operators(dim, p, ne):
    from geoflow_amd.device import Context, Mesh
    P1 = [1.3, 0.8, 2.1][:dim]
    bdy = [ga.GF_BDY_DIRICHLET] * (2 * dim)
    bg, og = ga.BoxGrid(dim, p, ne, P1=P1, bdy=bdy), oracle.Grid.box(dim, p, ne, P1=P1, bdy=bdy)
    m = Mesh(Context(0), bg)
    rng = np.random.default_rng(p)
    us = [rng.standard_normal(bg.ndof) for _ in range(dim)]
    q = rng.standard_normal(bg.ndof)
    dus, dq = [_dev(u) for u in us], _dev(q)
    for nu in (1.0, 0.03):
        for a, b in zip(m.burgers_rhs(dus, nu), og.burgers_rhs(us, nu)):
            assert _rel(a, b) <= TOL
    assert _rel(m.advect(dq, dus), og.advect(q, us)) <= TOL
    for d, g in enumerate(m.grad(dq)):
        assert _rel(g, og.deriv(q, d + 1)) <= TOL
    for d, g in enumerate(m.grefderivs(dq)):
        assert _rel(g, og.grefderiv(q, d + 1)) <= TOL
    # a missing component is a zero velocity
    if dim == 3:
        import ctypes
        from geoflow_amd._capi import lib
        from geoflow_amd.device import _ptr
        vp = ctypes.c_void_p
        out = m.new()
        v = (vp * 3)(None, dus[1].data_ptr(), None)
        m._c(lib().gf_advect(m.h, _ptr(dq), 3, v, _ptr(out)))
        z = np.zeros(bg.ndof)
        assert _rel(out, og.advect(q, [z, us[1], z])) <= TOL
        # fewer components than directions
        assert _rel(m.advect(dq, dus[:2]), og.advect(q, us[:2] + [z])) <= TOL


@pytest.mark.parametrize("p,ne,bdy", [(1, [3, 2, 1], 0), (2, [5, 1, 3], 6), (3, [2, 3, 2], 0),
                                      (4, [3, 1, 1], 6), (5, [1, 1, 1], 6), (6, [3, 2, 1], 6),
                                      (7, [2, 1, 3], 0), (8, [2, 2, 1], 6), (9, [1, 2, 1], 0)])
def test_fused_adjoint(p, ne, bdy):
    """The adjoint kernels at every element order: the right-hand side's
    adjoint added to a cotangent, and the step's adjoint of orders 2-4 on the
    box path from a discontinuous state, against the oracle."""
    from geoflow_amd.device import Context, Mesh
    bg, og = ga.BoxGrid(3, p, ne, bdy=[bdy] * 6), oracle.Grid.box(3, p, ne, bdy=[bdy] * 6)
    m = Mesh(Context(0), bg)
    rng = np.random.default_rng(40 + p)
    f = lambda: [rng.standard_normal(bg.ndof) for _ in range(3)]  # noqa: E731
    u, w, l0 = f(), f(), f()
    ref = og.burgers_rhs_adjoint(u, w, [a.copy() for a in l0], 0.03)
    got = m.burgers_rhs_adjoint([_dev(a) for a in u], [_dev(a) for a in w],
                                [_dev(a) for a in l0], 0.03)
    for a, b in zip(got, ref):
        assert _rel(a, b) <= TOL
    for order in (2, 3, 4):
        dt = 1e-3 / (p + 1) ** 4
        ref = og.burgers_step_adjoint(u, [a.copy() for a in w], 0.04, dt, order=order)
        got = m.burgers_step_adjoint([_dev(a) for a in u], [_dev(a) for a in w], 0.04, dt,
                                     order=order)
        for a, b in zip(got, ref):
            assert _rel(a, b) <= TOL, order


@pytest.mark.parametrize("order", [2, 3, 4])
@pytest.mark.parametrize("p,ne,bdy", [(1, [5, 3], [6] * 4), (2, [1, 1], [6] * 4),
                                      (4, [7, 3], [0] * 4), (5, [3, 2], [6, 6, 0, 0]),
                                      (7, [2, 5], [6] * 4), (11, [3, 1], [0] * 4)])
def test_steps_2d(p, ne, bdy, order):
    """2-D steps from a state whose copies of a node disagree against the
    oracle, n steps in a call equal to n calls bit for bit, and the state
    continuous afterwards; boxes of both kinds of direction too."""
    from geoflow_amd.device import Context, Mesh
    bg, og = ga.BoxGrid(2, p, ne, bdy=bdy), oracle.Grid.box(2, p, ne, bdy=bdy)
    m = Mesh(Context(0), bg)
    rng = np.random.default_rng(7 * p + order)
    us = [np.cos(2 * np.pi * (bg.xyz[0] + c * bg.xyz[1])) + 0.1 * rng.standard_normal(bg.ndof)
          for c in range(2)]
    dt = 1e-3 / (p + 1) ** 4
    ref, one = [u.copy() for u in us], [_dev(u) for u in us]
    for n in range(1, 4):
        og.burgers_step(ref, 0.02, dt, order=order)
        m.burgers_step(one, 0.02, dt, order=order)
        many = [_dev(u) for u in us]
        m.burgers_steps(many, 0.02, dt, n, order=order)
        for c in range(2):
            assert _rel(many[c], ref[c]) <= TOL, (n, c)
            assert torch.equal(many[c], one[c]), (n, c)
            assert torch.equal(m.dss(many[c].clone(), "max"), many[c]), (n, c)
