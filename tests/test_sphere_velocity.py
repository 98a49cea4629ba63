"""Pure advection on the sphere whose velocity has the state as one of its
components: steps in one call give what single calls give, bit for bit, as they
do with a velocity of its own."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
import geoflow_amd as ga

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


@pytest.mark.parametrize("comp", [None, 0, 2])
@pytest.mark.parametrize("order", [1, 2, 3, 4])
def test_steps_equal_single_calls(order, comp):
    from geoflow_amd.device import Context, Mesh
    print("sphere velocity", order, comp, flush=True)
    g = ga.IcosGrid(3, 1, radius=1.0)
    m = Mesh(Context(0), g)
    x, y, z = g.xyz

    def state():
        h = torch.from_numpy(1.0 + 0.5 * x * y + 0.2 * z).cuda()
        v = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (-y, x, 0.0 * z)]
        if comp is not None:
            v[comp] = h
        return [h] + v

    a, b = state(), state()
    m.burgers_steps(a, 1e-3, 5e-3, 3, mode=1, order=order)
    for _ in range(3):
        m.burgers_steps(b, 1e-3, 5e-3, 1, mode=1, order=order)
    assert torch.equal(a[0], b[0])
    assert not torch.equal(a[0], state()[0])
