"""gf_time_kernel's kernels run on data that stay finite (it checks its fields
after the repetitions): a kernel timed on infinities or NaN is not the kernel that
a solve runs."""
import pytest

torch = pytest.importorskip("torch")
import geoflow_amd as ga

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


@pytest.mark.parametrize("bdy", [ga.GF_BDY_DIRICHLET, ga.GF_BDY_PERIODIC])
@pytest.mark.parametrize("p", [2, 5, 7])
def test_timed_kernels_stay_finite(p, bdy):
    from geoflow_amd.device import Context, Mesh
    print("time kernel", p, bdy, flush=True)
    m = Mesh(Context(0), ga.BoxGrid(3, p, [3, 2, 2], bdy=[bdy] * 6))
    for which in ("cg_update", "cg_update_f32", "cg_apply", "cg_apply_f32", "burgers_stage",
                  "burgers_stage_box", "rk_out_box", "helmholtz"):
        assert m.time_kernel(which, reps=20) > 0.0, which
