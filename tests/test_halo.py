"""The LDS halo of the structured-box RK stages: its fill and its group sums'
order on the CPU at every element order (tests/halo_check.cpp), and the steps
that use it against the oracle on the GPU."""
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def test_halo_groups(tmp_path):
    exe = str(tmp_path / "halo_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "geoflow_amd", "csrc"),
                    "-I", "/opt/rocm/include", "-D__HIP_PLATFORM_AMD__",
                    os.path.join(HERE, "halo_check.cpp"), "-o", exe],
                   check=True, capture_output=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.gpu
@pytest.mark.parametrize("order", [2, 3, 4])
@pytest.mark.parametrize("p,ne,bdy", [(1, [3, 2, 4], 6), (2, [5, 1, 2], 6), (3, [2, 3, 2], 0),
                                      (4, [1, 1, 1], 6), (4, [3, 2, 1], 0), (5, [3, 1, 2], 6),
                                      (6, [2, 1, 3], 6), (7, [3, 2, 2], 0), (7, [1, 3, 2], 6),
                                      (8, [2, 2, 1], 6), (9, [1, 2, 2], 0)])
def test_box_steps_every_order(p, ne, bdy, order):
    """Steps of the box path at every element order, from a state whose copies
    of a node disagree (step_b smooths the final-stage input, the first three
    stages read the state as it is), against the oracle's steps: 1e-12 of the
    largest value, as the other step tests."""
    import torch
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    import geoflow_amd as ga
    import oracle
    from geoflow_amd.device import Context, Mesh
    bg = ga.BoxGrid(3, p, ne, bdy=[bdy] * 6)
    og = oracle.Grid.box(3, p, ne, bdy=[bdy] * 6)
    m = Mesh(Context(0), bg)
    assert m.flags & 1
    rng = np.random.default_rng(100 * p + order)
    us = [np.cos(2 * np.pi * (bg.xyz[0] + c * bg.xyz[1])) + 0.3 * np.sin(2 * np.pi * bg.xyz[2])
          + 0.1 * rng.standard_normal(bg.ndof) for c in range(3)]
    ref = [u.copy() for u in us]
    # a small step: the noise must not grow over the three steps
    dt = 1e-3 / (p + 1) ** 4
    for n in range(1, 4):
        og.burgers_step(ref, 0.02, dt, order=order)
        dus = [torch.from_numpy(u).cuda() for u in us]
        m.burgers_steps(dus, 0.02, dt, n, order=order)
        for c in range(3):
            err = np.abs(dus[c].cpu().numpy() - ref[c]).max() / np.abs(ref[c]).max()
            assert err <= 1e-12, (n, c)
