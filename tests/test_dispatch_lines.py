"""The size lines of the dispatch (gf_internal.hpp) lie where the tests of both
sides of them (test_stage_split.py, test_cg_update.py) take them to lie: were a
line moved, both of their meshes could run one form and still pass."""
import os
import subprocess

import test_cg_update
import test_stage_split

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _lines(tmp_path):
    src = tmp_path / "lines.cpp"
    src.write_text('#include "gf_internal.hpp"\n#include <cstdio>\n'
                   'int main() {\n'
                   '  for (int N = 2; N <= 10; N++) printf("%zu ", stage_split_max(N));\n'
                   '  printf("%zu\\n", kNrefMax);\n}\n')
    exe = str(tmp_path / "lines")
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "include"),
                    "-I" + os.path.join(ROOT, "geoflow_amd", "csrc"), str(src), "-o", exe],
                   check=True, capture_output=True)
    v = [int(x) for x in subprocess.run([exe], check=True, capture_output=True,
                                        text=True).stdout.split()]
    return dict(zip(range(2, 11), v[:9])), v[9]


def test_lines_lie_between_the_tests_meshes(tmp_path):
    split, nref = _lines(tmp_path)
    assert split == test_stage_split.LIMIT
    cases = [c for mark in test_cg_update.test_cg_update_2d.pytestmark
             if mark.name == "parametrize" and mark.args[0] == "p,ne" for c in mark.args[1]]
    nodes = sorted(ne[0] * ne[1] * (p + 1) ** 2 for p, ne in cases)
    assert nodes[-2] <= nref < nodes[-1]
