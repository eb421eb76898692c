"""The rule that lets an event read a point's second shell at fixed index
steps (shell_inside, mskg_lattice.h), compiled for the host: it holds exactly
for the points whose shell, (+-6, +-6, 0) and permutations, neither wraps nor
leaves the box, at every point of boxes lower and higher than two shell steps,
and the steps then give the shell's own points."""
import os
import shutil
import subprocess

import pytest

from mulskips_amd import _build

ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
PROGRAM = r"""
#include "mskg_lattice.h"
#include <cstdio>
using namespace mskg;
int main() {
  long inside = 0, wrong = 0;
  for (int lx : {12, 24, 36})
    for (int ly : {12, 24})
      for (int lz = 1; lz <= 26; lz++) {
        const Box b = make_box(lx, ly, lz);
        for (int64_t p = 0; p < b.npts; p++) {
          int x, y, z;
          pxyz(b, p, x, y, z);
          bool in = true, steps = true;
          for (int k = 0; k < 12; k++) {
            const int a = (k & 2) ? -6 : 6, c = (k & 1) ? -6 : 6, g = k >> 2;
            const int dx = g == 2 ? 0 : a, dy = g == 0 ? c : (g == 1 ? 0 : a), dz = g == 0 ? 0 : c;
            const int64_t q = pidx_checked(b, x + dx, y + dy, z + dz);
            in &= q >= 0;
            steps &= q == p + dz * b.plane + (int64_t)(dy / 2) * b.hx + dx / 2;
          }
          const bool says = shell_inside(b, x, y, z);
          inside += says;
          if (says != in || (says && !steps)) {
            if (!wrong) printf("box %d %d %d, point (%d,%d,%d): rule %d, shell inside %d\n", lx, ly, lz, x, y, z, says, in);
            wrong++;
          }
        }
      }
  printf("%ld %ld\n", inside, wrong);
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_rule_holds_exactly_where_the_shell_lies_in_the_box(tmp_path):
    src = tmp_path / "shell.cpp"
    src.write_text(PROGRAM)
    exe = str(tmp_path / "shell")
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-D__align__(n)=__attribute__((aligned(n)))",
                    "-I", os.path.join(ROCM, "include"), "-I", os.path.join(_build.HERE, "csrc"), str(src), "-o", exe],
                   check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout.splitlines()
    inside, wrong = (int(v) for v in out[-1].split())
    assert inside > 0 and wrong == 0, out
