"""LDS of the constant-viscosity apply (diff_plan.hpp): every wavefront that a
launch starts, those past the last vertex included, stays inside the doubles
that the host reserves for it.  The header is plain C++, compiled here."""
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = """
#include "diff_plan.hpp"
#include <cstdio>
#include <vector>
// stdin: vertices, vertices per wavefront, wavefronts per workgroup, then each
// vertex's stored faces and faces; out: reserved doubles, the fullest launched
// wavefront's need, wavefronts without a vertex
int main() {
  long V; int per, waves;
  if (scanf("%ld %d %d", &V, &per, &waves) != 3) return 1;
  std::vector<int> size(V);
  for (long v = 0; v < V; v++) {
    int ni, nf;
    if (scanf("%d %d", &ni, &nf) != 2) return 1;
    size[v] = sfv::apply_lds<false>(ni, nf);
  }
  const int reserved = sfv::apply_lds_wave(V, per, [&](long v) { return size[v]; });
  const long groups = (V + (long)per * waves - 1) / ((long)per * waves);
  int most = 0, spare = 0;
  for (long w = 0; w < groups * waves; w++) {
    int sum = 0;
    for (int g = 0; g < per; g++) {
      const long v = sfv::apply_vertex(w, per, g, V);
      if (v < 0) { spare++; break; }
      if (v >= V) return 2;
      sum += size[v];
    }
    if (sum > most) most = sum;
  }
  printf("%d %d %d", reserved, most, spare);
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    src, exe = d / "plan.cpp", d / "plan"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "subfv_amd", "csrc"), "-o", str(exe),
                    str(src)], check=True)

    def run(per, waves, faces):
        text = f"{len(faces)} {per} {waves}\n" + "\n".join(f"{a} {b}" for a, b in faces)
        out = subprocess.run([str(exe)], input=text, capture_output=True, text=True, check=True).stdout
        return [int(x) for x in out.split()]
    return run


@pytest.mark.parametrize("per,waves", [(4, 4), (4, 1), (2, 4), (2, 1)])
@pytest.mark.parametrize("n", [1, 2, 3, 5, 16, 17, 18, 21, 33])
def test_launched_wavefronts_fit_their_lds(plan, per, waves, n):
    """The last vertex is the largest, as a pole of a shell of hexahedra with
    prisms around it can be: 12 stored faces where the others have 4."""
    small, large = (4, 8), (12, 24)
    reserved, most, spare = plan(per, waves, [small] * (n - 1) + [large])
    assert most <= reserved
    assert spare == -(-n // (per * waves)) * waves - (-(-n // per))
    # no more than the fullest of them needs
    assert reserved == most


def test_random_sizes_fit(plan):
    rng = np.random.default_rng(4)
    for n in rng.integers(1, 70, 12):
        nf = rng.integers(0, 40, n)
        ni = (nf * rng.random(n)).astype(int).clip(0, 10)
        for per in (4, 2):
            reserved, most, _ = plan(per, 4, list(zip(ni, nf)))
            assert most == reserved
