"""The lanes' face nodes of the 3D stage (face_node_of in euler3d_stage.hpp) on
the host, for every polydeg and workgroup shape: the lanes of all passes hold
each face node of the workgroup's elements once, and a lane without one is left
with a slot of the workgroup, so that the LDS read which follows on every lane
(slot, direction, node of [slots][9][n^3]) stays inside its array."""
import os
import shutil
import subprocess

import pytest

HIPCC = "/opt/rocm/bin/hipcc"
CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "trixiatmo.jl_amd", "csrc")

SOURCE = r"""
#include <cstdio>
#include <vector>
#include "euler3d_stage.hpp"
using namespace atmo;

template <int N, int EPB>
int check() {
  using F = FacePrefetch<N, EPB>;
  constexpr int N2 = N * N, N3 = N2 * N;
  int bad = 0;
  for (int n_valid = 1; n_valid <= F::SLOTS; ++n_valid) {
    std::vector<int> seen(F::SLOTS * F::NF, 0);
    for (int ps = 0; ps < F::PASSES; ++ps)
      for (int t = 0; t < F::GB; ++t) {
        int es = 0, fid = 0, f = 0, d = 0, node = 0;
        const bool has = face_node_of<N, EPB>(t, ps, n_valid, es, fid, f, d, node);
        const bool inside = es >= 0 && es < F::SLOTS && fid >= 0 && fid < F::NF && d >= 0 &&
                            d < 3 && node >= 0 && node < N3;
        if (!inside) {
          if (bad++ < 4)
            std::printf("N %d EPB %d n_valid %d pass %d lane %d: slot %d node %d\n", N, EPB,
                        n_valid, ps, t, es, node);
          continue;
        }
        if (!has) continue;
        const int c[3] = {node % N, (node / N) % N, node / N2};
        if (d != f / 2 || f != fid / N2 || c[d] != (f % 2 ? N - 1 : 0)) ++bad;
        ++seen[es * F::NF + fid];
      }
    for (int q = 0; q < F::SLOTS * F::NF; ++q) bad += seen[q] != (q < n_valid * F::NF);
  }
  return bad;
}

int main() {
  const int bad = check<2, 1>() + check<3, 1>() + check<4, 1>() + check<5, 1>() + check<6, 1>() +
                  check<7, 1>() + check<8, 1>() + check<4, 2>() + check<5, 2>() + check<2, 0>() +
                  check<3, 0>() + check<4, 0>() + check<5, 0>() + check<6, 0>() + check<7, 0>();
  std::printf("%d wrong\n", bad);
  return bad != 0;
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC) or shutil.which("g++") is None,
                    reason="needs hipcc")
def test_face_nodes_of_every_shape(tmp_path):
    src, exe = tmp_path / "slots.hip", tmp_path / "slots"
    src.write_text(SOURCE)
    build = subprocess.run([HIPCC, "--cuda-host-only", "-O1", "-std=c++17", f"-I{CSRC}", str(src),
                            "-o", str(exe)], capture_output=True, text=True, timeout=300)
    assert build.returncode == 0, build.stderr[-4000:]
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout
