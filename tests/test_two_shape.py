"""The tile of a level's two-stage passes (two_shape, psb_two.h) is the cheapest
of every row count and slab depth, the first one of equal cost, and is found
without walking them all: the search is part of every new matrix's first solve.
Host code of the header, compiled here; CPU only."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

SRC = r"""
#include "psb_two.h"
#include <algorithm>
#include <chrono>
#include <cstdio>
#include <cstring>
using namespace psb;
// every row count, every even depth
template <typename T>
static TwoShape walk(const Grid &g) {
  constexpr int V = 16 / (int)sizeof(T);
  TwoShape s{};
  if (g.nz % V) return s;
  const int nv = g.nz / V;
  double best = 0.0;
  for (int KO : {nv, 64, 32, 16}) {
    if (KO > nv || (KO != nv && best > 0.0)) continue;
    const int KT = KO == nv ? nv : KO + 2, ntk = (nv + KO - 1) / KO;
    for (int R = 2; (R + 2) * KT <= kTwoThreads; R += 2) {
      const size_t lds = (size_t)(2 * (R + 4) + 2 * (R + 2) + R) * KT * V;
      if (lds * sizeof(T) > 150 * 1024) break;
      const int waves = ((R + 2) * KT + 63) / 64, per_cu = std::max(1, 12 / waves);
      const int ntj = (g.ny + R - 1) / R;
      for (int TI = 2; TI < g.nx + 2; TI += 2) {
        const long long nb = (long long)ntj * ntk * ((g.nx + TI - 1) / TI);
        const long long rounds = (nb + 256 * per_cu - 1) / (256 * per_cu);
        const long long act = std::min<long long>(per_cu, (nb + 255) / 256);
        const double cost = (double)rounds * (TI + 2) * (4 + waves * act);
        if (nb >= (1 << 30) || (best > 0.0 && cost >= best)) continue;
        best = cost;
        s = TwoShape{R + 2, KT, KO, ntj, ntk, TI, (int)nb, waves * 64, lds};
      }
    }
  }
  return s;
}
static double t_walk, t_search;
template <typename T>
static bool same(int nx, int ny, int nz) {
  Grid g{};
  g.nx = nx; g.ny = ny; g.nz = nz; g.sI = ny * nz; g.N = nx * g.sI;
  auto t0 = std::chrono::steady_clock::now();
  const TwoShape a = walk<T>(g);
  auto t1 = std::chrono::steady_clock::now();
  const TwoShape b = two_shape<T>(g);
  auto t2 = std::chrono::steady_clock::now();
  t_walk += std::chrono::duration<double>(t1 - t0).count();
  t_search += std::chrono::duration<double>(t2 - t1).count();
  const bool ok = a.RT == b.RT && a.KT == b.KT && a.KO == b.KO && a.ntj == b.ntj &&
                  a.ntk == b.ntk && a.TI == b.TI && a.nblocks == b.nblocks &&
                  a.threads == b.threads && a.lds == b.lds;
  if (!ok) std::printf("%d x %d x %d, %d bytes: TI %d RT %d against TI %d RT %d\n", nx, ny, nz,
                       (int)sizeof(T), b.TI, b.RT, a.TI, a.RT);
  return ok;
}
int main() {
  bool ok = true;
  const int n[] = {1, 2, 3, 4, 7, 8, 12, 16, 21, 24, 32, 36, 48, 64, 100, 128, 200, 256, 400};
  for (int nx : n)
    for (int ny : n)
      for (int nz : {2, 4, 6, 8, 12, 16, 32, 44, 64, 128, 384, 400, 512, 800, 1024, 1600, 7})
        ok = same<float>(nx, ny, nz) && same<double>(nx, ny, nz) && ok;
  t_walk = t_search = 0.0;
  for (int q = 0; q < 5; q++)
    ok = same<float>(1024, 1024, 8) && same<double>(512, 512, 16) && same<float>(2048, 512, 12) &&
         ok;
  std::printf("walk %.3f ms, search %.3f ms\n", t_walk * 1e3, t_search * 1e3);
  return ok ? t_walk > 5.0 * t_search ? 0 : 2 : 1;
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_search_finds_the_cheapest_tile(tmp_path):
    src, exe = tmp_path / "shape.hip", tmp_path / "shape"
    src.write_text(SRC)
    subprocess.check_call([HIPCC, "--offload-host-only", "-O2", "-std=c++17", "-w",
                           "-I" + os.path.join(ROOT, "psi-boil_amd", "csrc"), str(src),
                           "-o", str(exe)])
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, (r.returncode, r.stdout)
    print(r.stdout)
