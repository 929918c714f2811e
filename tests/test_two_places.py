"""The places the threads of a two-stage pass (psb_two.h) address in LDS and in
the level's arrays, for every thread of a block and every tile a launch may
choose: inside what the launch asked for, also for the threads of the last wave
that lie past the tile.  Host code of the header, compiled here; CPU only."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

SRC = r"""
#include "psb_two.h"
#include <cstdio>
using namespace psb;
static long bad = 0, seen = 0;
static void want(bool ok, const char *what, const TwoShape &s, int V, int t) {
  seen++;
  if (ok) return;
  if (bad++ < 5) std::printf("%s: RT %d KT %d KO %d V %d thread %d of %d\n", what, s.RT, s.KT,
                             s.KO, V, t, s.threads);
}
template <int V>
static void tile(int ny, int nv, int KO, int R) {
  Grid g{};
  g.nx = 6; g.ny = ny; g.nz = nv * V; g.sI = ny * g.nz; g.N = g.nx * g.sI;
  TwoShape s{};
  s.RT = R + 2;
  s.KO = KO;
  s.KT = KO == nv ? nv : KO + 2;
  s.ntj = (ny + R - 1) / R;
  s.ntk = (nv + KO - 1) / KO;
  s.TI = 4;
  s.nblocks = s.ntj * s.ntk * 2;
  s.threads = (s.RT * s.KT + 63) / 64 * 64;
  const int pitch = s.KT * V, n0 = (s.RT + 2) * pitch, n1 = s.RT * pitch;
  for (int wi = 0; wi < s.nblocks; wi++)
    for (int t = 0; t < kTwoThreads; t++) {  // (a batch launches its largest block)
      const TwoAt a = two_place<V>(g, s, wi, t);
      const int own0 = (a.rr + 1) * pitch + a.kk * V, own1 = a.rr * pitch + a.kk * V;
      want(own0 >= 0 && own0 + V <= n0, "operand", s, V, t);
      want(own1 >= 0 && own1 + V <= n1, "swept", s, V, t);
      if (a.in) {
        want(own0 + a.os >= 0 && own0 + a.on + V <= n0, "operand rows", s, V, t);
        want(own0 + a.ob >= 0 && own0 + a.ot < n0, "operand ends", s, V, t);
      }
      if (a.out) {
        want(own1 + a.os >= 0 && own1 + a.on + V <= n1, "swept rows", s, V, t);
        want(own1 + a.ob >= 0 && own1 + a.ot < n1, "swept ends", s, V, t);
      }
      if (a.halo) want(a.hrow >= 0 && (a.hrow + 1) * V <= n0, "halo", s, V, t);
      const uint32_t last = (uint32_t)(g.sI - V);
      want(a.P <= last && a.HP <= last && a.Pn <= last && a.Pt <= last, "plane", s, V, t);
      want(a.i0 >= 0 && a.i0 < a.i1 && a.i1 <= g.nx, "slab", s, V, t);
    }
}
int main() {
  for (int nv = 1; nv <= 192; nv++) {
    const int KT = nv;
    for (int R = 2; (R + 2) * KT <= kTwoThreads; R += nv < 4 ? 22 : 2) {
      tile<4>(R + 3, nv, nv, R);
      tile<2>(R + 3, nv, nv, R);
    }
  }
  for (int KO : {64, 32, 16})
    for (int R = 2; (R + 2) * (KO + 2) <= kTwoThreads; R += 2) {
      tile<4>(2 * R + 2, 2 * KO + 3, KO, R);
      tile<2>(2 * R + 2, 2 * KO + 3, KO, R);
    }
  std::printf("%ld checks, %ld outside\n", seen, bad);
  return bad != 0;
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_every_thread_stays_inside_its_tile(tmp_path):
    src, exe = tmp_path / "places.hip", tmp_path / "places"
    src.write_text(SRC)
    subprocess.check_call([HIPCC, "--offload-host-only", "-O2", "-std=c++17", "-w",
                           "-I" + os.path.join(ROOT, "psi-boil_amd", "csrc"), str(src),
                           "-o", str(exe)])
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
