"""CPU check of the bounded sweeps' copies into LDS over every block they plan:
csrc/bounded_impl.h compiled for the host, the copy of the tables and of a
stretched mesh's metrics run thread by thread for every line length, precision
and number of tables that has a plan.  Every word has to arrive, also where a
block has fewer threads than its lines have points (single precision from 758
points on)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include <cstdio>
#include <vector>
#include "bounded_impl.h"
using namespace x3d;
template <typename T, int N, int R>
static bool copied(int nthr, int words) {
  std::vector<T> table(N * words), lds(N * words, T(-1));
  const T *src[N];
  for (int t = 0; t < N; ++t) {
    src[t] = &table[t * words];
    for (int i = 0; i < words; ++i) table[t * words + i] = T(t * words + i);
  }
  for (int tid = 0; tid < nthr; ++tid) {
    BoundCopy<T, N, R> c;
    c.load(src, tid, nthr, words);
    c.store(lds.data(), src, tid, nthr, words);
  }
  return lds == table;
}
template <typename T, int NT>
static int walk(const char *name) {
  int bad = 0, plans = 0, few = 0;
  for (int stretched = 0; stretched < 2; ++stretched)
    for (int n = 16; n <= 1100; ++n) {
      BoundPick<T> Y;
      if (!Y.plan(n, NT, 3, [&](int) { return stretched ? 3 * (size_t)n : (size_t)0; })) continue;
      ++plans;
      const int L = BoundShape<T>::L + (Y.longer ? 1 : 0), nthr = Y.TL * Y.P;
      few += stretched && nthr < n;
      bool ok = nthr <= 1024 && Y.P * L >= n && copied<T, NT, 2>(nthr, 4 * Y.P * L);
      if (stretched) ok = ok && copied<T, 3, 1>(nthr, n);
      bad += !ok;
    }
  std::printf("%s %d tables: plans %d, stretched with fewer threads than points %d, bad %d\n", name, NT, plans, few, bad);
  return bad || !plans;
}
int main() { return walk<double, 2>("f64") + walk<double, 3>("f64") + walk<float, 2>("f32") + walk<float, 3>("f32"); }
"""


def test_tables_and_metrics_reach_lds(tmp_path):
    from incompact3d_amd import build as b
    try:
        cc = b.hipcc()
    except RuntimeError:
        pytest.skip("hipcc not found")
    src, exe = tmp_path / "plan.cpp", tmp_path / "plan"
    src.write_text(SRC)
    r = subprocess.run([cc, "-O1", "-std=c++17", "-x", "hip", f"--offload-arch={b.ARCH}",
                        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-I", b.CSRC,
                        str(src), "-o", str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
