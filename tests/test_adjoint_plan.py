"""How many segments of an adjoint solve stay resident (dg_adj_plan.h): never
more than what the solve then allocates fits into the memory it may use, the
work arrays included, and never fewer than fit it and the setting."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include "dg_adj_plan.h"
#include <cstdio>
#include <cstdlib>
using dgk::AdjPlan;
using dgk::adj_stride;
// what the solve allocates, buffer by buffer
static size_t held(const AdjPlan &p, int nres) {
  const int n = p.nseg();
  size_t b = (size_t)(p.S + 2) * adj_stride(p.sb) + p.eps_b;  // stage weights, two g
  auto seg = [&](int ns) {
    size_t x = 0;
    for (int i = 0; i < ns * p.S + 1; i++) x += adj_stride(p.sb);
    if (p.kst_b) for (int i = 0; i < ns * p.S; i++) x += adj_stride(p.kst_b);
    return x;
  };
  for (int q = 0; q < n; q++) {
    const bool resident = q >= n - nres, walked = nres == 0 && q == n - 1;
    if (resident) b += seg(p.len(q));
    else if (!walked) b += adj_stride(p.sb);  // a checkpoint
  }
  if (nres < n) b += seg(p.every);
  return b;
}
int main() {
  long cases = 0, some = 0, full = 0;
  for (int S = 2; S <= 4; S++)
    for (int nsteps : {1, 2, 7, 16, 33, 100})
      for (int every : {1, 3, 10, 16, 100})
        for (size_t sb : {(size_t)24, (size_t)1 << 20, (size_t)3 << 30})
          for (int eps = 0; eps < 2; eps++) {
            if (every > nsteps) continue;
            AdjPlan p{nsteps, every, S, sb, eps ? sb * 2 / 3 : 0, eps ? 2 * adj_stride(sb / 8) : 0};
            const size_t top = held(p, p.nseg());
            for (int k = 0; k <= 24; k++) {
              const size_t avail = held(p, 0) / 2 + top / 20 * k;
              for (double cap : {1e30, (double)top / 3, (double)sb / 2}) {
                const int r = p.resident(cap, avail);
                cases++;
                some += r > 0;
                full += r == p.nseg();
                if (r < 0 || r > p.nseg() || (r && held(p, r) > avail)) {
                  std::printf("S %d steps %d every %d sb %zu eps %d avail %zu: %d resident need %zu\n",
                              S, nsteps, every, sb, eps, avail, r, held(p, r));
                  return 1;
                }
                // as many as the memory holds where the setting does not bind
                // (all but segment 0, then all)
                if (cap == 1e30 && r < p.nseg() - 1 && held(p, r + 1) <= avail) return 2;
                if (cap == 1e30 && r < p.nseg() && top <= avail) return 3;
                if (cap < sb && r) return 4;
              }
            }
          }
  std::printf("%d %d %d\n", cases > 4000, some > 500, full > 100);
  return 0;
}
"""


def test_resident_segments_fit_with_everything_else(tmp_path):
    src, exe = tmp_path / "plan.cpp", tmp_path / "plan"
    src.write_text(SRC)
    subprocess.run([os.environ.get("CXX", "g++"), "-O1", "-std=c++17", "-Wall", "-Werror",
                    "-I", os.path.join(ROOT, "dgcuda_amd", "csrc"), "-o", str(exe), str(src)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "1 1 1\n", (r.returncode, r.stdout, r.stderr)
