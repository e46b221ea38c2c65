"""The buffers that handles keep between adjoint solves (dg_workspace.h), with
a stand-in for device memory: the bound and what goes first, what gives them
back, and that threads that solve while others reclaim never meet in one
buffer or free one twice."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include "dg_workspace.h"
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <thread>
struct Buf { std::atomic<int> state{0}; };  // 0 idle, 1 in use, 2 freed
static std::atomic<int> live{0};
static void buf_free(void *p) {
  int idle = 0;
  if (!((Buf *)p)->state.compare_exchange_strong(idle, 2)) { std::puts("freed in use or twice"); std::abort(); }
  live--;  // (leaked, so that a second free is seen)
}
static Buf *fresh() { live++; return new Buf; }
static dgk::KeptBuffers<buf_free> K;
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
int main() {
  int h[4];
  size_t n = 9;
  CHECK(!K.take(&h[0], 0, 1, &n) && n == 0);
  Buf *a = fresh(), *b = fresh(), *c = fresh(), *d = fresh();
  K.give(&h[0], 0, a, 40, 100);
  K.give(&h[1], 0, b, 50, 100);
  K.give(&h[2], 1, c, 100, 100);          // another device: its own bound
  CHECK(live == 4 && K.idle(0) == 90 && K.idle(1) == 100 && K.idle(2) == 0);
  K.give(&h[3], 0, d, 60, 100);           // 150: the oldest goes, then the next
  CHECK(a->state == 2 && b->state == 2 && c->state == 0 && live == 2);
  CHECK(K.take(&h[3], 0, 61, &n) == nullptr && K.take(&h[3], 2, 1, &n) == nullptr);
  CHECK(K.take(&h[3], 0, 60, &n) == d && n == 60);
  K.give(&h[3], 0, d, 101, 100);          // larger than the bound: not kept
  CHECK(d->state == 2 && K.take(&h[3], 0, 1, &n) == nullptr && live == 1);
  CHECK(K.idle(0) == 0 && !K.reclaim(0) && K.reclaim(1) && c->state == 2 && !K.reclaim(1) && live == 0);
  a = fresh(); b = fresh();
  K.give(&h[0], 0, a, 10, 100);
  K.give(&h[1], 0, b, 10, 100);
  K.drop(&h[0]);
  CHECK(a->state == 2 && b->state == 0 && K.take(&h[1], 0, 10, &n) == b);
  K.give(&h[1], 0, b, 10, 100);
  K.drop(&h[1]);
  CHECK(live == 0);
  // another handle's: its own first, else the smallest with room, now its own
  a = fresh(); b = fresh(); c = fresh();
  K.give(&h[0], 0, a, 30, 100);
  K.give(&h[1], 0, b, 20, 100);
  K.give(&h[2], 0, c, 10, 100);
  CHECK(K.take(&h[0], 0, 5, &n) == a && n == 30);
  CHECK(K.take(&h[3], 0, 11, &n) == b && n == 20);
  K.give(&h[3], 0, b, 20, 100);
  K.drop(&h[1]);
  CHECK(b->state == 0);
  K.drop(&h[3]);
  CHECK(b->state == 2 && K.take(&h[3], 0, 10, &n) == c);
  buf_free(a);
  buf_free(c);
  CHECK(live == 0);
  // eight owners on two devices, each its own thread
  std::vector<std::thread> t;
  static char own[8];
  for (int i = 0; i < 8; i++)
    t.emplace_back([i] {
      unsigned r = 12345u + i;
      for (int q = 0; q < 20000; q++) {
        r = r * 1664525u + 1013904223u;
        const int dev = i & 1;
        if ((r >> 24) < 16) K.reclaim(dev);
        if ((r >> 24) > 250) K.drop(&own[i]);
        size_t have, need = 1 + (r >> 8) % 60;
        Buf *p = (Buf *)K.take(&own[i], dev, need, &have);
        if (p && have < need) { std::puts("too small"); std::abort(); }
        if (!p) { p = fresh(); have = need; }
        int idle = 0;
        if (!p->state.compare_exchange_strong(idle, 1)) { std::puts("two owners"); std::abort(); }
        p->state = 0;
        K.give(&own[i], dev, p, have, 100);
      }
    });
  for (auto &x : t) x.join();
  K.reclaim(0);
  K.reclaim(1);
  CHECK(live == 0);
  std::puts("ok");
  return 0;
}
"""


def test_kept_buffers(tmp_path):
    src, exe = tmp_path / "kept.cpp", tmp_path / "kept"
    src.write_text(SRC)
    subprocess.run([os.environ.get("CXX", "g++"), "-O1", "-std=c++17", "-pthread", "-Wall", "-Werror",
                    "-I", os.path.join(ROOT, "dgcuda_amd", "csrc"), "-o", str(exe), str(src)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
