// dg_workspace.h -- device buffers that are kept between adjoint solves.
//
// A solve's work buffers are gigabytes that live for milliseconds: allocating
// and freeing 1 GB took 1 to 28 ms beside 8 ms of gradient (Euler p = 4, 131,072
// triangles, 8 steps) and 5.6 GB 1.7 to 100 ms beside 25 (TE p = 3, 199,712
// triangles, 32 steps), by the machine.  So a solve's buffers stay for the next
// solve on the device, but only where they are in nobody's way:
//   bounded     all idle buffers of a device together hold at most `limit`
//               bytes; the oldest go first, and larger ones are never kept
//   given back  with their handle or its mesh, on request, and whenever an
//               allocation of the library fails on that device, whichever
//               handle or ensemble makes it (reclaim, then the allocation again)
//   safe        only idle buffers are here, whose last solve has been waited
//               for: a solve takes one out and is its one owner until it gives
//               it back.  Any thread may call; the memory itself is freed
//               outside the lock.
// Host code without HIP: FREE is what frees a buffer.
#pragma once

#include <cstddef>
#include <mutex>
#include <vector>

namespace dgk {

template <void (*FREE)(void *)>
class KeptBuffers {
  struct Kept {
    const void *owner;
    int device;
    void *p;
    size_t bytes;
  };
  std::mutex m;
  std::vector<Kept> v;  // oldest first

  // frees every kept buffer that `goes` names
  template <class F>
  bool release(const F &goes) {
    std::vector<void *> out;
    {
      std::lock_guard<std::mutex> l(m);
      out.reserve(v.size());
      size_t n = 0;
      for (const Kept &k : v) {
        if (goes(k))
          out.push_back(k.p);
        else
          v[n++] = k;
      }
      v.erase(v.begin() + (ptrdiff_t)n, v.end());
    }
    for (void *p : out) FREE(p);
    return !out.empty();
  }

 public:
  // a buffer of the device with room for `need`, out of here (nullptr: none);
  // *bytes its size.  The owner's own, or the smallest of the others': handles
  // that solve in turn share one.
  void *take(const void *owner, int device, size_t need, size_t *bytes) {
    std::lock_guard<std::mutex> l(m);
    size_t best = v.size();
    for (size_t i = 0; i < v.size(); i++) {
      if (v[i].device != device || v[i].bytes < need) continue;
      if (v[i].owner == owner) {
        best = i;
        break;
      }
      if (best == v.size() || v[i].bytes < v[best].bytes) best = i;
    }
    *bytes = 0;
    if (best == v.size()) return nullptr;
    void *p = v[best].p;
    *bytes = v[best].bytes;
    v.erase(v.begin() + (ptrdiff_t)best);
    return p;
  }
  // a buffer that the owner is done with (std::bad_alloc: nothing done)
  void give(const void *owner, int device, void *p, size_t bytes, size_t limit) {
    if (bytes > limit) {
      FREE(p);
      return;
    }
    std::vector<void *> out;
    {
      std::lock_guard<std::mutex> l(m);
      v.reserve(v.size() + 1);
      out.reserve(v.size());
      size_t sum = bytes;
      for (const Kept &k : v)
        if (k.device == device) sum += k.bytes;
      for (size_t i = 0; sum > limit;) {
        if (v[i].device != device) {
          i++;
          continue;
        }
        sum -= v[i].bytes;
        out.push_back(v[i].p);
        v.erase(v.begin() + (ptrdiff_t)i);
      }
      v.push_back({owner, device, p, bytes});
    }
    for (void *q : out) FREE(q);
  }
  // bytes of the device in idle buffers
  size_t idle(int device) {
    std::lock_guard<std::mutex> l(m);
    size_t sum = 0;
    for (const Kept &k : v)
      if (k.device == device) sum += k.bytes;
    return sum;
  }
  void drop(const void *owner) {
    release([&](const Kept &k) { return k.owner == owner; });
  }
  // every idle buffer of the device; whether there was one
  bool reclaim(int device) {
    return release([&](const Kept &k) { return k.device == device; });
  }
};

}  // namespace dgk
