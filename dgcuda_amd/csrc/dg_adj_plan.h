// dg_adj_plan.h -- device memory of one checkpointed adjoint solve (host code
// without HIP).
#pragma once

#include <algorithm>
#include <cstddef>

namespace dgk {

// a buffer's share of an allocation: 256-byte multiples, 8 KiB apart
inline size_t adj_stride(size_t bytes) { return (bytes + 255) / 256 * 256 + 8192; }

// nsteps steps of S stages in segments of `every` steps, of which the last
// `nres` ("resident") keep the stage data of the forward pass itself.
// Segments 0 .. nrec - 1 are recomputed from checkpoints.  The last one never
// is: the sweep starts there, so its forward pass leaves its stage data in the
// recompute's buffers, unless it is resident anyway.
struct AdjPlan {
  int nsteps, every, S;
  size_t sb;     // bytes of a state
  size_t kst_b;  // of a stage's E rows of k (0: no permittivity gradient)
  size_t eps_b;  // of the permittivity gradient's own arrays, strides included

  int nseg() const { return (nsteps + every - 1) / every; }
  int len(int q) const { return std::min(every, nsteps - q * every); }
  int nrec(int nres) const { return nres ? nseg() - nres : nseg() - 1; }
  // stage inputs of one segment and its final state, and the E rows
  size_t seg_bytes(int ns) const { return ((size_t)ns * S + 1) * sb + (size_t)ns * S * kst_b; }
  size_t seg_strides(int ns) const {
    return ((size_t)ns * S + 1) * adj_stride(sb) + (kst_b ? (size_t)ns * S * adj_stride(kst_b) : 0);
  }
  // the solve's one allocation: work arrays, checkpoints, recompute buffers
  size_t need(int nres) const {
    return adj_stride(sb) * (size_t)(S + 2 + nrec(nres)) +
           (nres < nseg() ? seg_strides(every) : 0) + eps_b;
  }

  // The resident segments that a setting of `cap` bytes and `avail` bytes of
  // memory hold.  The setting counts the stage data, checkpoints and recompute
  // buffers (segment 0 is recomputed unless every segment is resident; a
  // resident segment saves its checkpoint); the memory has to hold every
  // allocation of the solve.
  int resident(double cap, size_t avail) const {
    const int n = nseg();
    size_t all = 0;
    for (int q = 0; q < n; q++) all += seg_strides(len(q));
    size_t raw = 0;
    for (int q = 0; q < n; q++) raw += seg_bytes(len(q));
    if ((double)raw <= cap && need(n) + all <= avail) return n;
    size_t used = seg_bytes(every) + (size_t)n * sb, held = 0;
    int r = 0;
    for (int q = n - 1; q > 0; q--) {
      used += seg_bytes(len(q)) - sb;
      held += seg_strides(len(q));
      if ((double)used > cap || need(r + 1) + held > avail) break;
      r++;
    }
    return r;
  }
};

}  // namespace dgk
