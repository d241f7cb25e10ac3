// Look-back and counting routines shared by the radix sort's kernels.
#pragma once

#include <type_traits>

#include "radix_sort.hpp"

namespace mgs {

#ifndef MGS_LB_SPIN_LIMIT
#define MGS_LB_SPIN_LIMIT (1u << 20)
#endif
constexpr uint32_t kLookbackSpinLimit = MGS_LB_SPIN_LIMIT;

// Predecessor descriptors read per look-back round trip of the pass kernels
// (the window registers stay live across the digit scan and the scatter).
#ifndef MGS_PASS_LB_WINDOW
#define MGS_PASS_LB_WINDOW 2
#endif

constexpr int kPassWindow = MGS_PASS_LB_WINDOW;

// Issues the loads of the descriptors of predecessor tiles t, t-1, ...,
// t-NW+1 (those >= 0) for digit d of a chain whose first tile's
// descriptors start at `desc`.
template <typename D, int NW>
__device__ __forceinline__ void lookback_load(const D* desc, int64_t t, uint32_t d, D (&v)[NW]) {
#pragma unroll
  for (int j = 0; j < NW; ++j) v[j] = (t - j >= 0) ? ld_agent(desc + (size_t)(t - j) * kRadix + d) : D(0);
}

// Look-back for one digit starting from a window already loaded at
// predecessor t: sums aggregates, walking back, until an inclusive prefix is
// found (or the chain's first tile is passed).  Issuing the first window
// before the tile publishes its own aggregate keeps that store's completion
// off the critical path.
// Sums the leading published descriptors of a window loaded at predecessor
// t into `prefix`; returns how many were consumed and sets `done` when an
// inclusive prefix ended the walk.
template <typename D, int NW>
__device__ __forceinline__ int lookback_consume(int64_t t, int parity, const D (&v)[NW], uint32_t& prefix,
                                                bool& done) {
  int consumed = 0;
  done = false;
#pragma unroll
  for (int j = 0; j < NW; ++j) {
    if (done || consumed != j || t - j < 0) continue;
    const uint32_t st = Desc<D>::status(v[j], parity);
    if (st == kStEmpty) continue;
    prefix += (uint32_t)Desc<D>::value(v[j]);
    consumed = j + 1;
    if (st == kStInclusive) done = true;
  }
  return consumed;
}

// One look-back round that does not wait for the next one: consumes the
// window loaded at predecessor t and, unless the walk is over, moves t back
// and issues the loads of the next window.  Returns true when the prefix is
// complete.
template <typename D, int NW>
__device__ __forceinline__ bool lookback_step(const D* desc, int64_t& t, uint32_t d, int parity, D (&v)[NW],
                                              uint32_t& prefix) {
  bool done;
  const int consumed = lookback_consume(t, parity, v, prefix, done);
  if (done || t - consumed < 0) return true;
  t -= consumed;
  lookback_load(desc, t, d, v);
  return false;
}

template <typename D, int NW>
__device__ __forceinline__ uint32_t lookback_from(const D* desc, int64_t t, uint32_t d, int parity,
                                                  D (&v)[NW], uint32_t prefix, uint32_t spin_limit, bool& gave_up) {
  uint32_t spins = 0;
  gave_up = false;
  for (;;) {
    bool done;
    const int consumed = lookback_consume(t, parity, v, prefix, done);
    if (done || t - consumed < 0) break;
    if (consumed == 0) {
      // Bounded wait: a predecessor tile always publishes within microseconds.
      // The bound keeps a corrupted descriptor array (or a chain no
      // workgroup serves) from hanging the GPU; the caller records it in the
      // status word, since the prefix is then incomplete (every store stays
      // in bounds).
      if (++spins > spin_limit) {
        gave_up = true;
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
    t -= consumed;
    lookback_load(desc, t, d, v);
  }
  return prefix;
}

}  // namespace mgs
