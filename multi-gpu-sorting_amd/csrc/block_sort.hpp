// Stable sort of up to BLOCK * IPT records by one workgroup, in registers
// and LDS (shared by the kernels whose pieces fit one workgroup).
//
// The caller gives the smallest and largest encoded key.  Their distance says
// how many low bits of a key's distance to the smallest differ at all; the
// sort takes at most three LSD passes of 9 bits over the top 27 of these (the
// window).  Among 4096 random keys one pair in a workgroup of 16 shares a
// window value, so 4-byte and 8-byte keys alike cost two or three passes; the
// write-out compares neighbours, and where a record is above its successor
// one thread puts the records that share their window value in order.  A
// group longer than kTieReach would make that slow: the workgroup then takes
// the passes over all differing bits instead.
//
// Measured in the local sort of 2^28 u64 keys (batches of 4096, two
// workgroups of 512 threads per CU): moving the records through registers
// alone 0.93 ms, with two passes 1.15 ms; two passes and the look around
// every record (the window of 18 bits leaves 1.6% of them in groups) took
// 1.75 ms.
#pragma once

#include <type_traits>
#include <utility>

#include "radix_device.hpp"

namespace mgs {

// f(0), ..., f(N - 1) with constant arguments.  (Item loops that the compiler
// only unrolls late leave the item arrays as register vectors of 16 or 32,
// which spill.)
template <typename F, int... I>
__device__ __forceinline__ void static_for_each(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_each(static_cast<F&&>(f), std::make_integer_sequence<int, N>{});
}

// Fewer records than this are put in order by one thread on each side of one
// below its predecessor.
constexpr uint32_t kTieReach = 16;
// LDS counter rows of the 9-bit digits, one per wavefront.  The row stride
// puts the two threads that scan one digit's 16 rows on different banks.
// (16-bit counters, two to a word, halve the rows but measured 4% slower:
// the unpacking costs more than the LDS they free.)
constexpr int kBlockDigitBits = 9;
constexpr int kBlockDigits = 1 << kBlockDigitBits;
template <int BLOCK>
struct BlockRows {
  static_assert(BLOCK == 512 || BLOCK == 1024, "a scan thread takes eight rows of one digit");
  static constexpr int W = BLOCK / kWave;
  static constexpr int kParts = BLOCK / kBlockDigits;  // scan threads per digit
  static constexpr int kStride = kBlockDigits + (kParts == 2 ? 4 : 0);
};

template <typename Bits, typename V, int BLOCK, int IPT>
struct BlockSortSmem {
  using VS = typename std::conditional<kHasVal<V>, V, uint32_t>::type;
  Bits keys[BLOCK * IPT];
  VS vals[kHasVal<V> ? BLOCK * IPT : 1];
  alignas(16) uint32_t off[BlockRows<BLOCK>::W * BlockRows<BLOCK>::kStride];
  uint32_t wsum[BlockRows<BLOCK>::W];
  Bits lo[BlockRows<BLOCK>::W], hi[BlockRows<BLOCK>::W];
};

// Turns the counts off[wavefront][digit] into the first position of every
// (digit, wavefront) pair, digits outermost.  Every thread of the block calls
// it; the counts are complete (a barrier precedes), the positions are
// visible to the block on return.
template <int BLOCK>
__device__ __forceinline__ void block_digit_offsets(uint32_t* off, uint32_t* wsum) {
  using R = BlockRows<BLOCK>;
  const int t = threadIdx.x, d = t / R::kParts, q = t % R::kParts, lane = t & (kWave - 1);
  const int w = (int)readfirstlane((uint32_t)(t / kWave));
  uint32_t* row = off + 8 * q * R::kStride + d;
  uint32_t c[8], s = 0;
#pragma unroll
  for (int i = 0; i < 8; ++i) c[i] = row[i * R::kStride];
#pragma unroll
  for (int i = 0; i < 8; ++i) s += c[i];
  const uint32_t incl = wave_inclusive_sum(s);
  if (lane == kWave - 1) wsum[w] = incl;
  __syncthreads();
  const uint32_t before = wave_inclusive_sum(lane < R::W ? wsum[lane] : 0u);
  uint32_t run = incl - s;
  if (w > 0) run += (uint32_t)__builtin_amdgcn_readlane((int)before, w - 1);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    row[i * R::kStride] = run;
    run += c[i];
  }
  __syncthreads();
}

// Clears this wavefront's counter row.
template <int BLOCK>
__device__ __forceinline__ void block_clear_row(uint32_t* off) {
  using R = BlockRows<BLOCK>;
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
  uint4* row = reinterpret_cast<uint4*>(off + w * R::kStride);
#pragma unroll
  for (int i = 0; i < kBlockDigits / (4 * kWave); ++i) row[i * kWave + lane] = make_uint4(0, 0, 0, 0);
}

template <typename Bits>
__device__ __forceinline__ int bit_width(Bits x) {
  if constexpr (sizeof(Bits) == 8)
    return x ? 64 - __builtin_clzll(x) : 0;
  else
    return x ? 32 - __builtin_clz(x) : 0;
}

// The value of the lane below (lane 0: its own).
template <typename Bits>
__device__ __forceinline__ Bits lane_below(Bits x) {
  uint32_t lo = (uint32_t)x;
  lo = (uint32_t)__builtin_amdgcn_update_dpp((int)lo, (int)lo, 0x138, 0xf, 0xf, false);  // wave_shr:1
  if constexpr (sizeof(Bits) == 8) {
    uint32_t hi = (uint32_t)(x >> 32);
    hi = (uint32_t)__builtin_amdgcn_update_dpp((int)hi, (int)hi, 0x138, 0xf, 0xf, false);
    return ((Bits)hi << 32) | lo;
  }
  return (Bits)lo;
}
// Smallest and largest encoded key of the block's m records (m > 0), held as
// k[i] at position wb + 64 i, i < nit.
template <int KT, typename V, int BLOCK, int IPT>
__device__ __forceinline__ void block_min_max(BlockSortSmem<typename Codec<KT>::Bits, V, BLOCK, IPT>& sm,
                                              const typename Codec<KT>::Bits (&k)[IPT], uint32_t wb, uint32_t m,
                                              uint32_t nit, typename Codec<KT>::Bits& mn,
                                              typename Codec<KT>::Bits& mx) {
  using Bits = typename Codec<KT>::Bits;
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
  Bits a = ~Bits(0), b = 0;
  static_for<IPT>([&](auto i) {
    if ((uint32_t)i < nit && wb + i * kWave < m) {
      const Bits e = Codec<KT>::enc(k[i]);
      a = e < a ? e : a;
      b = e > b ? e : b;
    }
  });
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const Bits x = __shfl_xor(a, o, kWave), y = __shfl_xor(b, o, kWave);
    a = x < a ? x : a;
    b = y > b ? y : b;
  }
  if (lane == 0) {
    sm.lo[w] = a;
    sm.hi[w] = b;
  }
  __syncthreads();
  a = sm.lo[0];
  b = sm.hi[0];
#pragma unroll
  for (int i = 1; i < BLOCK / kWave; ++i) {
    const Bits x = sm.lo[i], y = sm.hi[i];
    a = x < a ? x : a;
    b = y > b ? y : b;
  }
  mn = a;
  mx = b;
}

// Items per thread in use for m records, and the position of a thread's item
// 0: wavefront w holds the positions [64 nit w, 64 nit (w + 1)), item i of a
// lane at block_first + 64 i.
template <int BLOCK>
__device__ __forceinline__ uint32_t block_items(uint32_t m) {
  return (m + BLOCK - 1) / BLOCK;
}
template <int BLOCK>
__device__ __forceinline__ uint32_t block_first(uint32_t nit) {
  return (threadIdx.x / kWave) * nit * kWave + (threadIdx.x & (kWave - 1));
}

// Sorts the block's m records (1 <= m <= BLOCK * IPT) stably by enc(key) and
// writes them to kout[0, m) (and vout).  mn and mx bound every enc(key); mx is
// the image of a key, or all ones.
// Item slots beyond the m records hold dec(mx) on entry: padding
// behind the last record and not below any, so every pass leaves it there
// and the passes need no bounds checks.  The counter rows are clear on entry
// and on return; the caller puts a barrier between two calls.
template <int KT, typename V, int BLOCK, int IPT>
__device__ __forceinline__ void block_sort(BlockSortSmem<typename Codec<KT>::Bits, V, BLOCK, IPT>& sm,
                                           typename Codec<KT>::Bits (&k)[IPT],
                                           typename BlockSortSmem<typename Codec<KT>::Bits, V, BLOCK, IPT>::VS (&v)[IPT],
                                           uint32_t m, typename Codec<KT>::Bits mn, typename Codec<KT>::Bits mx,
                                           typename Codec<KT>::Bits* kout, V* vout) {
  using Bits = typename Codec<KT>::Bits;
  using R = BlockRows<BLOCK>;
  using VS = typename BlockSortSmem<Bits, V, BLOCK, IPT>::VS;
  constexpr bool HV = kHasVal<V>;
  constexpr uint32_t TILE = (uint32_t)BLOCK * IPT;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), w = (int)readfirstlane((uint32_t)(tid / kWave));
  m = readfirstlane(m);
  const uint32_t nit = block_items<BLOCK>(m), wb = block_first<BLOCK>(nit);
  // The window: the bits from `low` on of the distance to mn rounded down to
  // a multiple of 2^low, so that two keys share a window value exactly if
  // they agree from bit `low` on; at most three digits.
  constexpr int kWin = 3 * kBlockDigitBits;
  const int bits = bit_width<Bits>(mx - mn);
  int low = bits > kWin ? bits - kWin : 0;
  if (low > 0 && ((mx >> low) - (mn >> low)) >> kWin) ++low;
  const uint32_t wbase = (uint32_t)(mn >> low);
  const int wbits = bit_width<uint32_t>((uint32_t)(mx >> low) - wbase);
  uint32_t* const ct = sm.off + w * R::kStride;
  auto reload = [&]() {
    static_for<IPT>([&](auto i) {
      if ((uint32_t)i < nit) {
        k[i] = sm.keys[wb + i * kWave];
        if constexpr (HV) v[i] = sm.vals[wb + i * kWave];
      }
    });
  };
  // one stable pass by digit(key); the loops are apart so that every LDS
  // operation of one is issued before the first wait
  auto pass = [&](auto digit) {
    uint32_t r[IPT];
    const uint32_t d0 = digit(k[0]);
    // runs of one digit (sorted input, duplicates, padding) would put the
    // lanes on one counter in turn: such a wavefront gives the first lane's
    // digit one atomic
    if (__popcll(ballot64(d0 == readfirstlane(d0))) >= 16) {
      static_for<IPT>([&](auto i) {
        if ((uint32_t)i < nit) r[i] = rank_wave_atomic<true>(digit(k[i]), ct);
      });
    } else {
      static_for<IPT>([&](auto i) {
        if ((uint32_t)i < nit) r[i] = rank_wave_atomic<false>(digit(k[i]), ct);
      });
    }
    __syncthreads();
    block_digit_offsets<BLOCK>(sm.off, sm.wsum);
    static_for<IPT>([&](auto i) {
      if ((uint32_t)i < nit) r[i] += ct[digit(k[i])];
    });
    static_for<IPT>([&](auto i) {
      if ((uint32_t)i < nit) {
        sm.keys[r[i]] = k[i];
        if constexpr (HV) sm.vals[r[i]] = v[i];
      }
    });
    block_clear_row<BLOCK>(sm.off);
    __syncthreads();
  };
  // byte offsets from the uniform base: one address register per store
  auto store = [&](uint32_t p, Bits x) {
    *reinterpret_cast<Bits*>(reinterpret_cast<char*>(kout) + p * (uint32_t)sizeof(Bits)) = x;
  };
  auto store_val = [&](uint32_t p, VS x) {
    if constexpr (HV) *reinterpret_cast<V*>(reinterpret_cast<char*>(vout) + p * (uint32_t)sizeof(V)) = x;
  };
  if (bits == 0) {  // equal keys: in order already
    static_for<IPT>([&](auto i) {
      if ((uint32_t)i < nit && wb + i * kWave < m) {
        store(wb + i * kWave, k[i]);
        store_val(wb + i * kWave, v[i]);
      }
    });
    return;
  }
  {
    const int passes = (wbits + kBlockDigitBits - 1) / kBlockDigitBits;
    const int width = (wbits + passes - 1) / passes;  // even digits
    const uint32_t mask = (1u << width) - 1u;
    for (int shift = 0;;) {
      pass([&](Bits x) { return (((uint32_t)(Codec<KT>::enc(x) >> low) - wbase) >> shift) & mask; });
      shift += width;
      if (shift >= wbits) break;
      reload();
    }
  }
  // write-out: thread t has the records t, t + BLOCK, ..., U loads in flight
  constexpr uint32_t U = sizeof(Bits) + kValBytes<V> <= 8 ? 8 : 4;
  // (the check's result: bit j for a j-th record below its predecessor)
  static_assert(IPT <= 32, "a bit per record of a thread");
  auto write_out = [&](auto check) -> uint32_t {
    uint32_t down = 0;
#pragma unroll 1
    for (uint32_t j = 0; j < nit; j += U) {
      Bits x[U], edge[U];
      VS y[U];
      static_for<(int)U>([&](auto u) {
        const uint32_t p = min((j + u) * BLOCK + tid, TILE - 1);
        x[u] = sm.keys[p];
        if constexpr (check.value) edge[u] = sm.keys[lane == 0 ? max(p, 1u) - 1 : p];
        if constexpr (HV) y[u] = sm.vals[p];
      });
      static_for<(int)U>([&](auto u) {
        const uint32_t p = (j + u) * BLOCK + tid;
        if constexpr (check.value) {
          // the record before: the lane below's, or for the first lane the edge
          const Bits b = lane_below(x[u]);
          if (p < m && Codec<KT>::enc(lane == 0 ? edge[u] : b) > Codec<KT>::enc(x[u])) down |= 1u << (j + u);
        }
        if (p < m) {
          store(p, x[u]);
          store_val(p, y[u]);
        }
      });
    }
    return down;
  };
  if (low == 0) {
    write_out(std::integral_constant<bool, false>{});
    return;
  }
  uint32_t down = write_out(std::integral_constant<bool, true>{});
  // (the stores below may follow another thread's to the same place)
  auto stored = [] { __builtin_amdgcn_s_waitcnt(0); };
  stored();
  if (!__syncthreads_or(down != 0 ? 1 : 0)) return;
  // A group that reaches kTieReach from a record below its predecessor is left to
  // the passes over all bits.  Every such record is asked before any group
  // is mended: keys that crowd in the window (log-uniform ones: half of them)
  // have many, and walking through their groups first took longer than the
  // passes: 2000 u64 keys 75 us, now 21.
  const Bits lim = Bits(1) << low;
  auto image = [&](uint32_t p) { return Codec<KT>::enc(sm.keys[p]); };
  bool longer = false;
  for (uint32_t rest = down; rest != 0; rest &= rest - 1) {
    const uint32_t p = (uint32_t)__builtin_ctz(rest) * BLOCK + tid;
    const Bits e = image(p);
    longer |= p + kTieReach < m && (image(p + kTieReach) ^ e) < lim;
    longer |= p > kTieReach && (image(p - 1 - kTieReach) ^ e) < lim;
  }
  if (!__syncthreads_or(longer ? 1 : 0)) {
    // the thread that sees the first record of a group below its predecessor
    // writes the whole group in order
    while (down != 0) {
      const uint32_t p = (uint32_t)__builtin_ctz(down) * BLOCK + tid;
      down &= down - 1;
      uint32_t l = p - 1, r = p;
      Bits e = image(l);
      bool first = true;
      while (l > 0 && first) {
        const Bits x = image(l - 1);
        if ((x ^ e) >= lim) break;
        first = x <= e;
        e = x;
        --l;
      }
      if (!first) continue;
      while (r + 1 < m && (image(r + 1) ^ e) < lim) ++r;
      for (uint32_t q = l; q <= r; ++q) {
        const Bits raw = sm.keys[q], x = Codec<KT>::enc(raw);
        uint32_t to = l;
        for (uint32_t t = l; t <= r; ++t) {
          const Bits y = image(t);
          to += (y < x || (y == x && t < q)) ? 1u : 0u;
        }
        store(to, raw);
        if constexpr (HV) store_val(to, sm.vals[q]);
      }
    }
    return;
  }
  // all differing bits, from the present order
  for (int shift = 0; shift < bits; shift += kBlockDigitBits) {
    reload();
    pass([&](Bits x) { return (uint32_t)((Codec<KT>::enc(x) - mn) >> shift) & ((1u << kBlockDigitBits) - 1u); });
  }
  write_out(std::integral_constant<bool, false>{});
}

}  // namespace mgs
