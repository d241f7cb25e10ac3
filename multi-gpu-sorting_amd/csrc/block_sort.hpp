// Stable sort of up to BLOCK * IPT records by one workgroup, in registers
// and LDS (shared by the kernels whose pieces fit one workgroup).
//
// The caller gives the smallest and largest encoded key.  Their distance says
// how many low bits of enc(key) - smallest differ at all; the sort takes at
// most two LSD passes of 9 bits over the top 18 of these (the window), and
// the write-out puts the few records that share a window value in order by
// comparing neighbours.  Two passes leave random keys in groups of one or two
// (8192 keys, 262144 window values), so 4-byte and 8-byte keys alike cost two
// passes whatever their width.  A group longer than kTieReach records that
// are not all equal would make the comparisons quadratic: the workgroup then
// takes the passes over all differing bits instead.
#pragma once

#include <type_traits>

#include "radix_device.hpp"

namespace mgs {

// Records a thread looks at on each side of its own in the write-out.
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

// The value of the lane below (lane 0: its own) and above (lane 63: its own).
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
template <typename Bits>
__device__ __forceinline__ Bits lane_above(Bits x) {
  uint32_t lo = (uint32_t)x;
  lo = (uint32_t)__builtin_amdgcn_update_dpp((int)lo, (int)lo, 0x130, 0xf, 0xf, false);  // wave_shl:1
  if constexpr (sizeof(Bits) == 8) {
    uint32_t hi = (uint32_t)(x >> 32);
    hi = (uint32_t)__builtin_amdgcn_update_dpp((int)hi, (int)hi, 0x130, 0xf, 0xf, false);
    return ((Bits)hi << 32) | lo;
  }
  return (Bits)lo;
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
// writes them to kout[0, m) (and vout).  mn and mx bound every enc(key).
// Item slots beyond the m records hold the key dec(mx) on entry: padding
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
  constexpr bool HV = kHasVal<V>;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), w = (int)readfirstlane((uint32_t)(tid / kWave));
  m = readfirstlane(m);
  const uint32_t nit = block_items<BLOCK>(m), wb = block_first<BLOCK>(nit);
  const int bits = bit_width<Bits>(mx - mn);
  uint32_t* const ct = sm.off + w * R::kStride;
  auto reload = [&]() {
#pragma unroll
    for (int i = 0; i < IPT; ++i)
      if ((uint32_t)i < nit) {
        k[i] = sm.keys[wb + i * kWave];
        if constexpr (HV) v[i] = sm.vals[wb + i * kWave];
      }
  };
  // one stable pass over `width` bits; the loops are apart so that every LDS
  // operation of one is issued before the first wait
  auto pass = [&](int shift, int width) {
    const uint32_t mask = (1u << width) - 1u;
    auto digit = [&](Bits x) { return (uint32_t)((Codec<KT>::enc(x) - mn) >> shift) & mask; };
    uint32_t r[IPT];
    const uint32_t d0 = digit(k[0]);
    // runs of one digit (sorted input, duplicates, padding) would put the
    // lanes on one counter in turn: such a wavefront gives the first lane's
    // digit one atomic
    if (__popcll(ballot64(d0 == readfirstlane(d0))) >= 16) {
#pragma unroll
      for (int i = 0; i < IPT; ++i)
        if ((uint32_t)i < nit) r[i] = rank_wave_atomic<true>(digit(k[i]), ct);
    } else {
#pragma unroll
      for (int i = 0; i < IPT; ++i)
        if ((uint32_t)i < nit) r[i] = rank_wave_atomic<false>(digit(k[i]), ct);
    }
    __syncthreads();
    block_digit_offsets<BLOCK>(sm.off, sm.wsum);
#pragma unroll
    for (int i = 0; i < IPT; ++i)
      if ((uint32_t)i < nit) r[i] += ct[digit(k[i])];
#pragma unroll
    for (int i = 0; i < IPT; ++i)
      if ((uint32_t)i < nit) {
        sm.keys[r[i]] = k[i];
        if constexpr (HV) sm.vals[r[i]] = v[i];
      }
    block_clear_row<BLOCK>(sm.off);
    __syncthreads();
  };
  const int low = bits > 2 * kBlockDigitBits ? bits - 2 * kBlockDigitBits : 0;
  if (bits == 0) {  // equal keys: in order already
#pragma unroll
    for (int i = 0; i < IPT; ++i)
      if ((uint32_t)i < nit) {
        sm.keys[wb + i * kWave] = k[i];
        if constexpr (HV) sm.vals[wb + i * kWave] = v[i];
      }
    __syncthreads();
  } else {
    const int first = min(bits - low, kBlockDigitBits);
    pass(low, first);
    if (low + first < bits) {
      reload();
      pass(low + first, bits - low - first);
    }
  }
  // write-out: thread t has the records t, t + BLOCK, ...; with bits below
  // the window a record moves left past the larger records of its group
  // before it, right past the smaller ones after it
#pragma unroll
  for (int j = 0; j < IPT; ++j)
    if ((uint32_t)j < nit) k[j] = sm.keys[j * BLOCK + tid];
  if (low > 0) {
    bool slow = false;
    uint32_t np[IPT];
    auto image = [&](uint32_t p) { return Codec<KT>::enc(sm.keys[p]) - mn; };
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
      const uint32_t p = (uint32_t)(j * BLOCK + tid);
      np[j] = p;
      if ((uint32_t)j < nit) {
        const Bits e = Codec<KT>::enc(k[j]) - mn;
        Bits el = lane_below(e), er = lane_above(e);
        if (lane == 0) el = p > 0 ? image(p - 1) : ~e;
        if (lane == kWave - 1) er = p + 1 < m ? image(p + 1) : ~e;
        const bool sl = ((e ^ el) >> low) == 0, sr = ((e ^ er) >> low) == 0;
        const uint64_t left = ballot64(sl), right = ballot64(sr);
        if ((left | right) != 0) {
          // a group of two inside the wavefront needs no further look
          const bool head = sr && !sl && lane < kWave - 1 && ((right >> 1 >> lane) & 1u) == 0;
          const bool tail = sl && !sr && lane > 0 && ((left << 1 >> lane) & 1u) == 0;
          if (head) np[j] = p + (er < e ? 1u : 0u);
          if (tail) np[j] = p - (el > e ? 1u : 0u);
          // a larger group needs a look if it reaches across the wavefront's
          // ends or has a record above its successor
          bool look = (sl || sr) && !head && !tail && p < m;
          if (ballot64(look) != 0) {
            const uint64_t down = ballot64(sl && el > e);
            const uint64_t upto = ~left & ((2ull << lane) - 1u), after = ~left >> 1 >> lane;
            const int a = 63 - (int)__builtin_clzll(upto | 1u);           // the group's first lane
            const int b = after ? lane + (int)__builtin_ctzll(after) : 63;  // and its last
            look = look && (upto == 0 || (after == 0 && right >> 63) || (down & ((2ull << b) - 1u) & ~((2ull << a) - 1u)) != 0);
          }
          if (look) {
            bool differ = false, longer = false;
            uint32_t at = p;
            for (uint32_t r = 1; r <= p; ++r) {
              const Bits x = image(p - r);
              if (((x ^ e) >> low) != 0) break;
              if (r > kTieReach) {
                longer = true;
                break;
              }
              differ |= x != e;
              at -= x > e ? 1u : 0u;
            }
            for (uint32_t r = 1; p + r < m; ++r) {
              const Bits x = image(p + r);
              if (((x ^ e) >> low) != 0) break;
              if (r > kTieReach) {
                longer = true;
                break;
              }
              differ |= x != e;
              at += x < e ? 1u : 0u;
            }
            // a group that reaches further is in order if its records are
            // all equal; otherwise the first different one on either side
            // sees both the difference and the long run before it
            slow |= differ && longer;
            np[j] = at;
          }
        }
      }
    }
    if (!__syncthreads_or(slow ? 1 : 0)) {
#pragma unroll
      for (int j = 0; j < IPT; ++j)
        if ((uint32_t)j < nit && (uint32_t)(j * BLOCK + tid) < m) {
          kout[np[j]] = k[j];
          if constexpr (HV) vout[np[j]] = sm.vals[j * BLOCK + tid];
        }
      return;
    }
    for (int shift = 0; shift < bits; shift += kBlockDigitBits) {
      reload();
      pass(shift, min(bits - shift, kBlockDigitBits));
    }
#pragma unroll
    for (int j = 0; j < IPT; ++j)
      if ((uint32_t)j < nit) k[j] = sm.keys[j * BLOCK + tid];
  }
  if constexpr (HV) {
#pragma unroll
    for (int j = 0; j < IPT; ++j)
      if ((uint32_t)j < nit) v[j] = sm.vals[j * BLOCK + tid];
  }
#pragma unroll
  for (int j = 0; j < IPT; ++j)
    if ((uint32_t)j < nit && (uint32_t)(j * BLOCK + tid) < m) {
      kout[j * BLOCK + tid] = k[j];
      if constexpr (HV) vout[j * BLOCK + tid] = v[j];
    }
}

}  // namespace mgs
