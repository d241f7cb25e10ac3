// Scatter pass of the three-pass paths (msd_sort.hip, msd_wide.hip).
#pragma once

#include <type_traits>

#include "msd_sort.hpp"
#include "radix_device.hpp"

namespace mgs {

// The window values' counts of bucket b, summed over the ranges' slices into
// cnt[256], by a block of 256 threads: 32 threads take a slice's row of 256
// 16-bit counters (16 bytes each), eight groups of them every eighth slice,
// with up to 16 loads in flight.  Bound by latency: a row of 512 bytes per
// slice and workgroup, one workgroup per CU.  (A thread per window value with
// 4 loads in flight: the scan 23 us at 256 slices; with 8, 19; so 11 to 13.)
__device__ __forceinline__ void sum_slices(const uint32_t* __restrict__ slices, uint32_t ranges, uint32_t b,
                                           uint32_t* cnt) {
  const uint32_t d = threadIdx.x, col = d & 31, part = d >> 5;
  cnt[d] = 0;
  const uint4* const row = reinterpret_cast<const uint4*>(slices + (size_t)b * (kRadix / 2)) + col;
  uint32_t lo[4] = {}, hi[4] = {};
  auto add = [&](const uint4& x) {
    const uint32_t v[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      lo[i] += v[i] & 0xFFFFu;
      hi[i] += v[i] >> 16;
    }
  };
  constexpr uint32_t U = 16;
  uint32_t c = part;
  for (; c + 8 * (U - 1) < ranges; c += 8 * U) {
    uint4 x[U];
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) x[u] = row[(size_t)(c + 8 * u) * (kMsdBins / 8)];
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) add(x[u]);
  }
  for (; c < ranges; c += 8) add(row[(size_t)c * (kMsdBins / 8)]);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    atomicAdd(&cnt[8 * col + 2 * i], lo[i]);
    atomicAdd(&cnt[8 * col + 2 * i + 1], hi[i]);
  }
  __syncthreads();
}


constexpr uint32_t kNoWork = 0xFFFFFFFFu;

// The eight bits of the encoded key from `shift` on (any shift).
template <int KT>
__device__ __forceinline__ uint32_t digit_at(typename Codec<KT>::Bits raw, int shift) {
  if constexpr (sizeof(raw) == 8)
    return (uint32_t)(Codec<KT>::enc(raw) >> shift) & 0xFFu;
  else
    return digit_of<KT>(raw, shift);
}

// ---------------------------------------------------------------------------
// passes 1 and 2: onesweep passes over chains of tiles with decoupled
// look-back inside each chain (the look-back of the LSD pass kernel).
//   pass 1  8 chains: equal ranges of the input; the digit bases of chain C
//           are the byte-3 bucket starts plus the keys of that digit in
//           the ranges before it (the upfront's per-range histograms)
//   pass 2  256 chains: the byte-3 buckets; digit bases = sub-bucket starts
// Chain c is served by the workgroups of XCD c mod 8 (when the upfront ran
// on all eight XCDs), which start together on their XCD's first chain and
// move on together, so at any time the 32 workgroups of an XCD work on
// consecutive tiles of one chain: every digit run of the chain's output is
// then written by consecutive tiles at about the same time.
// ---------------------------------------------------------------------------
template <typename Bits, typename V>
struct MsdPassArgs {
  const Bits* src;
  Bits* dst;
  const V* vsrc;
  V* vdst;
  uint32_t n;
  uint32_t chains;             // 8 (pass 1) or 256 (pass 2)
  const uint32_t* bucket_start;
  const uint32_t* chain_pref;  // pass 1: prefix over the upfront's ranges per digit
  uint32_t ranges_per_chain;   // pass 1: upfront ranges per chain
  uint32_t chain_keys;         // pass 1: keys per chain
  const uint32_t* sub_off;     // pass 2: sub-bucket offsets inside each bucket
  const uint32_t* tile_base;   // first descriptor tile of each chain
  uint32_t* counters;          // tiles taken per chain
  uint32_t* desc;              // look-back descriptors, 256 per tile
  int parity;                  // descriptor status rotation of this pass
  const MsdCtl* ctl;
  uint32_t* status;
  uint32_t spin_limit;
  // pass 2 of the wider records' path also writes the local sort's batch
  // table (batches NULL: not): entry batch_base[b] + k is batch k of bucket b,
  // {first record, records, first window value, last window value}
  const uint32_t* leaders;
  const uint32_t* batch_cnt;
  const uint32_t* batch_base;
  uint4* batches;
};

__device__ __forceinline__ void msd_publish(uint32_t* p, uint32_t v, bool xcd_local) {
  if (xcd_local)
    st_wg(p, v);
  else
    st_agent(p, v);
}

template <int KT, typename V, int PASS, int BLOCK, int IPT, int WAVES>
__global__ __launch_bounds__(BLOCK, WAVES) void msd_pass_kernel(MsdPassArgs<typename Codec<KT>::Bits, V> a) {
  using Bits = typename Codec<KT>::Bits;
  constexpr int W = BLOCK / kWave;
  constexpr int TILE = BLOCK * IPT;
  constexpr bool HV = kHasVal<V>;
  using VS = typename std::conditional<HV, V, uint32_t>::type;
  using D = uint32_t;
  if (a.ctl->off) return;
  const bool runs = a.ctl->runs != 0;
  const int shift = (int)a.ctl->low + (PASS == 1 ? 8 : 0);  // the window's high or low byte

  __shared__ Bits keys[TILE];
  __shared__ VS vstage[HV ? TILE : 1];
  __shared__ uint32_t off[W][kRadix];
  __shared__ uint32_t gbase[kRadix];
  __shared__ uint32_t s_prefix[kRadix];
  __shared__ uint32_t sums[4];
  __shared__ uint32_t s_tile;

  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int w = tid / kWave;
  const bool lb_wave = tid >= kRadix && tid < 2 * kRadix;
  const int taker = kRadix;
  for (int i = tid; i < W * kRadix; i += BLOCK) (&off[0][0])[i] = 0;

  auto chain_lo = [&](uint32_t c) -> uint32_t {
    if constexpr (PASS == 1) return c * a.chain_keys;
    else return a.bucket_start[c];
  };
  auto chain_hi = [&](uint32_t c) -> uint32_t {
    if constexpr (PASS == 1) return (uint32_t)std::min<size_t>((size_t)(c + 1) * a.chain_keys, a.n);
    else return a.bucket_start[c + 1];
  };
  // thread d < 256: output position of the chain's first key of digit d
  auto digit_base = [&](uint32_t c, uint32_t d) -> uint32_t {
    if constexpr (PASS == 1) return a.bucket_start[d] + a.chain_pref[(size_t)c * a.ranges_per_chain * kRadix + d];
    else return a.bucket_start[c] + a.sub_off[c * kRadix + d];
  };

  const bool xcd_local = a.chains % kXcds == 0 && a.ctl->xcd_mask == (1u << kXcds) - 1;
  uint32_t my_chain = blockIdx.x % a.chains, chains_left = a.chains, chain_step = 1;
  if (xcd_local) {
    my_chain = xcc_id();
    chains_left = a.chains / kXcds;
    chain_step = kXcds;
  }
  // next tile: (chain, tile inside the chain) packed as chain << 20 | tile
  auto take = [&]() -> uint32_t {
    while (chains_left > 0) {
      const uint32_t t = atomicAdd(&a.counters[my_chain], 1u);
      const uint32_t lo = chain_lo(my_chain), hi = chain_hi(my_chain);
      if (t < (hi - lo + TILE - 1) / TILE) return (my_chain << 20) | t;
      my_chain += chain_step;
      if (my_chain >= a.chains) my_chain -= a.chains;
      --chains_left;
    }
    return kNoWork;
  };

  if (tid == taker) s_tile = take();
  if constexpr (PASS == 2) {
    if (a.batches != nullptr && tid < kRadix) {
      for (uint32_t b = blockIdx.x; b < (uint32_t)kRadix; b += gridDim.x) {
        const uint32_t k = tid, cnt = a.batch_cnt[b];
        if (k < cnt) {
          const uint32_t s0 = a.leaders[b * kRadix + k];
          const uint32_t s1 = k + 1 < cnt ? a.leaders[b * kRadix + k + 1] : (uint32_t)kRadix;
          const uint32_t beg = a.bucket_start[b] + a.sub_off[b * kRadix + s0];
          const uint32_t end = s1 < (uint32_t)kRadix ? a.bucket_start[b] + a.sub_off[b * kRadix + s1] : a.bucket_start[b + 1];
          a.batches[a.batch_base[b] + k] = make_uint4(beg, end - beg, b * kRadix + s0, b * kRadix + s1 - 1);
        }
      }
    }
  }
  __syncthreads();
  uint32_t cur = s_tile;
  uint32_t cur_chain = 0xFFFFFFFFu, cur_base = 0, clo = 0, chi = 0;
  Bits kc[IPT];
  VS vc[IPT];
  auto load = [&](uint32_t lo, uint32_t hi, uint32_t t) {
    const uint32_t tb = lo + t * (uint32_t)TILE;
    const uint32_t wb = tb + (uint32_t)(w * IPT * kWave + lane);
    if (hi - tb >= (uint32_t)TILE) {
#pragma unroll
      for (int i = 0; i < IPT; ++i) kc[i] = a.src[wb + i * kWave];
      if constexpr (HV) {
#pragma unroll
        for (int i = 0; i < IPT; ++i) vc[i] = a.vsrc[wb + i * kWave];
      }
    } else {
#pragma unroll
      for (int i = 0; i < IPT; ++i) {
        const uint32_t idx = wb + i * kWave;
        kc[i] = idx < hi ? a.src[idx] : Bits(0);
        if constexpr (HV) vc[i] = idx < hi ? a.vsrc[idx] : VS(0);
      }
    }
  };
  if (cur != kNoWork) load(chain_lo(cur >> 20), chain_hi(cur >> 20), cur & 0xFFFFFu);

  while (cur != kNoWork) {
    const uint32_t chain = cur >> 20, lt = cur & 0xFFFFFu;
    if (chain != cur_chain) {
      clo = chain_lo(chain);
      chi = chain_hi(chain);
    }
    const uint32_t tb = clo + lt * (uint32_t)TILE;
    const uint32_t tile_cnt = min((uint32_t)TILE, chi - tb);
    const bool full = tile_cnt == (uint32_t)TILE;
    const uint32_t wb = tb + (uint32_t)(w * IPT * kWave + lane);
    uint32_t pk[IPT];
    uint32_t* ct = off[w];
    if (full) {
      uint32_t dg[IPT];
#pragma unroll
      for (int i = 0; i < IPT; ++i) dg[i] = digit_at<KT>(kc[i], shift);
      if (runs)
        rank_items_full<IPT, true>(dg, ct, pk);
      else
        rank_items_full<IPT, false>(dg, ct, pk);
    } else {
#pragma unroll
      for (int i = 0; i < IPT; ++i) {
        const uint32_t d = digit_at<KT>(kc[i], shift);
        pk[i] = (wb + i * kWave < chi) ? ((d << 16) | rank_wave_atomic<false>(d, ct)) : 0u;
      }
    }
#pragma unroll
    for (int i = 0; i < IPT; ++i) asm volatile("" : "+v"(kc[i]));
    __syncthreads();

    uint32_t total = 0;
    D* chain_desc = a.desc + (size_t)a.tile_base[chain] * kRadix;
    D win[kPassWindow];
    uint32_t taken = kNoWork;
    if (lb_wave) {
      const uint32_t d = (uint32_t)tid - kRadix;
      if (tid == taker) taken = take();
#pragma unroll
      for (int i = 0; i < W; ++i) total += off[i][d];
      msd_publish(chain_desc + (size_t)lt * kRadix + d,
                  Desc<D>::make(lt == 0 ? kStInclusive : kStAggregate, (D)total, a.parity), xcd_local);
      if (lt > 0) lookback_load(chain_desc, (int64_t)lt - 1, d, win);
    } else if (tid < kRadix) {
#pragma unroll
      for (int i = 0; i < W; ++i) total += off[i][tid];
    }
    const uint32_t excl = block_excl_scan_256(tid < kRadix ? total : 0u, sums, tid);
    if (tid < kRadix) {
      uint32_t r = excl;
#pragma unroll
      for (int i = 0; i < W; ++i) {
        const uint32_t c = off[i][tid];
        off[i][tid] = r;
        r += c;
      }
      if (chain != cur_chain) cur_base = digit_base(chain, (uint32_t)tid);
      s_prefix[tid] = cur_base - excl;
    }
    cur_chain = chain;
    if (tid == taker) s_tile = taken;
    __syncthreads();
    int64_t lb_t = (int64_t)lt - 1;
    uint32_t lb_prefix = 0;
    bool lb_done = false;
    if (lb_wave && lt > 0)
      lb_done = lookback_step(chain_desc, lb_t, (uint32_t)tid - kRadix, a.parity, win, lb_prefix);
    if (full) {
      uint32_t pos[IPT];
#pragma unroll
      for (int i = 0; i < IPT; ++i) pos[i] = min(off[w][pk[i] >> 16] + (pk[i] & 0xFFFFu), (uint32_t)TILE - 1);
#pragma unroll
      for (int i = 0; i < IPT; ++i) {
        keys[pos[i]] = kc[i];
        if constexpr (HV) vstage[pos[i]] = vc[i];
      }
    } else {
#pragma unroll
      for (int i = 0; i < IPT; ++i) {
        const uint32_t pos = off[w][pk[i] >> 16] + (pk[i] & 0xFFFFu);
        if (wb + i * kWave < chi && pos < (uint32_t)TILE) {
          keys[pos] = kc[i];
          if constexpr (HV) vstage[pos] = vc[i];
        }
      }
    }
    const uint32_t nxt = s_tile;
    if (nxt != kNoWork) {
      const uint32_t nc = nxt >> 20;
      load(chain_lo(nc), chain_hi(nc), nxt & 0xFFFFFu);
    }
    for (int i = lane; i < kRadix; i += kWave) off[w][i] = 0;
    if (lb_wave) {
      const uint32_t d = (uint32_t)tid - kRadix;
      if (lt > 0) {
        bool gave_up = false;
        const uint32_t prefix =
            lb_done ? lb_prefix : lookback_from(chain_desc, lb_t, d, a.parity, win, lb_prefix, a.spin_limit, gave_up);
        if (gave_up) atomicOr(a.status, kStatusLookback);
        msd_publish(chain_desc + (size_t)lt * kRadix + d, Desc<D>::make(kStInclusive, (D)(prefix + total), a.parity),
                    xcd_local);
        gbase[d] = s_prefix[d] + prefix;
      } else {
        gbase[d] = s_prefix[d];
      }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
      const uint32_t i = (uint32_t)(j * BLOCK + tid);
      if (full || i < tile_cnt) {
        const Bits kk = keys[i];
        const uint32_t o = min(gbase[digit_at<KT>(kk, shift)] + i, a.n - 1);
        a.dst[o] = kk;
        if constexpr (HV) a.vdst[o] = vstage[i];
      }
    }
    __syncthreads();
    cur = nxt;
  }
}

}  // namespace mgs
