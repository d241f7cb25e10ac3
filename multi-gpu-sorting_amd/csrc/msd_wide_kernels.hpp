// Kernels and launch sequence of the three-pass path of one record type
// (msd_wide.hpp); instantiated per key type by msd_wide_*.hip.
#pragma once

#include <type_traits>

#include "block_sort.hpp"
#include "msd_pass.hpp"
#include "msd_wide.hpp"

namespace mgs {

namespace wide {

constexpr int kUpfrontBlock = 1024;

// The sample turns the path off before the read
// - when more than crowd_pairs() pairs of its 1024 keys share their window
//   value: c pairs say that a key's sub-bucket holds on average c n / 523776
//   records, and the largest one of a smooth density (normal keys) about 1.4
//   times that.  Uniform keys have 8 such pairs (1024^2 / 2 / 65536), more
//   than 24 once in a million inputs;
// - when one value has more than crowd_keys() of its keys, half again as many
//   as a sub-bucket of `cap` records has (heavy duplicates).  Five keys of
//   one value are in 5e-7 of uniform samples.
__device__ __forceinline__ uint32_t crowd_pairs(uint32_t n, uint32_t cap) {
  return max(24u, (uint32_t)((uint64_t)cap * 523776u * 5u / (7ull * n)));
}
__device__ __forceinline__ uint32_t crowd_keys(uint32_t n, uint32_t cap) {
  return max(4u, (uint32_t)((uint64_t)cap * 1536u / n));
}

// One read of the keys: workgroup c counts the window values of range c in a
// 65536-bin LDS histogram of 16-bit counters and stores it as its slice
// (bound by HBM up to 8-byte keys; 128 KB of LDS, one workgroup per CU).
template <int KT, bool VEC>
__global__ __launch_bounds__(kUpfrontBlock) void upfront_kernel(
    const typename Codec<KT>::Bits* __restrict__ keys, uint32_t n, uint32_t range_keys, uint32_t cap,
    MsdCtl* __restrict__ ctl, uint32_t* __restrict__ slices, uint32_t* __restrict__ range_hist,
    uint32_t* __restrict__ range_bad, uint32_t* __restrict__ xcd_of, uint32_t* __restrict__ desc, uint32_t desc_tiles,
    uint32_t* __restrict__ status) {
  using Bits = typename Codec<KT>::Bits;
  constexpr uint32_t kBits = sizeof(Bits) * 8;
  // bin b in word b >> 1, half b & 1
  __shared__ uint32_t h[kMsdBins / 2];
  __shared__ uint32_t s_rows[kRadix];
  __shared__ uint32_t s_runs, s_stray, s_pairs, s_crowd;
  __shared__ Bits s_and[kUpfrontBlock / kWave], s_or[kUpfrontBlock / kWave];
  const int tid = threadIdx.x;
  const uint32_t c = blockIdx.x;
  const int lane = tid & (kWave - 1), w = tid / kWave;
  for (int i = tid; i < kMsdBins / 2; i += kUpfrontBlock) h[i] = 0;
  if (tid == 0) {
    xcd_of[c] = xcc_id();
    s_stray = 0;
    s_pairs = 0;
    s_crowd = 0;
    s_runs = 0;
  }
  // the window: every workgroup reads the same 1024 keys, evenly spaced over
  // the input, and derives the same bits from them
  const Bits e_sample = Codec<KT>::enc(keys[((uint64_t)tid * (n - 1)) / (kUpfrontBlock - 1)]);
  {
    Bits ea = e_sample, eo = e_sample;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      ea &= __shfl_xor(ea, o, kWave);
      eo |= __shfl_xor(eo, o, kWave);
    }
    if (lane == 0) {
      s_and[w] = ea;
      s_or[w] = eo;
    }
  }
  __syncthreads();
  Bits s_a = ~Bits(0), s_o = 0;
#pragma unroll
  for (int i = 0; i < kUpfrontBlock / kWave; ++i) {
    s_a &= s_and[i];
    s_o |= s_or[i];
  }
  const uint32_t used = (uint32_t)bit_width<Bits>(s_a ^ s_o);  // low bits in which the sample differs
  const uint32_t low = used > 16u ? used - 16u : 0u;
  const Bits hi_mask = low + 16u < kBits ? ~Bits(0) << (low + 16u) : Bits(0);  // the shared bits above the window
  const Bits hi_val = s_a & hi_mask;
  auto window = [&](Bits enc) { return (uint32_t)(enc >> low) & 0xFFFFu; };
  auto add = [&](uint32_t b, uint32_t k) -> uint32_t {
    const uint32_t sh = (b & 1u) << 4;
    return (__hip_atomic_fetch_add(&h[b >> 1], k << sh, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) >> sh) &
           0xFFFFu;
  };
  {
    // sampled keys that share a window value
    const uint32_t b = window(e_sample);
    const uint32_t earlier = add(b, 1u);
    if (earlier) atomicAdd(&s_pairs, earlier);
    if (earlier >= crowd_keys(n, cap)) s_crowd = 1u;
    __syncthreads();
    h[b >> 1] = 0;
  }
  if (s_crowd || s_pairs > crowd_pairs(n, cap)) {
    if (c == 0 && tid == 0) ctl->off = kMsdOffSample;  // (the LSD sort clears the status word)
    return;
  }
  if (c == 0 && tid == 0) {  // nothing else writes these during this kernel
    *status = 0;
    ctl->off = 0;
    ctl->batch_next = 0;
    ctl->xcd_mask = 0;
    ctl->low = low;
    ctl->high[0] = (uint32_t)hi_val;
    ctl->high[1] = (uint32_t)((uint64_t)hi_val >> 32);
  }
  {
    // look-back descriptors of both passes: the tiles of the input read as
    // "empty" by pass 1 (status rotation 0) and, once pass 1 has left them
    // inclusive, by pass 2 (rotation 1); the further tiles of pass 2 (one
    // partial tile per bucket) start as "empty" under rotation 1
    uint4* d4 = reinterpret_cast<uint4*>(desc);
    const size_t words = (size_t)desc_tiles * kRadix;
    const size_t total = words + (size_t)(kRadix + kXcds) * kRadix;
    const size_t g = (size_t)c * kUpfrontBlock + tid, st = (size_t)gridDim.x * kUpfrontBlock;
    const uint32_t empty1 = Desc<uint32_t>::make(kStEmpty, 0u, 1);
    for (size_t i = g; i < total / 4; i += st) {
      const uint32_t v = 4 * i < words ? 0u : empty1;
      d4[i] = make_uint4(v, v, v, v);
    }
  }
  __syncthreads();
  const size_t lo = (size_t)c * range_keys;
  const size_t hi = std::min<size_t>((size_t)n, lo + range_keys);
  Bits stray = 0;  // bits above the window where a key differs from the sample
  uint32_t run_keys = 0;
  auto count = [&](Bits k) {
    const Bits e = Codec<KT>::enc(k);
    stray |= (e & hi_mask) ^ hi_val;
    add(window(e), 1u);
  };
  // consecutive keys of a lane: one add when they share a bin, and one for
  // all the lanes whose keys fall in the first lane's bin (runs of sorted
  // keys would put every lane on one counter); these are counted in run_keys
  constexpr int N = 16 / (int)sizeof(Bits);
  using Vec = typename std::conditional<sizeof(Bits) == 4, uint4, ulonglong2>::type;
  auto count_vec = [&](const Vec& v) {
    Bits x[N];
    if constexpr (N == 4) {
      x[0] = v.x, x[1] = v.y, x[2] = v.z, x[3] = v.w;
    } else {
      x[0] = v.x, x[1] = v.y;
    }
    uint32_t b[N];
    bool same = true;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const Bits e = Codec<KT>::enc(x[i]);
      stray |= (e & hi_mask) ^ hi_val;
      b[i] = window(e);
      same &= b[i] == b[0];
    }
    const bool in = same && b[0] == readfirstlane(b[0]);
    const uint64_t grp = ballot64(in);
    const uint32_t k = (uint32_t)N * (uint32_t)__popcll(grp);
    if (mbcnt64(ballot64(true)) == 0) run_keys += k;
    if (in) {
      if (mbcnt64(grp) == 0) add(b[0], k);
    } else if (same) {
      add(b[0], (uint32_t)N);
    } else {
#pragma unroll
      for (int i = 0; i < N; ++i) add(b[i], 1u);
    }
  };
  if (lo < hi) {
    if constexpr (VEC) {
      // range_keys is a multiple of the tile, so [lo, hi) starts 16-byte aligned
      constexpr int U = 4;
      const Vec* kv = reinterpret_cast<const Vec*>(keys + lo);
      const size_t nv = (hi - lo) / N;
      size_t i = tid;
      for (; i + (U - 1) * kUpfrontBlock < nv; i += U * kUpfrontBlock) {
        Vec v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = kv[i + u * kUpfrontBlock];
#pragma unroll
        for (int u = 0; u < U; ++u) count_vec(v[u]);
      }
      for (; i < nv; i += kUpfrontBlock) count_vec(kv[i]);
      for (size_t k = lo + nv * N + tid; k < hi; k += kUpfrontBlock) count(keys[k]);
    } else {
      for (size_t k = lo + tid; k < hi; k += kUpfrontBlock) count(keys[k]);
    }
  }
  __syncthreads();
  if (run_keys) atomicAdd(&s_runs, run_keys);
  if (stray) s_stray = 1u;
  // the range's histogram of the high byte: row r is the words [128 r, 128 r + 128)
  for (int r = w; r < kRadix; r += kUpfrontBlock / kWave) {
    const uint32_t a = h[r * 128 + lane], b = h[r * 128 + 64 + lane];
    uint32_t s = (a & 0xFFFFu) + (a >> 16) + (b & 0xFFFFu) + (b >> 16);
    s = wave_inclusive_sum(s);
    if (lane == kWave - 1) s_rows[r] = s;
  }
  __syncthreads();
  if (tid < kRadix) range_hist[(size_t)c * kRadix + tid] = s_rows[tid];
  if (tid < kWave) {
    // a wrapped 16-bit counter loses 65536 (high half) or 65535 (low half,
    // whose carry lands in the high half): the rows then fall short
    const uint32_t s = wave_inclusive_sum(s_rows[tid] + s_rows[tid + 64] + s_rows[tid + 128] + s_rows[tid + 192]);
    if (tid == kWave - 1)
      range_bad[c] = (s != (uint32_t)(hi > lo ? hi - lo : 0) || s_stray ? 1u : 0u) | (s_runs << 1);
  }
  uint4* dst = reinterpret_cast<uint4*>(slices + (size_t)c * (kMsdBins / 2));
  const uint4* src = reinterpret_cast<const uint4*>(h);
  for (int i = tid; i < kMsdBins / 8; i += kUpfrontBlock) dst[i] = src[i];
}

// Sort of the batches in place: workgroup g takes batches g, g + G, ... (G
// workgroups, two per CU, so that one loads or stores while the other
// sorts).  A batch's keys share the bits above the window and lie between
// its first and last window value.  Workgroup 0 also checks that both passes
// took every tile of every chain.
template <int KT, typename V, int BLOCK, int IPT>
__global__ __launch_bounds__(BLOCK, 4) void local_kernel(typename Codec<KT>::Bits* keys, V* vals,
                                                         const MsdCtl* __restrict__ ctl,
                                                         const uint4* __restrict__ batches,
                                                         const uint32_t* __restrict__ counters,
                                                         const uint32_t* __restrict__ bucket_start, uint32_t chains1,
                                                         uint32_t chain_keys1, uint32_t n, uint32_t tile,
                                                         uint32_t* __restrict__ status) {
  using Bits = typename Codec<KT>::Bits;
  using Smem = BlockSortSmem<Bits, V, BLOCK, IPT>;
  using VS = typename Smem::VS;
  if (ctl->off) return;
  __shared__ Smem sm;
  const int tid = threadIdx.x;
  if (blockIdx.x == 0) {
    // counters: [0, 256) pass 2 per bucket, [256, 264) pass 1 per chain
    if (tid < kRadix) {
      const uint32_t len = bucket_start[tid + 1] - bucket_start[tid];
      if (counters[tid] < (len + tile - 1) / tile) atomicOr(status, kStatusChainUnserved);
    } else if (tid < kRadix + (int)chains1) {
      const uint32_t c = tid - kRadix;
      const uint32_t len = min(n - c * chain_keys1, chain_keys1);
      if (counters[tid] < (len + tile - 1) / tile) atomicOr(status, kStatusChainUnserved);
    }
  }
  const uint32_t total = ctl->batches, low = ctl->low;
  const Bits high = (Bits)(((uint64_t)ctl->high[1] << 32) | ctl->high[0]);
  block_clear_row<BLOCK>(sm.off);
  for (uint32_t bi = blockIdx.x; bi < total; bi += gridDim.x) {
    const uint4 bt = batches[bi];
    const uint32_t m = readfirstlane(bt.y);
    if (m == 0) continue;
    const Bits mn = high | (Bits)bt.z << low;
    const Bits mx = high | (Bits)bt.w << low | ((Bits(1) << low) - 1);
    const Bits pad = Codec<KT>::dec(mx);
    const uint32_t nit = block_items<BLOCK>(m), wb = block_first<BLOCK>(nit);
    Bits k[IPT];
    VS v[IPT];
    const Bits* kb = keys + bt.x;
    static_for<IPT>([&](auto i) {
      k[i] = pad;
      if (wb + i * kWave < m && (uint32_t)i < nit) k[i] = kb[wb + i * kWave];
    });
    if constexpr (kHasVal<V>) {
      const V* vb = vals + bt.x;
      static_for<IPT>([&](auto i) {
        v[i] = 0;
        if (wb + i * kWave < m && (uint32_t)i < nit) v[i] = vb[wb + i * kWave];
      });
    }
    V* vo = nullptr;
    if constexpr (kHasVal<V>) vo = vals + bt.x;
    block_sort<KT, V, BLOCK, IPT>(sm, k, v, m, mn, mx, keys + bt.x, vo);
    __syncthreads();
  }
}

}  // namespace wide

template <int KT, int VT>
int wide_launch(const void* kin, void* kout, void* kalt, const void* vin, void* vout, void* valt, size_t n, char* t,
                const WideLayout& L, uint32_t* status, uint32_t spin_limit, hipStream_t s, Marks& mark) {
  using Bits = typename Codec<KT>::Bits;
  using V = typename ValOf<VT>::T;
  constexpr int KB = sizeof(Bits), VB = kValBytes<V>, REC = KB + VB;
  using Cfg = WideCfg<KB, VB>;
  const WidePlan P = wide_plan(REC, n);
  auto at = [&](size_t o) { return reinterpret_cast<uint32_t*>(t + o); };
  MsdCtl* ctl = reinterpret_cast<MsdCtl*>(t + L.ctl);
  const Bits* ki = static_cast<const Bits*>(kin);
  const uint32_t nn = (uint32_t)n;

  mark(s, "wide_upfront");
  if (reinterpret_cast<uintptr_t>(kin) % 16 == 0)
    wide::upfront_kernel<KT, true><<<P.ranges, wide::kUpfrontBlock, 0, s>>>(
        ki, nn, P.range_keys, Cfg::kCap, ctl, at(L.slices), at(L.range_hist), at(L.range_bad), at(L.xcd_of),
        at(L.desc), P.tiles, status);
  else
    wide::upfront_kernel<KT, false><<<P.ranges, wide::kUpfrontBlock, 0, s>>>(
        ki, nn, P.range_keys, Cfg::kCap, ctl, at(L.slices), at(L.range_hist), at(L.range_bad), at(L.xcd_of),
        at(L.desc), P.tiles, status);
  int rc = wide_tables(REC, n, P, t, L, s, mark);
  if (rc != MGS_OK) return rc;

  MsdPassArgs<Bits, V> a{};
  a.n = nn;
  a.bucket_start = at(L.bucket_start);
  a.chain_pref = at(L.range_pref);
  a.ranges_per_chain = P.ranges_per_chain;
  a.chain_keys = P.ranges_per_chain * P.range_keys;
  a.sub_off = at(L.sub_off);
  a.desc = at(L.desc);
  a.ctl = ctl;
  a.status = status;
  a.spin_limit = spin_limit;
  auto pass1 = msd_pass_kernel<KT, V, 1, Cfg::kBlock, Cfg::kIpt, 2>;
  auto pass2 = msd_pass_kernel<KT, V, 2, Cfg::kBlock, Cfg::kIpt, 2>;
  mark(s, "wide_pass1");
  a.src = ki;
  a.dst = static_cast<Bits*>(kalt);
  a.vsrc = static_cast<const V*>(vin);
  a.vdst = static_cast<V*>(valt);
  a.chains = P.chains1;
  a.tile_base = at(L.tile_base1);
  a.counters = at(L.counters) + kRadix;
  a.parity = 0;
  // (every chain has a home workgroup when the chains are not XCD-local)
  pass1<<<std::max(std::min(resident_blocks(pass1, Cfg::kBlock), P.tiles), P.chains1), Cfg::kBlock, 0, s>>>(a);
  mark(s, "wide_pass2");
  a.src = static_cast<const Bits*>(kalt);
  a.dst = static_cast<Bits*>(kout);
  a.vsrc = static_cast<const V*>(valt);
  a.vdst = static_cast<V*>(vout);
  a.chains = kRadix;
  a.tile_base = at(L.tile_base2);
  a.counters = at(L.counters);
  a.parity = 1;
  a.leaders = at(L.leaders);
  a.batch_cnt = at(L.batch_cnt);
  a.batch_base = at(L.batch_base);
  a.batches = reinterpret_cast<uint4*>(t + L.batches);
  pass2<<<resident_blocks(pass2, Cfg::kBlock), Cfg::kBlock, 0, s>>>(a);
  mark(s, "wide_local");
  constexpr int LB = 512, LI = Cfg::kLocalIpt;
  auto local = wide::local_kernel<KT, V, LB, LI>;
  local<<<resident_blocks(local, LB), LB, 0, s>>>(static_cast<Bits*>(kout), static_cast<V*>(vout), ctl,
                                                 reinterpret_cast<const uint4*>(t + L.batches), at(L.counters),
                                                 at(L.bucket_start), P.chains1, a.ranges_per_chain * P.range_keys, nn,
                                                 (uint32_t)Cfg::kTile, status);
  return check_launch();
}

}  // namespace mgs
