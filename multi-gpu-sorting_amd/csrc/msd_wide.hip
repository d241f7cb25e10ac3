// Three-pass path of 8-byte keys and of keys with payloads (msd_wide.hpp):
// eligibility, scratch layout and the kernels that do not depend on the
// record type.
#include <cmath>
#include <cstdlib>

#include "msd_pass.hpp"
#include "msd_wide.hpp"
#include "radix_device.hpp"

namespace mgs {

namespace {


// ---------------------------------------------------------------------------
// scan: one workgroup of 256 threads per bucket b (the window's high byte),
// thread d = its low byte
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void wide_scan_kernel(const uint32_t* __restrict__ slices, uint32_t ranges,
                                                        uint32_t n, uint32_t cap,
                                                        const uint32_t* __restrict__ range_hist,
                                                        uint32_t* __restrict__ range_pref, MsdCtl* __restrict__ ctl,
                                                        uint32_t* __restrict__ sub_off,
                                                        uint32_t* __restrict__ bucket_tot,
                                                        uint32_t* __restrict__ leaders,
                                                        uint32_t* __restrict__ batch_cnt,
                                                        const uint32_t* __restrict__ range_bad,
                                                        const uint32_t* __restrict__ xcd_of) {
  if (ctl->off & kMsdOffSample) return;
  __shared__ uint32_t sums[4];
  __shared__ uint32_t s_max;
  const uint32_t b = blockIdx.x, d = threadIdx.x;
  const uint32_t s = b * kRadix + d;
  if (d == 0) s_max = 0;
  if (b == 0) {
    uint32_t m = 0, runs = 0;
    for (uint32_t c = d; c < ranges; c += kRadix) {
      const uint32_t cb = range_bad[c];
      if (cb & 1u) atomicOr(&ctl->off, kMsdOffOverflow);
      runs += cb >> 1;
      m |= 1u << (xcd_of[c] & 31u);
    }
    atomicOr(&ctl->xcd_mask, m);
    const uint32_t before = block_excl_scan_256(runs, sums, (int)d);
    if (d == kRadix - 1) ctl->runs = before + runs > n / 16 ? 1u : 0u;
    __syncthreads();  // every thread has read the scan's partial sums
  }
  __shared__ uint32_t s_cnt[kRadix];
  sum_slices(slices, ranges, b, s_cnt);
  const uint32_t cnt = s_cnt[d];
  if (cnt > cap) atomicOr(&ctl->off, kMsdOffSubBucket);
  const uint32_t excl = block_excl_scan_256(cnt, sums, (int)d);
  sub_off[s] = excl;
  if (d == kRadix - 1) bucket_tot[b] = excl + cnt;
  // Batches: a sub-bucket above cap / 2 is a batch by itself; the others are
  // cut where floor(offset / T) changes, with T = cap - (the largest of
  // them), so that a batch, which holds less than T plus its last
  // sub-bucket, fits the cap.
  const bool big = cnt > cap / 2;
  if (!big && cnt > 0) atomicMax(&s_max, cnt);
  __shared__ uint32_t s_off[kRadix], s_big[kRadix];
  s_off[d] = excl;
  s_big[d] = big ? 1u : 0u;
  __syncthreads();
  const uint32_t T = cap - s_max;
  const bool lead = d == 0 || big || s_big[d - 1] || excl / T != s_off[d - 1] / T;
  const uint32_t rank = block_excl_scan_256(lead ? 1u : 0u, sums, (int)d);
  if (lead) leaders[s - d + rank] = d;
  if (d == kRadix - 1) batch_cnt[b] = rank + (lead ? 1u : 0u);
  __syncthreads();
  // records of bucket b in the ranges before range c
  uint32_t carry = 0;
  for (uint32_t c0 = 0; c0 < ranges; c0 += kRadix) {
    const uint32_t c = c0 + d;
    const uint32_t v = c < ranges ? range_hist[(size_t)c * kRadix + b] : 0u;
    const uint32_t e = block_excl_scan_256(v, sums, (int)d);
    if (c < ranges) range_pref[(size_t)c * kRadix + b] = carry + e;
    carry += sums[0] + sums[1] + sums[2] + sums[3];
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// finish: one workgroup of 256 threads.  (A kernel of its own: as the last
// workgroup of the scan it needs an agent-scope release by each of the 256,
// which cost 20 us more than the launch.)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void wide_finish_kernel(MsdCtl* __restrict__ ctl, uint32_t n, uint32_t tile,
                                                          const uint32_t* __restrict__ bucket_tot,
                                                          uint32_t* __restrict__ bucket_start,
                                                          const uint32_t* __restrict__ batch_cnt,
                                                          uint32_t* __restrict__ batch_base, uint32_t chains1,
                                                          uint32_t tpc1, uint32_t* __restrict__ tile_base1,
                                                          uint32_t* __restrict__ tile_base2,
                                                          uint32_t* __restrict__ counters) {
  if (ctl->off) return;
  __shared__ uint32_t sums[4];
  __shared__ uint32_t s_xcd[kXcds];
  const uint32_t d = threadIdx.x;
  if (d < kXcds) s_xcd[d] = 0;
  const uint32_t bt = bucket_tot[d];
  const uint32_t bs = block_excl_scan_256(bt, sums, (int)d);
  bucket_start[d] = bs;
  if (d == kRadix - 1) bucket_start[kRadix] = bs + bt;
  atomicAdd(&s_xcd[d % kXcds], bt);
  __syncthreads();
  // pass 2 serves bucket b on XCD b mod 8: one XCD with more than twice its
  // share (and a few tiles) would leave the others idle
  if (d < kXcds && s_xcd[d] > 2 * (n / kXcds) + 64 * tile) atomicOr(&ctl->off, kMsdOffBucket);
  const uint32_t bc = batch_cnt[d];
  const uint32_t bb = block_excl_scan_256(bc, sums, (int)d);
  batch_base[d] = bb;
  if (d == kRadix - 1) {
    batch_base[kRadix] = bb + bc;
    ctl->batches = bb + bc;
  }
  __syncthreads();
  const uint32_t nt = (bt + tile - 1) / tile;
  tile_base2[d] = block_excl_scan_256(nt, sums, (int)d);
  if (d < chains1) tile_base1[d] = d * tpc1;
  counters[d] = 0;                          // pass 2
  if (d < kXcds) counters[kRadix + d] = 0;  // pass 1
}

}  // namespace

size_t wide_max(int rec) {
  // the mean sub-bucket plus seven deviations within the cap
  const double c = (double)wide_cap(rec), r = (std::sqrt(49.0 + 4.0 * c) - 7.0) / 2.0;
  return (size_t)(r * r * (double)kMsdBins);
}

bool wide_eligible(int kb, int vb, size_t n) {
  if (!msd_enabled() || n > wide_max(kb + vb)) return false;
  return n >= msd_min_override(wide_min(kb));
}

WidePlan wide_plan(int rec, size_t n) {
  WidePlan P{};
  const uint32_t tile = (uint32_t)wide_tile(rec);
  P.tiles = (uint32_t)((n + tile - 1) / tile);
  P.tiles_per_range = (P.tiles + kWideRanges - 1) / kWideRanges;
  P.range_keys = P.tiles_per_range * tile;
  P.ranges = (uint32_t)((n + P.range_keys - 1) / P.range_keys);
  P.ranges_per_chain = kWideRanges / kXcds;
  // fewer ranges than that: spread them over the eight chains all the same
  if (P.ranges < kWideRanges) P.ranges_per_chain = (P.ranges + kXcds - 1) / kXcds;
  P.chains1 = (P.ranges + P.ranges_per_chain - 1) / P.ranges_per_chain;
  return P;
}

WideLayout wide_layout(int rec, size_t n, size_t at, size_t ctl_at) {
  WideLayout L{};
  size_t o = at;
  auto take = [&](size_t bytes) {
    const size_t r = o;
    o = (o + bytes + 255) / 256 * 256;
    return r;
  };
  const size_t tile = (size_t)wide_tile(rec);
  const size_t tiles = (n + tile - 1) / tile;
  const size_t ranges = std::min<size_t>(tiles, kWideRanges);
  L.ctl = ctl_at;
  L.desc = take((tiles + kRadix + kXcds) * kRadix * 4);
  L.slices = take(ranges * (kMsdBins / 2) * 4);
  L.range_hist = take((size_t)kWideRanges * kRadix * 4);
  L.range_pref = take((size_t)kWideRanges * kRadix * 4);
  L.range_bad = take(kWideRanges * 4);
  L.xcd_of = take(kWideRanges * 4);
  L.sub_off = take((size_t)kMsdBins * 4);
  L.bucket_tot = take(kRadix * 4);
  L.bucket_start = take((kRadix + 1) * 4);
  L.leaders = take((size_t)kMsdBins * 4);
  L.batch_cnt = take(kRadix * 4);
  L.batch_base = take((kRadix + 1) * 4);
  L.batches = take((size_t)kMsdBins * 16);
  L.tile_base1 = take(kXcds * 4);
  L.tile_base2 = take(kRadix * 4);
  L.counters = take((kRadix + kXcds) * 4);
  L.end = o;
  return L;
}

int wide_tables(int rec, size_t n, const WidePlan& P, char* t, const WideLayout& L, hipStream_t s, Marks& mark) {
  auto at = [&](size_t o) { return reinterpret_cast<uint32_t*>(t + o); };
  MsdCtl* ctl = reinterpret_cast<MsdCtl*>(t + L.ctl);
  mark(s, "wide_scan");
  wide_scan_kernel<<<kRadix, kRadix, 0, s>>>(at(L.slices), P.ranges, (uint32_t)n, wide_cap(rec), at(L.range_hist),
                                             at(L.range_pref), ctl, at(L.sub_off), at(L.bucket_tot), at(L.leaders),
                                             at(L.batch_cnt), at(L.range_bad), at(L.xcd_of));
  mark(s, "wide_finish");
  wide_finish_kernel<<<1, kRadix, 0, s>>>(ctl, (uint32_t)n, (uint32_t)wide_tile(rec), at(L.bucket_tot),
                                          at(L.bucket_start), at(L.batch_cnt), at(L.batch_base), P.chains1,
                                          P.ranges_per_chain * P.tiles_per_range, at(L.tile_base1), at(L.tile_base2),
                                          at(L.counters));
  return check_launch();
}

}  // namespace mgs
