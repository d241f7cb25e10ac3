// Batched segmented sort: thousands of independent arrays in a fixed launch
// sequence whose grid sizes depend only on (nseg, max_total_keys, tuning), so
// a call can be captured once in a hipGraph and replayed for new data.
//
//   classify  one workgroup: resolves each segment's position (offsets form:
//             [offsets[s], offsets[s+1]); ranges form: [ranges[2s],
//             ranges[2s+1]) anywhere in the array, non-overlapping) and its
//             place in the compact scratch buffer; a segment of at most
//             small_max records becomes a batch of the local sort, a longer
//             one a node of the first split level
//   split level l (up to three): every node is scattered into at most 256
//             children in key order, by
//     count     per tile of every node: the digit of each key and their
//               counts.  A node's digits are its own: 254 equal steps of the
//               encoded key between (about) the first and the last hundredth
//               of 255 sampled keys, and one digit for what lies below and
//               above; or, where too many keys would share a step, the
//               samples themselves as bounds, with a digit of its own for a
//               value that several have -- monotone in the key whatever the
//               sample missed
//     chunk     where segments are very long: the offsets inside each 64 tiles
//     scan      per node: the tiles' (or chunks') offsets, and what becomes of the
//               children: consecutive ones that fit one workgroup together
//               become a batch, one that does not becomes a node of the next
//               level, and one whose keys are all equal is done
//     scatter   per tile: the records to their child, in input order
//   long      children that are still too long after the last level: one
//             workgroup each streams them through HBM byte by byte
//   local     every batch is sorted in LDS (block_sort.hpp)
//
// A level moves a record once and reads its key twice, so an 8-byte key with
// a payload takes one to two levels and the local sort instead of eight LSD
// passes.  Bounds from the sample divide keys of any distribution into children
// of at most about a fortieth, so the levels bring them to what one workgroup
// sorts in LDS up to chance: of 868 calls with 23 distributions one left children,
// two (49 us).  (Inputs made against the sample's fixed places may leave long ones:
// one workgroup takes 6 to 9 ns a record of 8-byte keys.)  With equal steps alone,
// log-uniform u64 keys left 61% of 2^23 records to one workgroup: 45.6 ms, now 0.28;
// 2^26 doubles 1 - eps 336 ms, now 1.55.
// Against LSD passes over all long segments at once and one
// workgroup for each middle one: u64 + u32, 1024 segments of 2^8 to 2^22, 26.3
// -> 12.3 ms; u32, 256 ranges of 2^10 to 2^18, 331 -> 166 us; f64, normal, 64
// of 2^10 to 2^22, 2518 -> 752 us.
#include <type_traits>

#include "block_sort.hpp"
#include "internal.hpp"
#include "radix_device.hpp"

namespace mgs {

namespace {

constexpr int kMaxLevels = 3;

struct SegCtl {
  uint32_t status;   // the call's status word (first word of temp)
  uint32_t skipped;  // segments left unsorted: malformed bounds or beyond max_total
  uint32_t n_batches, n_long;
  uint64_t alloc[kMaxLevels + 1];  // level's nodes << 32 | their tiles
};

// A range of a segment to be split: records [off, off + len), its tiles from
// tile0 of the level on, and its digits (written by the count): 0 below
// `base`, 255 above `top`, between them 1 + the step, which is the high word
// of ((key - base) >> shift) mul (254 even steps), or key - base itself where
// mul is 0 (every value a step).
// shift kBySample: the sample's values are the bounds of the digits instead,
// and the bits of `same` tell which digits hold one value only.
// shift kDone (written by the scan): one key in all places, nothing to scatter.
struct Node {
  uint32_t seg, off, len, tile0;
  uint64_t base, top;
  uint32_t mul, shift;
  uint64_t same[kRadix / kWave];
};
enum : uint32_t { kBySample = 64, kDone = 65 };

// Where a batch's records are.
enum : uint32_t { kSrcIn = 0, kSrcAlt = 1, kSrcOut = 2 };

// Per-segment table written by classify: first key in the key array, first
// payload in the payload array, first slot in the compact scratch buffer.
struct SegTab {
  uint64_t* begin;
  uint64_t* vbegin;
  uint64_t* alt;
};

constexpr int kClassifyBlock = 1024;

// Exclusive scan of three counters across a 1024-thread block.
__device__ inline void block_scan3(uint32_t a, uint32_t b, uint32_t c, uint32_t& ea, uint32_t& eb, uint32_t& ec,
                                   uint32_t& ta, uint32_t& tb, uint32_t& tc, uint32_t (*sm)[16]) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const uint32_t ia = wave_inclusive_sum(a), ib = wave_inclusive_sum(b), ic = wave_inclusive_sum(c);
  if (lane == 63) {
    sm[0][w] = ia;
    sm[1][w] = ib;
    sm[2][w] = ic;
  }
  __syncthreads();
  uint32_t ba = 0, bb = 0, bc = 0, sa = 0, sb = 0, sc = 0;
  for (int i = 0; i < kClassifyBlock / 64; ++i) {
    if (i < w) {
      ba += sm[0][i];
      bb += sm[1][i];
      bc += sm[2][i];
    }
    sa += sm[0][i];
    sb += sm[1][i];
    sc += sm[2][i];
  }
  ea = ba + ia - a;
  eb = bb + ib - b;
  ec = bc + ic - c;
  ta = sa;
  tb = sb;
  tc = sc;
  __syncthreads();
}

// Exclusive scan of 64-bit values across a 1024-thread block; *total gets
// the block sum.
__device__ inline uint64_t block_excl_scan_u64(uint64_t v, uint64_t* sm, uint64_t* total) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  uint64_t incl = v;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const uint64_t t = __shfl_up(incl, off, kWave);
    if (lane >= off) incl += t;
  }
  if (lane == 63) sm[w] = incl;
  __syncthreads();
  uint64_t base = 0, sum = 0;
  for (int i = 0; i < kClassifyBlock / 64; ++i) {
    if (i < w) base += sm[i];
    sum += sm[i];
  }
  *total = sum;
  __syncthreads();
  return base + incl - v;
}

// Inclusive running maximum of 64-bit values across a 1024-thread block;
// *total gets the block maximum.
__device__ inline uint64_t block_incl_max_u64(uint64_t v, uint64_t* sm, uint64_t* total) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  uint64_t incl = v;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const uint64_t t = __shfl_up(incl, off, kWave);
    if (lane >= off) incl = incl > t ? incl : t;
  }
  if (lane == 63) sm[w] = incl;
  __syncthreads();
  uint64_t base = 0, all = 0;
  for (int i = 0; i < kClassifyBlock / 64; ++i) {
    if (i < w) base = base > sm[i] ? base : sm[i];
    all = all > sm[i] ? all : sm[i];
  }
  *total = all;
  __syncthreads();
  return incl > base ? incl : base;
}

template <bool RANGES>
__global__ __launch_bounds__(kClassifyBlock) void seg_classify_kernel(const uint64_t* __restrict__ bounds,
                                                                      const uint64_t* __restrict__ val_begin,
                                                                      uint32_t nseg, uint64_t max_total,
                                                                      uint64_t max_seg,
                                                                      uint32_t small_max, uint32_t tile, SegTab tab,
                                                                      uint4* batches, Node* nodes, SegCtl* ctl) {
  __shared__ uint32_t sm[3][16];
  __shared__ uint64_t sm64[16];
  const int tid = threadIdx.x;
  uint32_t run_s = 0, run_l = 0, run_t = 0, skipped = 0;
  uint64_t run_alt = 0, run_max = 0;
  const uint64_t base0 = RANGES ? 0 : bounds[0];
  for (uint32_t base = 0; base < nseg; base += kClassifyBlock) {
    const uint32_t s = base + tid;
    uint64_t b = 0, want = 0;
    bool ok = true;
    if (s < nseg) {
      const uint64_t lo = RANGES ? bounds[2 * (size_t)s] : bounds[s];
      const uint64_t hi = RANGES ? bounds[2 * (size_t)s + 1] : bounds[s + 1];
      b = lo;
      ok = hi >= lo && hi - lo < (uint64_t(1) << 32) && hi - lo <= max_seg;
      want = ok ? hi - lo : 0;
    }
    // compact scratch slot: the offsets form keeps the segment's distance
    // from the first offset; the ranges form packs the segments in order
    uint64_t alt = 0, chunk = 0;
    if (RANGES) {
      alt = run_alt + block_excl_scan_u64(want, sm64, &chunk);
      run_alt += chunk;
    } else {
      // offsets must not decrease: a segment is taken only if it starts at
      // or after every earlier offset, so the taken segments are disjoint
      // (b is at least every earlier offset iff the running maximum up to
      // and including it is b itself)
      const uint64_t m = block_incl_max_u64(s < nseg ? b : 0, sm64, &chunk);
      if (s < nseg && (m != b || b < run_max)) ok = false;
      run_max = run_max > chunk ? run_max : chunk;
      alt = b - base0;
    }
    if (s < nseg && (!ok || (!RANGES && b < base0) || alt > max_total || want > max_total - alt)) {
      ok = false;  // left unsorted rather than running past the scratch buffer
      want = 0;
    }
    const uint32_t len = (uint32_t)want;
    if (s < nseg) {
      tab.begin[s] = b;
      tab.vbegin[s] = (RANGES && val_begin != nullptr) ? val_begin[s] : b;
      tab.alt[s] = alt;
    }
    const uint32_t bad = (s < nseg && !ok) ? 1u : 0u;
    const uint32_t is_s = (s < nseg && len > 0 && len <= small_max) ? 1u : 0u;
    const uint32_t is_l = (s < nseg && len > small_max) ? 1u : 0u;
    const uint32_t nt = is_l ? (len + tile - 1) / tile : 0u;
    uint32_t es, el, et, eb, e1, e2, ts, tl, tt, tb, t1, t2;
    block_scan3(is_s, is_l, nt, es, el, et, ts, tl, tt, sm);
    block_scan3(bad, 0, 0, eb, e1, e2, tb, t1, t2, sm);
    if (is_s) batches[run_s + es] = make_uint4(s, 0, len, kSrcIn);
    if (is_l) nodes[run_l + el] = Node{s, 0, len, run_t + et, 0, 0, 0, 0, {}};
    run_s += ts;
    run_l += tl;
    run_t += tt;
    skipped += tb;
  }
  if (tid == 0) {
    ctl->n_batches = run_s;
    ctl->n_long = 0;
    ctl->alloc[0] = (uint64_t)run_l << 32 | run_t;
    for (int l = 1; l <= kMaxLevels; ++l) ctl->alloc[l] = 0;
    ctl->skipped = skipped;
    ctl->status = skipped ? kStatusSkipped : 0u;
  }
}

// ---------------------------------------------------------------------------
// Long ranges: one workgroup sorts a whole range, pass by pass, walking its
// tiles in order and carrying the per-digit running offsets in LDS, so no
// cross-workgroup look-back is needed.
// ---------------------------------------------------------------------------
template <int KT, typename V, int BLOCK, int IPT>
__device__ void medium_sort_block(const typename Codec<KT>::Bits* k_in, typename Codec<KT>::Bits* k_alt,
                                  typename Codec<KT>::Bits* k_out, const V* v_in, V* v_alt, V* v_out, uint32_t n) {
  using Bits = typename Codec<KT>::Bits;
  constexpr int W = BLOCK / kWave;
  constexpr int TILE = BLOCK * IPT;
  constexpr bool HV = kHasVal<V>;
  constexpr int P = (int)sizeof(Bits);
  using VS = typename std::conditional<HV, V, uint32_t>::type;
  __shared__ Bits keys[TILE];
  __shared__ VS vstage[HV ? TILE : 1];
  __shared__ uint32_t off[W][kRadix];
  __shared__ uint32_t hist[P][kRadix];
  __shared__ uint32_t run[kRadix];
  __shared__ uint32_t gbase[kRadix];
  __shared__ uint32_t sums[4];

  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int w = tid / kWave;

  // Histogram of every byte.
  for (int i = tid; i < P * kRadix; i += BLOCK) (&hist[0][0])[i] = 0;
  __syncthreads();
  for (uint32_t i = tid; i < n; i += BLOCK) {
    const Bits k = k_in[i];
#pragma unroll
    for (int p = 0; p < P; ++p) lds_count_wave(&hist[0][0], p * kRadix + digit_of<KT>(k, 8 * p));
  }
  __syncthreads();
  if (k_in == k_out) {  // one key in all places: in order
    const Bits k0 = k_in[0];
    bool one = true;
#pragma unroll
    for (int p = 0; p < P; ++p) one &= hist[p][digit_of<KT>(k0, 8 * p)] == n;
    if (one) return;
  }

  for (int p = 0; p < P; ++p) {
    const int shift = 8 * p;
    const Bits* src = p == 0 ? k_in : ((p & 1) ? k_alt : k_out);
    Bits* dst = (p & 1) ? k_out : k_alt;
    const V* vsrc = nullptr;
    V* vdst = nullptr;
    if constexpr (HV) {
      vsrc = p == 0 ? v_in : ((p & 1) ? v_alt : v_out);
      vdst = (p & 1) ? v_out : v_alt;
    }
    {  // running digit offsets start at the exclusive histogram scan
      const uint32_t c = tid < kRadix ? hist[p][tid] : 0u;
      const uint32_t e = block_excl_scan_256(c, sums, tid);
      if (tid < kRadix) run[tid] = e;
    }
    for (uint32_t tb = 0; tb < n; tb += TILE) {
      for (int i = tid; i < W * kRadix; i += BLOCK) (&off[0][0])[i] = 0;
      __syncthreads();
      const uint32_t tile_cnt = min((uint32_t)TILE, n - tb);
      Bits key[IPT];
      VS val[IPT];
      uint32_t dg[IPT], rk[IPT];
      const uint32_t wb = tb + (uint32_t)(w * IPT * kWave + lane);
#pragma unroll
      for (int k = 0; k < IPT; ++k) {
        const uint32_t idx = wb + k * kWave;
        key[k] = idx < n ? src[idx] : Bits(0);
        if constexpr (HV) val[k] = idx < n ? vsrc[idx] : VS(0);
        dg[k] = digit_of<KT>(key[k], shift);
      }
#pragma unroll
      for (int k = 0; k < IPT; ++k)
        if (wb + k * kWave < n) rk[k] = rank_wave_atomic<true>(dg[k], off[w]);
      __syncthreads();
      uint32_t total = 0;
      if (tid < kRadix) {
#pragma unroll
        for (int i = 0; i < W; ++i) total += off[i][tid];
      }
      const uint32_t excl = block_excl_scan_256(total, sums, tid);
      if (tid < kRadix) {
        uint32_t r = excl;
#pragma unroll
        for (int i = 0; i < W; ++i) {
          const uint32_t c = off[i][tid];
          off[i][tid] = r;
          r += c;
        }
        gbase[tid] = run[tid] - excl;
        run[tid] += total;
      }
      __syncthreads();
#pragma unroll
      for (int k = 0; k < IPT; ++k) {
        const uint32_t pos = off[w][dg[k]] + rk[k];
        if (wb + k * kWave < n && pos < (uint32_t)TILE) {
          keys[pos] = key[k];
          if constexpr (HV) vstage[pos] = val[k];
        }
      }
      __syncthreads();
#pragma unroll
      for (int j = 0; j < IPT; ++j) {
        const uint32_t i = (uint32_t)(j * BLOCK + tid);
        if (i < tile_cnt) {
          const Bits kk = keys[i];
          const uint32_t o = gbase[digit_of<KT>(kk, shift)] + i;
          if (o < n) {
            dst[o] = kk;
            if constexpr (HV) vdst[o] = vstage[i];
          }
        }
      }
      __syncthreads();
    }
    __threadfence_block();
    __syncthreads();
  }
}

template <int KT, typename V, int BLOCK, int IPT>
__global__ __launch_bounds__(BLOCK) void seg_long_kernel(typename Codec<KT>::Bits* k_alt,
                                                         typename Codec<KT>::Bits* k_out, V* v_alt, V* v_out,
                                                         SegTab tab, const uint4* __restrict__ list,
                                                         const SegCtl* __restrict__ ctl) {
  const uint32_t cnt = ctl->n_long;
  for (uint32_t i = blockIdx.x; i < cnt; i += gridDim.x) {
    const uint4 e = list[i];
    const uint64_t ob = tab.begin[e.x] + e.y, ab = tab.alt[e.x] + e.y;
    V *va = nullptr, *vo = nullptr;
    if constexpr (kHasVal<V>) {
      va = v_alt + ab;
      vo = v_out + tab.vbegin[e.x] + e.y;
    }
    if (e.w == kSrcAlt) {  // (the passes start from the output)
      for (uint32_t j = threadIdx.x; j < e.z; j += BLOCK) {
        k_out[ob + j] = k_alt[ab + j];
        if constexpr (kHasVal<V>) vo[j] = va[j];
      }
      __threadfence_block();
      __syncthreads();
    }
    medium_sort_block<KT, V, BLOCK, IPT>(k_out + ob, k_alt + ab, k_out + ob, vo, va, vo, e.z);
    __syncthreads();
  }
}

// The node of tile g: the last one with tile0 <= g.
__device__ __forceinline__ uint32_t find_node(const Node* __restrict__ nodes, uint32_t n, uint32_t g) {
  uint32_t lo = 0, hi = n;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (nodes[mid].tile0 <= g)
      lo = mid;
    else
      hi = mid;
  }
  return lo;
}

// A node's digits, and the digit of a key.
template <typename Bits>
struct Steps {
  Bits base, top;
  uint32_t mul, shift;
};
template <typename Bits>
__device__ __forceinline__ uint32_t step_of(Bits e, const Steps<Bits>& st) {
  const uint32_t t = (uint32_t)((Bits)(e - st.base) >> st.shift);
  uint32_t d = (st.mul ? __umulhi(t, st.mul) : t) + 1u;
  d = e < st.base ? 0u : d;
  return e > st.top ? 255u : d;
}
template <int KT>
__device__ __forceinline__ uint32_t step_digit(typename Codec<KT>::Bits raw, const Steps<typename Codec<KT>::Bits>& st) {
  return step_of<typename Codec<KT>::Bits>(Codec<KT>::enc(raw), st);
}

// ---------------------------------------------------------------------------
// The sample of a range: kSamples of its keys, one at a hashed place in each
// of as many equal stretches (at even distances, keys that repeat with the
// stride would all look alike).
// Thread t of the first 256 gives the t-th key, encoded, and `sorted` holds
// them in order on return; key and rank are working space.  Every thread of
// the block calls it.
// ---------------------------------------------------------------------------
constexpr uint32_t kSamples = 255;

template <int KT, int BLOCK>
__device__ __forceinline__ void sort_sample(const typename Codec<KT>::Bits* __restrict__ keys, uint32_t len,
                                            typename Codec<KT>::Bits* key, uint32_t* rank,
                                            typename Codec<KT>::Bits* sorted) {
  using Bits = typename Codec<KT>::Bits;
  const uint32_t t = threadIdx.x;
  if (t < (uint32_t)kRadix) {
    Bits x = ~Bits(0);  // thread 255: a place behind the sample
    if (t < kSamples) {
      const uint32_t a = (uint32_t)((uint64_t)len * t / kSamples), b = (uint32_t)((uint64_t)len * (t + 1) / kSamples);
      uint32_t h = (t + 1) * 0x9E3779B9u ^ len;
      h = (h ^ (h >> 16)) * 0x85EBCA6Bu;
      h = (h ^ (h >> 13)) * 0xC2B2AE35u;
      x = Codec<KT>::enc(keys[min(a + __umulhi(h ^ (h >> 16), b - a), len - 1)]);
    }
    key[t] = x;
    rank[t] = 0;
  }
  __syncthreads();
  {
    // the rank of every key among a part of the others per thread (ties by place)
    constexpr uint32_t kPart = kRadix * kRadix / BLOCK;
    const uint32_t i = t & (kRadix - 1), from = t / kRadix * kPart;
    const Bits x = key[i];
    uint32_t r = 0;
#pragma unroll 8
    for (uint32_t j = from; j < from + kPart; ++j) r += (key[j] < x || (key[j] == x && j < i)) ? 1u : 0u;
    atomicAdd(&rank[i], r);
  }
  __syncthreads();
  if (t < (uint32_t)kRadix) sorted[rank[t]] = key[t];
  __syncthreads();
}

// Turns the sorted sample into the bounds of the digits: digit d holds the keys
// from bound d - 1 on and below bound d.  A value that the sample has more than
// once is followed by the value one above it, and so has a digit of its own
// (a sample sort with equality buckets: Sanders and Winkel, Super Scalar Sample
// Sort, 2004).  Returns whether digit threadIdx.x (< 256) holds one value only.
template <typename Bits>
__device__ __forceinline__ bool sample_bounds(Bits* sorted) {
  const uint32_t t = threadIdx.x;
  Bits x = 0;
  if (t < kSamples) {
    x = sorted[t];
    if (t > 0 && sorted[t - 1] == x && x != ~Bits(0)) ++x;
  }
  __syncthreads();
  if (t < kSamples) sorted[t] = x;
  __syncthreads();
  if (t >= (uint32_t)kRadix) return false;
  const Bits below = t > 0 ? sorted[t - 1] : Bits(0);
  return t < kSamples ? sorted[t] - below == 1 : below == ~Bits(0);
}

template <int KT>
__device__ __forceinline__ uint32_t sample_digit(typename Codec<KT>::Bits raw, const typename Codec<KT>::Bits* bounds) {
  using Bits = typename Codec<KT>::Bits;
  const Bits e = Codec<KT>::enc(raw);
  // (in byte offsets: a step is a compare, a select and an add beside the load)
  const char* const b = reinterpret_cast<const char*>(bounds);
  uint32_t o = 0;
#pragma unroll
  for (uint32_t s = kRadix / 2; s > 0; s >>= 1)
    o += *reinterpret_cast<const Bits*>(b + o + (s - 1) * sizeof(Bits)) <= e ? s * (uint32_t)sizeof(Bits) : 0u;
  return o / (uint32_t)sizeof(Bits);
}

// Whether the sample's values bound the digits of a node with `left` levels to
// go.  Even steps cost one multiplication per key instead of eight dependent
// LDS reads, and leave uniform keys in children of one size, where the largest
// of 256 digits between samples holds about 6 / 256 of the records (but that
// whatever the keys are).  So the samples bound them only where steps would not
// bring the children to the cap:
// - on the last level, where a step has more samples than half the cap's share
//   of them;
// - before it, where one surely has more than the cap's share (two deviations;
//   a step of uniform keys has one sample, the fullest of normal ones two), and
//   one of: the samples' largest child still fits (an eighth of the samples); the
//   step has more than the later levels bring to the cap if each of them leaves a
//   64th in its largest child; or the next level's steps, between the samples
//   that share a step, would not part these.  So a level of steps comes before
//   another where that helps: the exponents of floats fill a level's steps very
//   unevenly, but the keys of one exponent are even (normal floats, 2^20: 85 us
//   by steps, 114 with bounds from the sample on the first level).  The same value
//   several times counts as not parted: its digit ends here.
// Sorted samples that share a step are neighbours, so a step has more than K of
// them exactly if one shares it with the K-th after it: every wavefront looks at
// all of them by itself, without a barrier.  sorted: the sample; key, low and high:
// working space for 256 values each; every thread of the block calls it.
template <typename Bits>
__device__ __forceinline__ bool crowded(const Bits* sorted, const Steps<Bits>& st, uint32_t len, uint32_t cap, int left,
                                        uint32_t* key, Bits* low, Bits* high) {
  const uint32_t t = threadIdx.x, lane = t & (kWave - 1);
  const float share = (float)cap * kRadix / (float)len;  // samples among cap records
  const uint32_t may = max(4u, (uint32_t)(0.5f * share));
  const uint32_t must = max(8u, (uint32_t)((1.0f + sqrtf(1.0f + share)) * (1.0f + sqrtf(1.0f + share))));
  auto more_than = [&](uint32_t k, auto step) {
    bool any = false;
    for (uint32_t i = lane; i + k < kSamples; i += kWave) any |= step(i) == step(i + k);
    return ballot64(any) != 0;
  };
  auto step = [&](uint32_t i) { return step_of<Bits>(sorted[i], st); };
  if (left == 1) return more_than(may, step);
  if (!more_than(must, step)) return false;
  if (share >= 8.0f) return true;
  if (more_than(max(must, (uint32_t)min((float)kSamples, share * (left == 2 ? 64.0f : 4096.0f))), step)) return true;
  const uint32_t d = t < kSamples ? step(t) : 0u;
  if (t < kSamples) {
    if (t == 0 || step(t - 1) != d) low[d] = sorted[t];
    if (t == kSamples - 1 || step(t + 1) != d) high[d] = sorted[t];
  }
  __syncthreads();
  if (t < kSamples) {
    const Bits a = low[d], w = high[d] - a;
    key[t] = d * kRadix + (w ? (uint32_t)(254.0 * ((double)(sorted[t] - a) / (double)w)) : 0u);
  }
  __syncthreads();
  const bool both = more_than(left == 2 ? may : must, [&](uint32_t i) { return key[i]; });
  __syncthreads();  // key, low and high are the caller's again
  return both;
}

// ---------------------------------------------------------------------------
// count: workgroup b takes the tiles [T b / B, T (b + 1) / B) of the level,
// which mostly share a node; a node's digits are derived anew by every
// workgroup that meets it (from the same samples) and kept for the scatter by
// the one with its first tile.
// whole > 0 (first level only): the call sorts one array of so many records,
// and workgroup 0 writes what classify would.
// ---------------------------------------------------------------------------
constexpr int kCountBlock = 512;

template <int KT>
__global__ __launch_bounds__(kCountBlock, 8) void seg_count_kernel(const typename Codec<KT>::Bits* __restrict__ src,
                                                                SegTab tab, const uint64_t* place, Node* nodes,
                                                                uint32_t* __restrict__ rows, uint32_t tile,
                                                                uint32_t cap, SegCtl* ctl, int level, int left,
                                                                uint32_t whole) {
  using Bits = typename Codec<KT>::Bits;
  __shared__ Bits smp[kRadix], bounds[kRadix];
  __shared__ uint32_t rank[kRadix];
  __shared__ alignas(8) uint32_t h[kCountBlock / 128][kRadix];
  uint32_t n_nodes = 1, n_tiles = (whole + tile - 1) / tile;
  if (whole == 0) {
    n_nodes = (uint32_t)(ctl->alloc[level] >> 32);
    n_tiles = (uint32_t)ctl->alloc[level];
  } else if (blockIdx.x == 0 && threadIdx.x == 0) {
    tab.begin[0] = tab.vbegin[0] = tab.alt[0] = 0;
    nodes[0].seg = nodes[0].off = nodes[0].tile0 = 0;
    nodes[0].len = whole;
    ctl->status = ctl->skipped = ctl->n_batches = ctl->n_long = 0;
    ctl->alloc[0] = (uint64_t)1 << 32 | n_tiles;
    for (int l = 1; l <= kMaxLevels; ++l) ctl->alloc[l] = 0;
  }
  const uint32_t g0 = (uint32_t)((uint64_t)n_tiles * blockIdx.x / gridDim.x);
  const uint32_t g1 = (uint32_t)((uint64_t)n_tiles * (blockIdx.x + 1) / gridDim.x);
  if (g0 >= g1) return;
  const int tid = threadIdx.x;
  uint32_t* const my = h[tid / 128];  // one histogram per two wavefronts
  uint32_t ni = whole ? 0 : find_node(nodes, n_nodes, g0);
  bool fresh = true, by_sample = false;
  Steps<Bits> st{};
  uint32_t len = 0, tile0 = 0;
  const Bits* keys = nullptr;
  for (uint32_t g = g0; g < g1; ++g) {
    if (!fresh && ni + 1 < n_nodes && nodes[ni + 1].tile0 <= g) {
      ++ni;
      fresh = true;
    }
    if (fresh) {
      fresh = false;
      keys = src;
      len = whole;
      if (whole == 0) {
        keys += place[nodes[ni].seg] + nodes[ni].off;
        len = nodes[ni].len;
        tile0 = nodes[ni].tile0;
      }
      sort_sample<KT, kCountBlock>(keys, len, smp, rank, bounds);
      // between the third and the third last sample and a sixty-fourth of their
      // distance further on both sides, or a thirty-second where the steps then
      // still reach the cap (a sixty-fourth leaves more than 0.7% of uniform keys
      // below or above in one array of ten, and 2^20 u64 keys a second level:
      // 58 us -> 82); or a step per value around the samples where 254 values,
      // one below and one above cover them (keys of one byte)
      Bits lo = bounds[0], hi = bounds[kSamples - 1], more;
      if (hi - lo > 253 && hi - lo <= 255) {
        ++lo;
        hi = lo + 253;
        more = 0;
      } else if (hi - lo <= 253) {
        more = (253 - (hi - lo)) / 2;
      } else {
        lo = bounds[2];
        hi = bounds[kSamples - 3];
        more = (hi - lo) / (len / 238 <= cap ? 32 : 64);
      }
      lo = lo > more ? lo - more : Bits(0);
      hi = ~Bits(0) - hi > more ? hi + more : ~Bits(0);
      st.base = lo;
      st.top = hi;
      const Bits range = hi - lo;
      st.mul = 0;
      st.shift = 0;
      by_sample = false;
      if (range > 253) {  // 254 even steps
        st.shift = (uint32_t)max(bit_width<Bits>(range) - 32, 0);
        st.mul = (uint32_t)((254ull << 32) / ((uint64_t)(uint32_t)(range >> st.shift) + 1u));
        static_assert(sizeof(h) >= kRadix * sizeof(Bits), "working space");
        if (len > cap) by_sample = crowded<Bits>(bounds, st, len, cap, left, rank, smp, reinterpret_cast<Bits*>(&h[0][0]));
      }
      if (by_sample) {
        const uint64_t one = ballot64(sample_bounds<Bits>(bounds));
        if (tid < kRadix && (tid & (kWave - 1)) == 0 && tile0 >= g0) nodes[ni].same[tid / kWave] = one;
      }
      if (tid == 0 && tile0 >= g0) {
        nodes[ni].base = (uint64_t)st.base;
        nodes[ni].top = (uint64_t)st.top;
        nodes[ni].mul = st.mul;
        nodes[ni].shift = by_sample ? (uint32_t)kBySample : st.shift;
      }
    }
    for (int i = tid; i < (kCountBlock / 128) * kRadix; i += kCountBlock) (&h[0][0])[i] = 0;
    __syncthreads();
    const uint32_t t0 = (g - tile0) * tile, t1 = min(len, t0 + tile);
    // U keys at a time in flight
    auto count = [&](auto U, auto digit) {
      uint32_t i = t0 + tid;
      for (; i + (U - 1) * kCountBlock < t1; i += U * kCountBlock) {
        Bits k[U];
#pragma unroll
        for (int u = 0; u < U; ++u) k[u] = keys[i + u * kCountBlock];
#pragma unroll
        for (int u = 0; u < U; ++u) lds_count_wave(my, digit(k[u]));
      }
      for (; i < t1; i += kCountBlock) lds_count_wave(my, digit(keys[i]));
    };
    if (by_sample)
      count(std::integral_constant<int, 4>{}, [&](Bits x) { return sample_digit<KT>(x, bounds); });
    else
      count(std::integral_constant<int, 8>{}, [&](Bits x) { return step_digit<KT>(x, st); });
    __syncthreads();
    if (tid < kRadix) {
      uint32_t s = 0;
#pragma unroll
      for (int q = 0; q < kCountBlock / 128; ++q) s += h[q][tid];
      rows[(size_t)g * kRadix + tid] = s;
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// chunk (calls with segments of more than kChunkFrom tiles): the tiles of one
// node whose numbers agree but for the last kChunkBits are a chunk, number
// (tile >> kChunkBits) + node, which no other one has; a node's chunks follow
// one another.  A workgroup per kChunk tiles turns their counts into those of
// the chunk's tiles before, and the scan has a chunk's sums to go through
// instead of every tile's: f32, one segment of 2^26, 1128 -> 846 us (chunk 8 us,
// scan 9); u64 + u32, 2^27, 4.35 -> 3.82 ms.  Shorter segments leave it out: a
// launch more for every level, and nothing gained at 512 tiles.  (Prefixes
// kept by the count itself made that 3% slower for calls of many segments.)
// ---------------------------------------------------------------------------
constexpr int kChunkBits = 6;
constexpr uint32_t kChunk = 1u << kChunkBits;
constexpr uint32_t kChunkFrom = 1024;

__global__ __launch_bounds__(kRadix) void seg_chunk_kernel(const Node* __restrict__ nodes, uint32_t* __restrict__ rows,
                                                           uint32_t* __restrict__ chunks,
                                                           const SegCtl* __restrict__ ctl, int level) {
  const uint32_t n_nodes = (uint32_t)(ctl->alloc[level] >> 32), n_tiles = (uint32_t)ctl->alloc[level];
  const int d = threadIdx.x;
  for (uint32_t c = blockIdx.x; c < (n_tiles + kChunk - 1) / kChunk; c += gridDim.x) {
    const uint32_t g1 = min(n_tiles, (c + 1) * kChunk);
    uint32_t g = c * kChunk, ni = find_node(nodes, n_nodes, g);
    while (g < g1) {  // the tiles of one node
      const uint32_t e = ni + 1 < n_nodes ? min(g1, nodes[ni + 1].tile0) : g1;
      uint32_t sum = 0;
      for (; g + 8 <= e; g += 8) {
        uint32_t x[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) x[u] = rows[(size_t)(g + u) * kRadix + d];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          rows[(size_t)(g + u) * kRadix + d] = sum;
          sum += x[u];
        }
      }
      for (; g < e; ++g) {
        const uint32_t x = rows[(size_t)g * kRadix + d];
        rows[(size_t)g * kRadix + d] = sum;
        sum += x;
      }
      chunks[((size_t)c + ni) * kRadix + d] = sum;
      ++ni;
    }
  }
}

// ---------------------------------------------------------------------------
// scan: one workgroup of PARTS * 256 threads per node; thread (q, d) has
// digit d of the q-th part of the node's tiles, or of its chunks where the
// call has these.  The counts become the offsets inside the node of each
// tile's or chunk's digits.  Then the first 256 threads dispose of the
// children.  PARTS = 4 for the first level, whose segments have up to
// hundreds of tiles, 1 for the later ones, whose nodes are many and short.
// ---------------------------------------------------------------------------
template <int PARTS>
__global__ __launch_bounds__(PARTS * kRadix) void seg_scan_kernel(Node* __restrict__ nodes,
                                                                  uint32_t* __restrict__ rows,
                                                                  uint32_t* __restrict__ chunks, uint32_t tile,
                                                                  uint32_t cap, uint32_t src, uint32_t dst, int last,
                                                                  Node* __restrict__ next, uint4* __restrict__ batches,
                                                                  uint4* __restrict__ longs, SegCtl* __restrict__ ctl,
                                                                  int level) {
  __shared__ uint32_t part[PARTS][kRadix];
  __shared__ uint32_t s_off[kRadix + 1], s_step[kRadix];
  __shared__ uint32_t sums[4], sums2[4], sums3[4];
  __shared__ uint64_t s_own[kRadix / kWave], s_cut[kRadix / kWave], s_equal[kRadix / kWave];
  __shared__ uint32_t s_first[kRadix], s_src;
  __shared__ uint32_t s_max, s_batch, s_long;
  __shared__ uint64_t s_next;
  const int tid = threadIdx.x, q = tid / kRadix, d = tid & (kRadix - 1), lane = tid & (kWave - 1);
  const uint32_t n_nodes = (uint32_t)(ctl->alloc[level] >> 32);
  for (uint32_t ni = blockIdx.x; ni < n_nodes; ni += gridDim.x) {
    const Node nd = nodes[ni];
    uint32_t nt = (nd.len + tile - 1) / tile;
    uint32_t* col = rows + (size_t)nd.tile0 * kRadix + d;
    if (chunks != nullptr) {
      const uint32_t c0 = nd.tile0 >> kChunkBits;
      nt = ((nd.tile0 + nt - 1) >> kChunkBits) - c0 + 1;
      col = chunks + ((size_t)c0 + ni) * kRadix + d;
    }
    const uint32_t a = (uint32_t)((uint64_t)nt * q / PARTS), b = (uint32_t)((uint64_t)nt * (q + 1) / PARTS);
    uint32_t sum = 0, t = a;
    for (; t + 8 <= b; t += 8) {
      uint32_t c[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) c[u] = col[(size_t)(t + u) * kRadix];
#pragma unroll
      for (int u = 0; u < 8; ++u) sum += c[u];
    }
    for (; t < b; ++t) sum += col[(size_t)t * kRadix];
    part[q][d] = sum;
    if (tid == 0) s_max = 0;
    __syncthreads();
    uint32_t cnt = 0;
#pragma unroll
    for (int i = 0; i < PARTS; ++i) cnt += part[i][d];
    const uint32_t excl = block_excl_scan_256(tid < kRadix ? cnt : 0u, sums, tid);
    if (tid < kRadix) s_off[d] = excl;
    if (tid == 0) s_off[kRadix] = nd.len;
    // Children longer than the cap are done if every key is the same (equal: a
    // digit of one value; one that is all of the node stays where it is and the
    // scatter skips the node) or split again (big).  The others are batched where
    // floor(offset / T) agrees, T = cap - (the largest of them up to cap / 2; a
    // longer one is a batch by itself), so that a batch fits the cap.
    const bool child = tid < kRadix && cnt > 0;
    const bool over = child && cnt > cap;
    const bool equal = over && (nd.shift == kBySample ? ((nodes[ni].same[d / kWave] >> lane) & 1u) != 0
                                                      : nd.mul == 0 && d >= 1 && d <= 254);
    const bool big = over && !equal;
    const bool own = over || (child && cnt > cap / 2);  // not batched with others
    if (tid < kRadix) {
      const uint64_t m = ballot64(own);
      if (lane == 0) s_own[d / kWave] = m;
      if (child && !own) atomicMax(&s_max, cnt);
    }
    __syncthreads();
    {
      uint32_t run = s_off[d];
      for (int i = 0; i < q; ++i) run += part[i][d];
      for (t = a; t + 8 <= b; t += 8) {
        uint32_t c[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) c[u] = col[(size_t)(t + u) * kRadix];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          col[(size_t)(t + u) * kRadix] = run;
          run += c[u];
        }
      }
      for (; t < b; ++t) {
        const uint32_t c = col[(size_t)t * kRadix];
        col[(size_t)t * kRadix] = run;
        run += c;
      }
    }
    const uint32_t T = cap - s_max;
    const uint32_t step = excl / T;
    if (tid < kRadix) s_step[d] = step;
    __syncthreads();
    // a batch starts at every child of its own, behind it, and where the step
    // changes; it ends where the next one starts
    bool cut = false;
    if (tid < kRadix) {
      cut = d == 0 || own || ((s_own[(d - 1) / kWave] >> ((d - 1) & (kWave - 1))) & 1u) || s_step[d - 1] != step;
      const uint64_t m = ballot64(cut);
      if (lane == 0) s_cut[d / kWave] = m;
    }
    __syncthreads();
    uint32_t end = kRadix;
    if (cut) {
      uint64_t m = s_cut[d / kWave] >> 1 >> lane;
      if (m) {
        end = d + 1 + (uint32_t)__builtin_ctzll(m);
      } else {
        for (int i = d / kWave + 1; i < kRadix / kWave; ++i)
          if (s_cut[i]) {
            end = i * kWave + (uint32_t)__builtin_ctzll(s_cut[i]);
            break;
          }
      }
    }
    const uint32_t len = cut ? s_off[end] - excl : 0u;
    // batches of the local sort; an equal child that is not in the output is
    // cut into caps to be copied there
    const bool stays = equal && cnt == nd.len;
    if (stays) nodes[ni].shift = kDone;
    const uint32_t at = stays ? src : dst;
    uint32_t nb = cut && len > 0 && !over ? 1u : 0u;
    if (equal && at != kSrcOut) nb = (cnt + cap - 1) / cap;
    const uint32_t bigs = big ? 1u : 0u, bigt = big && !last ? (cnt + tile - 1) / tile : 0u;
    const uint32_t eb = block_excl_scan_256(nb, sums, tid);
    const uint32_t en = block_excl_scan_256(bigs, sums2, tid);
    const uint32_t et = block_excl_scan_256(bigt, sums3, tid);
    if (tid < kRadix) {
      const uint64_t m = ballot64(equal && nb > 0);
      if (lane == 0) s_equal[d / kWave] = m;
      s_first[d] = eb;
      if (equal && nb > 0) s_src = at;  // (one that stays is the node's only child)
    }
    if (tid == kRadix - 1) {
      if (eb + nb) s_batch = atomicAdd(&ctl->n_batches, eb + nb);
      if (en + bigs) {
        if (last)
          s_long = atomicAdd(&ctl->n_long, en + bigs);
        else
          s_next = atomicAdd(reinterpret_cast<unsigned long long*>(&ctl->alloc[level + 1]),
                             (unsigned long long)(en + bigs) << 32 | (et + bigt));
      }
    }
    __syncthreads();
    if (big) {
      if (last)
        longs[s_long + en] = make_uint4(nd.seg, nd.off + excl, cnt, dst);
      else
        next[(uint32_t)(s_next >> 32) + en] = Node{nd.seg, nd.off + excl, cnt, (uint32_t)s_next + et, 0, 0, 0, 0, {}};
    } else if (nb && !equal) {
      batches[s_batch + eb] = make_uint4(nd.seg, nd.off + excl, len, dst);
    }
    for (int g = 0; g < kRadix / kWave; ++g) {  // equal children may have thousands: the whole block writes each one's
      for (uint64_t m = s_equal[g]; m != 0; m &= m - 1) {
        const uint32_t c = g * kWave + (uint32_t)__builtin_ctzll(m), o = s_off[c], n = s_off[c + 1] - o;
        for (uint32_t i = tid; i * cap < n; i += PARTS * kRadix)
          batches[s_batch + s_first[c] + i] = make_uint4(nd.seg, nd.off + o + i * cap, min(cap, n - i * cap), s_src);
      }
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// scatter: a workgroup takes tiles of its XCD's part of the level: ranks its
// records by digit in LDS, stages them in digit order and writes every digit's
// run to the tile's offset.  Bound by HBM: one read and one write of
// every record.
// ---------------------------------------------------------------------------
template <int KT, typename V, int BLOCK, int IPT, int WAVES>
__global__ __launch_bounds__(BLOCK, WAVES) void seg_scatter_kernel(
    const typename Codec<KT>::Bits* __restrict__ src, const V* __restrict__ vsrc, typename Codec<KT>::Bits* __restrict__ dst,
    V* __restrict__ vdst, const uint64_t* __restrict__ sp, const uint64_t* __restrict__ svp,
    const uint64_t* __restrict__ dp, const uint64_t* __restrict__ dvp, const Node* __restrict__ nodes,
    const uint32_t* __restrict__ rows, const uint32_t* __restrict__ chunks, const SegCtl* __restrict__ ctl, int level) {
  using Bits = typename Codec<KT>::Bits;
  constexpr int W = BLOCK / kWave;
  constexpr int TILE = BLOCK * IPT;
  constexpr bool HV = kHasVal<V>;
  using VS = typename std::conditional<HV, V, uint32_t>::type;
  __shared__ Bits keys[TILE];
  __shared__ VS vstage[HV ? TILE : 1];
  __shared__ uint32_t off[W][kRadix];
  __shared__ uint32_t gbase[kRadix];
  __shared__ uint32_t sums[4];
  __shared__ Bits bounds[kRadix];
  __shared__ uint8_t dstage[TILE];  // digits between samples: a search is too long to repeat
  uint32_t bounds_of = 0xFFFFFFFFu;  // the node whose sample they are
  const uint32_t n_nodes = (uint32_t)(ctl->alloc[level] >> 32), n_tiles = (uint32_t)ctl->alloc[level];
  const int tid = threadIdx.x, lane = tid & (kWave - 1), w = (int)readfirstlane((uint32_t)(tid / kWave));
  for (int i = lane; i < kRadix; i += kWave) off[w][i] = 0;
  // Workgroups b, b + 8, ... run on one XCD: its eighth of the tiles is one
  // stretch, so that the ends of neighbouring tiles' runs meet in one L2.
  const uint32_t groups = min(kXcds, gridDim.x), x = blockIdx.x % groups, j0 = blockIdx.x / groups;
  const uint32_t stride = (gridDim.x - x + groups - 1) / groups;
  const uint32_t first = (uint32_t)((uint64_t)n_tiles * x / groups), stop = (uint32_t)((uint64_t)n_tiles * (x + 1) / groups);
  for (uint32_t g = first + j0; g < stop; g += stride) {
    const uint32_t ni = find_node(nodes, n_nodes, g);
    const Node nd = nodes[ni];
    if (nd.shift == kDone) continue;
    const bool by_sample = nd.shift == kBySample;
    const Steps<Bits> st{(Bits)nd.base, (Bits)nd.top, nd.mul, by_sample ? 0u : nd.shift};
    if (by_sample && bounds_of != ni) {  // the sample anew (the count's would take 2 KB of scratch per node)
      static_assert(TILE * sizeof(Bits) >= kRadix * (sizeof(Bits) + sizeof(uint32_t)), "sort_sample's working space");
      sort_sample<KT, BLOCK>(src + sp[nd.seg] + nd.off, nd.len, keys, reinterpret_cast<uint32_t*>(keys + kRadix), bounds);
      sample_bounds<Bits>(bounds);
      bounds_of = ni;
    }
    const uint32_t t0 = (g - nd.tile0) * (uint32_t)TILE;
    const uint32_t cnt = min((uint32_t)TILE, nd.len - t0);
    const bool full = cnt == (uint32_t)TILE;
    const Bits* in = src + sp[nd.seg] + nd.off + t0;
    const uint32_t wb = (uint32_t)(w * IPT * kWave + lane);
    uint32_t row = tid < kRadix ? rows[(size_t)g * kRadix + tid] : 0u;
    if (chunks != nullptr && tid < kRadix) row += chunks[((size_t)(g >> kChunkBits) + ni) * kRadix + tid];
    Bits k[IPT];
    VS v[IPT];
    if (full) {
      static_for<IPT>([&](auto i) { k[i] = in[wb + i * kWave]; });
    } else {
      static_for<IPT>([&](auto i) { k[i] = wb + i * kWave < cnt ? in[wb + i * kWave] : Bits(0); });
    }
    if constexpr (HV) {
      const V* vin = vsrc + svp[nd.seg] + nd.off + t0;
      if (full) {
        static_for<IPT>([&](auto i) { v[i] = vin[wb + i * kWave]; });
      } else {
        static_for<IPT>([&](auto i) { v[i] = wb + i * kWave < cnt ? vin[wb + i * kWave] : VS(0); });
      }
    }
    uint32_t r[IPT];  // digit << 16 | place among the wavefront's of this digit
    static_assert(TILE <= 65536, "a place takes 16 bits");
    uint32_t* const ct = off[w];
    if (by_sample) {
      static_for<IPT>([&](auto i) {
        r[i] = sample_digit<KT>(k[i], bounds);
        if constexpr (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // (more searches at once spill)
      });
    } else {
      static_for<IPT>([&](auto i) { r[i] = step_digit<KT>(k[i], st); });
    }
    if (full) {
      if (__popcll(ballot64(r[0] == readfirstlane(r[0]))) >= 16) {
        static_for<IPT>([&](auto i) { r[i] = r[i] << 16 | rank_wave_atomic<true>(r[i], ct); });
      } else {
        static_for<IPT>([&](auto i) { r[i] = r[i] << 16 | rank_wave_atomic<false>(r[i], ct); });
      }
    } else {
      static_for<IPT>([&](auto i) {
        if (wb + i * kWave < cnt) r[i] = r[i] << 16 | rank_wave_atomic<true>(r[i], ct);
        else r[i] = 0;
      });
    }
    __syncthreads();
    uint32_t total = 0;
    if (tid < kRadix) {
#pragma unroll
      for (int i = 0; i < W; ++i) total += off[i][tid];
    }
    const uint32_t excl = block_excl_scan_256(total, sums, tid);
    if (tid < kRadix) {
      uint32_t run = excl;
#pragma unroll
      for (int i = 0; i < W; ++i) {
        const uint32_t c = off[i][tid];
        off[i][tid] = run;
        run += c;
      }
      gbase[tid] = row - excl;
    }
    __syncthreads();
    if (by_sample) {
      static_for<IPT>([&](auto i) {
        if (full || wb + i * kWave < cnt) dstage[(r[i] & 0xFFFFu) + ct[r[i] >> 16]] = (uint8_t)(r[i] >> 16);
      });
    }
    static_for<IPT>([&](auto i) { r[i] = (r[i] & 0xFFFFu) + ct[r[i] >> 16]; });
    static_for<IPT>([&](auto i) {
      if (full || wb + i * kWave < cnt) {
        keys[r[i]] = k[i];
        if constexpr (HV) vstage[r[i]] = v[i];
      }
    });
    for (int i = lane; i < kRadix; i += kWave) off[w][i] = 0;
    __syncthreads();
    // a corrupted offset stays inside the node
    const uint32_t top = nd.len - 1;
    Bits* const ko = dst + dp[nd.seg] + nd.off;
    V* vo = nullptr;
    if constexpr (HV) vo = vdst + dvp[nd.seg] + nd.off;
    auto write = [&](int j, auto digit) {
      const uint32_t i = (uint32_t)(j * BLOCK + tid);
      if (full || i < cnt) {
        const Bits kk = keys[i];
        const uint32_t o = min(gbase[digit(kk, i)] + i, top);
        ko[o] = kk;
        if constexpr (HV) vo[o] = vstage[i];
      }
    };
    if (by_sample) {
#pragma unroll 4
      for (int j = 0; j < IPT; ++j) write(j, [&](Bits, uint32_t i) { return (uint32_t)dstage[i]; });
    } else {
#pragma unroll
      for (int j = 0; j < IPT; ++j) write(j, [&](Bits x, uint32_t) { return step_digit<KT>(x, st); });
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// local: workgroup b sorts the batches b, b + B, ... in LDS
// ---------------------------------------------------------------------------
template <int KT, typename V, int BLOCK, int IPT, int WAVES>
__global__ __launch_bounds__(BLOCK, WAVES) void seg_local_kernel(const typename Codec<KT>::Bits* k_in,
                                                                 const typename Codec<KT>::Bits* k_alt,
                                                                 typename Codec<KT>::Bits* k_out, const V* v_in,
                                                                 const V* v_alt, V* v_out, SegTab tab,
                                                                 const uint4* __restrict__ batches,
                                                                 const SegCtl* __restrict__ ctl) {
  using Bits = typename Codec<KT>::Bits;
  using Smem = BlockSortSmem<Bits, V, BLOCK, IPT>;
  using VS = typename Smem::VS;
  __shared__ Smem sm;
  const uint32_t total = ctl->n_batches;
  block_clear_row<BLOCK>(sm.off);
  for (uint32_t bi = blockIdx.x; bi < total; bi += gridDim.x) {
    const uint4 e = batches[bi];
    const uint32_t m = readfirstlane(e.z);
    if (m == 0) continue;
    const uint64_t ob = tab.begin[e.x] + e.y;
    const uint64_t ab = tab.alt[e.x] + e.y;
    const Bits* kb = e.w == kSrcIn ? k_in + ob : e.w == kSrcAlt ? k_alt + ab : k_out + ob;
    const uint32_t nit = block_items<BLOCK>(m), wb = block_first<BLOCK>(nit);
    Bits k[IPT];
    VS v[IPT];
    static_for<IPT>([&](auto i) {
      k[i] = 0;
      if (wb + i * kWave < m && (uint32_t)i < nit) k[i] = kb[wb + i * kWave];
    });
    V* vo = nullptr;
    if constexpr (kHasVal<V>) {
      const uint64_t vb = tab.vbegin[e.x] + e.y;
      const V* vs = e.w == kSrcIn ? v_in + vb : e.w == kSrcAlt ? v_alt + ab : v_out + vb;
      vo = v_out + vb;
      static_for<IPT>([&](auto i) {
        v[i] = 0;
        if (wb + i * kWave < m && (uint32_t)i < nit) v[i] = vs[wb + i * kWave];
      });
    }
    Bits mn, mx;
    block_min_max<KT, V, BLOCK, IPT>(sm, k, wb, m, nit, mn, mx);
    const Bits pad = Codec<KT>::dec(mx);
    static_for<IPT>([&](auto i) { k[i] = wb + i * kWave < m ? k[i] : pad; });
    block_sort<KT, V, BLOCK, IPT>(sm, k, v, m, mn, mx, k_out + ob, vo);
    __syncthreads();
  }
}

constexpr size_t kAlign = 256;
inline size_t align_up(size_t x) { return (x + kAlign - 1) / kAlign * kAlign; }

struct SegLayout {
  size_t ctl, alt_k, alt_v, tab_begin, tab_vbegin, tab_alt, nodes[kMaxLevels], batches, longs, rows, chunks, total;
  uint32_t nodes_ub[kMaxLevels], tiles_ub[kMaxLevels], batches_ub;
  int levels;
};

// Tile geometries of the scatter, chosen per call by
// mgs_tuning::large_variant (0 = the default; the autotuner times all of
// them per record width, payload and size):
//   record   variant 0        variant 1          variant 2
//   4 B      512 x 16         1024 x 18          512 x 8
//   8 B      512 x 20         512 x 28           512 x 12
//   12 B     512 x 20         512 x 16           512 x 12
//   16 B     512 x 14         512 x 12           512 x 8
// (threads x items per thread).  Variant 0: 16 items per thread for 4-byte
// keys (four workgroups per CU); wider records use the LDS of a whole CU, as
// the plain sort's large tiles do.  Variant 1 of the 4-byte keys is the
// plain sort's tile; the others trade tile size for occupancy.
constexpr int kSegVariants = 3;
template <int KB, int VB, int VAR>
struct SegLargeGeom {
  static constexpr int kRec = KB + VB;
  static constexpr int kBlock = (kRec <= 4 && VAR == 1) ? 1024 : 512;
  static constexpr int kIpt = kRec <= 4    ? (VAR == 0 ? 16 : VAR == 1 ? 18 : 8)
                              : kRec <= 8  ? (VAR == 0 ? 20 : VAR == 1 ? 28 : 12)
                              : kRec <= 12 ? (VAR == 0 ? 20 : VAR == 1 ? 16 : 12)
                                           : (VAR == 0 ? 14 : VAR == 1 ? 12 : 8);
  static constexpr int kTile = kBlock * kIpt;
  // wavefronts per SIMD: 1024-thread workgroups and tiles that leave the LDS
  // to a second workgroup run four, the others two
  static constexpr int kWaves = kBlock == 1024 || kTile * kRec <= 66 * 1024 ? 4 : 2;
};

template <int KB, int VB>
inline int seg_large_tile(int var) {
  switch (var) {
    case 1: return SegLargeGeom<KB, VB, 1>::kTile;
    case 2: return SegLargeGeom<KB, VB, 2>::kTile;
    default: return SegLargeGeom<KB, VB, 0>::kTile;
  }
}

template <int KB, int VB>
struct SegCfg {
  // one workgroup per long range streams it through tiles of this size
  using M = TileCfg<KB, VB, 16, 8, 8, 4, 4, MGS_OS_BLOCK>;
  // local sort: 512 threads, three workgroups per CU for 4-byte records, two
  // for wider ones: as many items as leave none in scratch registers at that
  // occupancy
  static constexpr int kRec = KB + VB;
  static constexpr int kLocalBlock = 512;
  static constexpr int kLocalIpt = kRec <= 4 ? 16 : kRec <= 8 ? 14 : kRec <= 12 ? 10 : 7;
  static constexpr int kLocalWaves = kRec <= 4 ? 6 : 4;
  static constexpr uint32_t kCap = (uint32_t)kLocalBlock * kLocalIpt;
};

// Nodes of the first level hold more than kMinSplit records, whatever the
// tuning, so the scratch size depends only on the sizes and the variant.
constexpr uint32_t kMinSplit = 256;

// wide_range: doubles.
template <int KB, int VB>
SegLayout seg_layout(size_t max_total, size_t nseg, size_t max_seg, int large_tile, bool wide_range) {
  constexpr size_t cap = SegCfg<KB, VB>::kCap;
  SegLayout L{};
  // Levels of splitting: two reach the cap for segments up to 2^20 records;
  // longer ones get a third, and so do doubles from 2^15 on: their encoded range
  // around zero spans 2000 exponents, and equal steps may take a level
  // to part these.
  L.levels = max_seg > (wide_range ? size_t(1) << 15 : size_t(1) << 20) ? 3 : 2;
  // a batch that a node's children form holds more than cap / 2 records on
  // average but for one per node and the breaks at children above cap / 2
  // (at most two per such child); equal children are cut into caps
  size_t nodes = 0;
  for (int l = 0; l < L.levels; ++l) {
    L.nodes_ub[l] = (uint32_t)(l == 0 ? std::min<size_t>(nseg, max_total / (kMinSplit + 1) + 1) : max_total / (cap + 1) + 1);
    L.tiles_ub[l] = (uint32_t)(max_total / (size_t)large_tile + L.nodes_ub[l] + 1);
    nodes += L.nodes_ub[l];
  }
  const size_t per_level = 8 * (max_total / cap + 1);
  L.batches_ub = (uint32_t)(nseg + 2 * nodes + L.levels * per_level);
  size_t o = 0;
  auto take = [&](size_t bytes) {
    const size_t at = o;
    o = align_up(o + bytes);
    return at;
  };
  L.ctl = take(sizeof(SegCtl));  // first: its status word is the call's status word
  L.alt_k = take(max_total * KB);
  L.alt_v = take(max_total * VB);
  L.tab_begin = take(nseg * 8);
  L.tab_vbegin = take(nseg * 8);
  L.tab_alt = take(nseg * 8);
  uint32_t tiles = 0;
  for (int l = 0; l < L.levels; ++l) {
    L.nodes[l] = take((size_t)L.nodes_ub[l] * sizeof(Node));
    tiles = std::max(tiles, L.tiles_ub[l]);
  }
  L.batches = take((size_t)L.batches_ub * 16);
  L.longs = take((max_total / (cap + 1) + 1) * 16);
  L.rows = take((size_t)tiles * kRadix * 4);
  if (max_seg / large_tile > kChunkFrom)
    L.chunks = take(((size_t)tiles / kChunk + 1 + std::max(L.nodes_ub[0], L.nodes_ub[1])) * kRadix * 4);
  L.total = o;
  return L;
}

// Longest segment the call accepts: the caller's hint (mgs_tuning::
// max_segment_keys) or max_total.  Longer segments are left unsorted and
// reported in the status word.
inline size_t segment_bound(size_t max_total, const mgs_tuning* tuning) {
  if (tuning != nullptr && tuning->max_segment_keys > 0)
    return std::min<size_t>(max_total, (size_t)tuning->max_segment_keys);
  return max_total;
}

inline int large_variant_of(const mgs_tuning* tuning) { return tuning != nullptr ? tuning->large_variant : 0; }

template <int KT, int VT>
int seg_typed(const void* kin, void* kout, const void* vin, void* vout, const uint64_t* bounds, bool ranges,
              const uint64_t* val_begin, size_t nseg, size_t max_total, const mgs_tuning* tuning, void* temp, size_t temp_bytes, hipStream_t s) {
  using Bits = typename Codec<KT>::Bits;
  using V = typename ValOf<VT>::T;
  constexpr int KB = sizeof(Bits);
  constexpr int VB = kValBytes<V>;
  using C = SegCfg<KB, VB>;
  using VP = typename std::conditional<kHasVal<V>, V, uint32_t>::type;

  // the longest segment that one workgroup sorts: the larger of the caller's
  // two single-workgroup limits, as many as fit its LDS by default
  uint32_t small_max = C::kCap;
  if (tuning && tuning->small_max > 0 && tuning->medium_max > 0)
    small_max = std::min<uint32_t>((uint32_t)std::max(tuning->small_max, tuning->medium_max), C::kCap);
  small_max = std::max(small_max, kMinSplit);
  const size_t max_seg = segment_bound(max_total, tuning);
  const int var = large_variant_of(tuning);
  if (var < 0 || var >= kSegVariants) return MGS_ERR_INVALID;
  const uint32_t tile = (uint32_t)seg_large_tile<KB, VB>(var);
  const SegLayout L = seg_layout<KB, VB>(max_total, nseg, max_seg, (int)tile, KT == MGS_KEY_F64);
  if (temp == nullptr || temp_bytes < L.total) return MGS_ERR_TEMP_TOO_SMALL;
  char* t = static_cast<char*>(temp);
  Bits* ka = reinterpret_cast<Bits*>(t + L.alt_k);
  V* va = reinterpret_cast<V*>(reinterpret_cast<VP*>(t + L.alt_v));
  SegCtl* ctl = reinterpret_cast<SegCtl*>(t + L.ctl);
  uint4* batches = reinterpret_cast<uint4*>(t + L.batches);
  uint4* longs = reinterpret_cast<uint4*>(t + L.longs);
  uint32_t* rows = reinterpret_cast<uint32_t*>(t + L.rows);
  uint32_t* chunks = max_seg / tile > kChunkFrom ? reinterpret_cast<uint32_t*>(t + L.chunks) : nullptr;
  Node* nodes[kMaxLevels];
  for (int l = 0; l < L.levels; ++l) nodes[l] = reinterpret_cast<Node*>(t + L.nodes[l]);
  const SegTab tab{reinterpret_cast<uint64_t*>(t + L.tab_begin), reinterpret_cast<uint64_t*>(t + L.tab_vbegin),
                   reinterpret_cast<uint64_t*>(t + L.tab_alt)};
  const Bits* ki = static_cast<const Bits*>(kin);
  Bits* ko = static_cast<Bits*>(kout);
  const V* vi = static_cast<const V*>(vin);
  V* vo = static_cast<V*>(vout);

  // (no bounds: one array, of more records than one workgroup sorts)
  const uint32_t whole = bounds == nullptr ? (uint32_t)max_total : 0u;
  if (bounds == nullptr && max_total <= small_max) return MGS_ERR_INVALID;
  if (bounds != nullptr && ranges)
    seg_classify_kernel<true><<<1, kClassifyBlock, 0, s>>>(bounds, val_begin, (uint32_t)nseg, max_total, max_seg,
                                                           small_max, tile, tab, batches, nodes[0], ctl);
  else if (bounds != nullptr)
    seg_classify_kernel<false><<<1, kClassifyBlock, 0, s>>>(bounds, val_begin, (uint32_t)nseg, max_total, max_seg,
                                                            small_max, tile, tab, batches, nodes[0], ctl);
  // level l reads the input, the scratch, the output and writes the scratch,
  // the output, the scratch
  auto level = [&](int l, auto scatter, int block) {
    const bool from_alt = l == 1, to_alt = l != 1;
    const Bits* ks = l == 0 ? ki : from_alt ? ka : ko;
    const V* vs = l == 0 ? vi : from_alt ? va : vo;
    const uint64_t* sp = from_alt ? tab.alt : tab.begin;
    const uint64_t* svp = from_alt ? tab.alt : tab.vbegin;
    const uint64_t* dp = to_alt ? tab.alt : tab.begin;
    const uint64_t* dvp = to_alt ? tab.alt : tab.vbegin;
    auto count = seg_count_kernel<KT>;
    count<<<std::min(L.tiles_ub[l], resident_blocks(count, kCountBlock)), kCountBlock, 0, s>>>(
        ks, tab, sp, nodes[l], rows, tile, C::kCap, ctl, l, L.levels - l, l == 0 ? whole : 0u);
    if (chunks != nullptr)
      seg_chunk_kernel<<<std::min(L.tiles_ub[l] / kChunk + 1, 2048u), kRadix, 0, s>>>(nodes[l], rows, chunks, ctl, l);
    const bool last = l + 1 == L.levels;
    const uint32_t from = l == 0 ? kSrcIn : from_alt ? kSrcAlt : kSrcOut, to = to_alt ? kSrcAlt : kSrcOut;
    if (l == 0)
      seg_scan_kernel<4><<<std::min(L.nodes_ub[l], 512u), 4 * kRadix, 0, s>>>(nodes[l], rows, chunks, tile, C::kCap, from, to, last ? 1 : 0,
                                                                             last ? nullptr : nodes[l + 1], batches,
                                                                             longs, ctl, l);
    else
      seg_scan_kernel<1><<<std::min(L.nodes_ub[l], 2048u), kRadix, 0, s>>>(nodes[l], rows, chunks, tile, C::kCap, from, to, last ? 1 : 0,
                                                                         last ? nullptr : nodes[l + 1], batches, longs,
                                                                         ctl, l);
    scatter<<<std::min(L.tiles_ub[l], resident_blocks(scatter, block)), block, 0, s>>>(
        ks, vs, to_alt ? ka : ko, to_alt ? va : vo, sp, svp, dp, dvp, nodes[l], rows, chunks, ctl, l);
  };
  if (max_seg > small_max) {
    for (int l = 0; l < L.levels; ++l) {
      switch (var) {
        case 1: {
          using G = SegLargeGeom<KB, VB, 1>;
          level(l, seg_scatter_kernel<KT, V, G::kBlock, G::kIpt, G::kWaves>, G::kBlock);
          break;
        }
        case 2: {
          using G = SegLargeGeom<KB, VB, 2>;
          level(l, seg_scatter_kernel<KT, V, G::kBlock, G::kIpt, G::kWaves>, G::kBlock);
          break;
        }
        default: {
          using G = SegLargeGeom<KB, VB, 0>;
          level(l, seg_scatter_kernel<KT, V, G::kBlock, G::kIpt, G::kWaves>, G::kBlock);
        }
      }
    }
    using MC = typename C::M;
    auto lng = seg_long_kernel<KT, V, MC::kBlock, MC::kIpt>;
    lng<<<std::min<uint32_t>((uint32_t)(max_total / (C::kCap + 1) + 1), resident_blocks(lng, MC::kBlock)), MC::kBlock, 0, s>>>(
        ka, ko, va, vo, tab, longs, ctl);
  }
  auto local = seg_local_kernel<KT, V, C::kLocalBlock, C::kLocalIpt, C::kLocalWaves>;
  local<<<std::min(L.batches_ub, resident_blocks(local, C::kLocalBlock)), C::kLocalBlock, 0, s>>>(ki, ka, ko, vi, va, vo, tab,
                                                                                           batches, ctl);
  return check_launch();
}

template <int KT>
int seg_by_val(mgs_val vt, const void* kin, void* kout, const void* vin, void* vout, const uint64_t* offsets,
               bool ranges, const uint64_t* val_begin, size_t nseg, size_t max_total, const mgs_tuning* tuning, void* temp, size_t temp_bytes,
               hipStream_t s) {
  switch (vt) {
    case MGS_VAL_NONE:
      return seg_typed<KT, MGS_VAL_NONE>(kin, kout, vin, vout, offsets, ranges, val_begin, nseg, max_total, tuning, temp,
                                                 temp_bytes, s);
    case MGS_VAL_U32:
      return seg_typed<KT, MGS_VAL_U32>(kin, kout, vin, vout, offsets, ranges, val_begin, nseg, max_total, tuning, temp,
                                                 temp_bytes, s);
    case MGS_VAL_U64:
      return seg_typed<KT, MGS_VAL_U64>(kin, kout, vin, vout, offsets, ranges, val_begin, nseg, max_total, tuning, temp,
                                                 temp_bytes, s);
  }
  return MGS_ERR_BAD_TYPE;
}

template <int KB, int VB>
size_t seg_bytes(size_t max_total, size_t nseg, size_t max_seg, int var, bool wide_range = false) {
  if (var < 0 || var >= kSegVariants) var = 0;
  return seg_layout<KB, VB>(max_total, nseg, max_seg, seg_large_tile<KB, VB>(var), wide_range).total;
}

template <int KB, int VB>
void seg_geom(int var, int32_t* block, int32_t* ipt) {
  switch (var) {
    case 1:
      *block = SegLargeGeom<KB, VB, 1>::kBlock;
      *ipt = SegLargeGeom<KB, VB, 1>::kIpt;
      break;
    case 2:
      *block = SegLargeGeom<KB, VB, 2>::kBlock;
      *ipt = SegLargeGeom<KB, VB, 2>::kIpt;
      break;
    default:
      *block = SegLargeGeom<KB, VB, 0>::kBlock;
      *ipt = SegLargeGeom<KB, VB, 0>::kIpt;
  }
}

}  // namespace

size_t segmented_temp_bytes(mgs_key kt, mgs_val vt, size_t max_total, size_t nseg, const mgs_tuning* tuning) {
  const int kb = key_bytes(kt), vb = val_bytes(vt);
  if (kb < 0 || vb < 0) return 0;
  const size_t ms = segment_bound(max_total, tuning);
  const int var = large_variant_of(tuning);
  if (kb == 4) {
    if (vb == 0) return seg_bytes<4, 0>(max_total, nseg, ms, var);
    if (vb == 4) return seg_bytes<4, 4>(max_total, nseg, ms, var);
    return seg_bytes<4, 8>(max_total, nseg, ms, var);
  }
  if (vb == 0) return seg_bytes<8, 0>(max_total, nseg, ms, var, kt == MGS_KEY_F64);
  if (vb == 4) return seg_bytes<8, 4>(max_total, nseg, ms, var, kt == MGS_KEY_F64);
  return seg_bytes<8, 8>(max_total, nseg, ms, var, kt == MGS_KEY_F64);
}

int segmented_variant(mgs_key kt, mgs_val vt, int var, int32_t* block, int32_t* ipt) {
  const int kb = key_bytes(kt), vb = val_bytes(vt);
  if (kb < 0 || vb < 0) return MGS_ERR_BAD_TYPE;
  if (var < 0 || var >= kSegVariants) return MGS_ERR_INVALID;
  int32_t b = 0, i = 0;
  if (kb == 4)
    (vb == 0 ? seg_geom<4, 0> : vb == 4 ? seg_geom<4, 4> : seg_geom<4, 8>)(var, &b, &i);
  else
    (vb == 0 ? seg_geom<8, 0> : vb == 4 ? seg_geom<8, 4> : seg_geom<8, 8>)(var, &b, &i);
  if (block) *block = b;
  if (ipt) *ipt = i;
  return MGS_OK;
}

int segmented_variant_count() { return kSegVariants; }

uint32_t split_local_cap(int kb, int vb) {
  if (kb == 4) return vb == 0 ? SegCfg<4, 0>::kCap : vb == 4 ? SegCfg<4, 4>::kCap : SegCfg<4, 8>::kCap;
  return vb == 0 ? SegCfg<8, 0>::kCap : vb == 4 ? SegCfg<8, 4>::kCap : SegCfg<8, 8>::kCap;
}

size_t split_sort_temp_bytes(mgs_key kt, mgs_val vt, size_t n) { return segmented_temp_bytes(kt, vt, n, 1, nullptr); }

int split_sort(mgs_key kt, mgs_val vt, const void* kin, void* kout, const void* vin, void* vout, size_t n, void* temp,
               size_t temp_bytes, hipStream_t s) {
  return segmented_dispatch(kt, vt, kin, kout, vin, vout, nullptr, false, nullptr, 1, n, nullptr, temp, temp_bytes, s);
}

int segmented_dispatch(mgs_key kt, mgs_val vt, const void* kin, void* kout, const void* vin, void* vout,
                       const uint64_t* d_offsets, bool ranges, const uint64_t* d_val_begin, size_t nseg, size_t max_total, const mgs_tuning* tuning,
                       void* temp, size_t temp_bytes, hipStream_t s) {
  switch (kt) {
    case MGS_KEY_U32:
      return seg_by_val<MGS_KEY_U32>(vt, kin, kout, vin, vout, d_offsets, ranges, d_val_begin, nseg, max_total, tuning, temp, temp_bytes, s);
    case MGS_KEY_U64:
      return seg_by_val<MGS_KEY_U64>(vt, kin, kout, vin, vout, d_offsets, ranges, d_val_begin, nseg, max_total, tuning, temp, temp_bytes, s);
    case MGS_KEY_I32:
      return seg_by_val<MGS_KEY_I32>(vt, kin, kout, vin, vout, d_offsets, ranges, d_val_begin, nseg, max_total, tuning, temp, temp_bytes, s);
    case MGS_KEY_I64:
      return seg_by_val<MGS_KEY_I64>(vt, kin, kout, vin, vout, d_offsets, ranges, d_val_begin, nseg, max_total, tuning, temp, temp_bytes, s);
    case MGS_KEY_F32:
      return seg_by_val<MGS_KEY_F32>(vt, kin, kout, vin, vout, d_offsets, ranges, d_val_begin, nseg, max_total, tuning, temp, temp_bytes, s);
    case MGS_KEY_F64:
      return seg_by_val<MGS_KEY_F64>(vt, kin, kout, vin, vout, d_offsets, ranges, d_val_begin, nseg, max_total, tuning, temp, temp_bytes, s);
  }
  return MGS_ERR_BAD_TYPE;
}

}  // namespace mgs
