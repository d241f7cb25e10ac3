// k-way merge of sorted runs on the device: the GPU counterpart of the
// reference's __gnu_parallel::multiway_merge of sorted chunks
// (src/gowanlock_sort.cuh:91-92), used by the heterogeneous sort's device
// merge backend in one pass instead of log2(k) pairwise merge rounds.
//
// Stable order: the output is the stable sort of the runs laid end to end in
// run order, i.e. the lexicographic order of (enc(key), run, index).
//
//   sample    every S-th key of every run (S = cap / (step + k), step = 3k or
//             5k, at least 8) with its sample id, ids numbered run by run
//   sort      the samples by key, stably (mgs_sort with the ids as payload):
//             (key, run, index) order
//   split     every step-th sorted sample (v, j, i) bounds a piece: run j'
//             contributes the keys that precede (v, j, i) -- upper bound of v
//             for j' < j, lower bound for j' > j, exactly i for j' = j
//   base      each boundary's output position (the sum of its splits)
//   piece     one workgroup per piece: its slices of the k runs, laid end to
//             end in run order, sorted stably in LDS (block_sort.hpp: two or
//             three radix passes whatever k is), which is their stable merge; or,
//             for up to 8 runs of 8-byte keys, merged by a tree of LDS
//             merge-path rounds (adjacent slices, earlier runs first on ties)
//
// A run contributes to a piece only the keys between two of its consecutive
// samples per sample of it inside the piece, plus one more stretch, so a
// piece holds at most (step + k) S <= cap keys and fits the LDS.
//
// One or two runs need no samples: they are mgs_merge's merge path
// (merge.hip), whose tiles cost less than the pieces (2 runs of 2^27 u32
// keys: 0.80 ms as pieces of one merge round, 0.45 ms).
#include <vector>

#include "block_sort.hpp"
#include "common.hpp"
#include "internal.hpp"
#include "radix_sort.hpp"

namespace mgs {

namespace {

// Pieces sorted by radix passes: 8192 4-byte keys in 49 KB of LDS, three
// workgroups of 512 threads per CU; 6144 8-byte keys in 66 KB, two.  The
// passes are bound by the LDS (62% of the cycles, half of these in bank
// conflicts of the random counters and positions), the vector instructions (74%:
// profiles/counters_by_kernel.txt) and by how far other
// workgroups fill the gaps between barriers: 1024-thread workgroups of as
// many keys measured 1.25 times slower, as did 16384 keys per piece.
// Measured, whole call, against the merge tree: u32, 8 runs of 2^26 2.81 ->
// 1.82 ms, 16 x 2^24 2.02 -> 1.13 ms, 64 x 2^22 3.6 -> 1.7 ms, 256 x 2^20
// 6.7 -> 3.2 ms; small merges of few runs were faster by the tree (4 x 2^22 147
// against 161 us).
constexpr int kMwBlock = 512;
template <typename Bits>
struct MwCfg {
  static constexpr int kIpt = sizeof(Bits) == 4 ? 16 : 12;
  static constexpr int kWaves = sizeof(Bits) == 4 ? 6 : 4;
  static constexpr uint32_t kCap = (uint32_t)kMwBlock * kIpt;  // keys per piece at most
};
// Pieces merged by a tree, ceil(log2 k) rounds: 8-byte keys, whose LDS
// traffic per radix pass is about twice that of 4-byte keys, up to 8 runs (4
// runs of 2^24 i64: 0.60 ms against 0.62-0.64 by radix passes; 8 x 2^23 with
// low bits all zero: 0.80 against 0.93-0.97; 16 x 2^22: 0.95 against 0.77,
// and with such keys 0.99 against 1.09).
constexpr int kTreeBlock = 1024;
constexpr uint32_t kTreeCap = 8192;
inline bool tree_pieces(int kb, size_t k) { return kb == 8 && k <= 8; }

inline uint32_t piece_cap(int kb, size_t k) {
  return tree_pieces(kb, k) ? kTreeCap : kb == 4 ? MwCfg<uint32_t>::kCap : MwCfg<uint64_t>::kCap;
}
// Sorted samples per piece: a piece holds on average step / (step + k) of the
// keys that fit it.  The tree takes 5/6 (every round reads the whole piece's
// slots); radix passes skip the slots a piece does not fill, and 3/4 leaves
// fewer samples to sort (64 x 2^22 u32 keys 1.73 -> 1.69 ms, 16 x 2^22 i64
// keys 0.73 -> 0.69 ms; 8 x 2^26 u32 keys 1.84 against 1.86 ms).
inline uint32_t piece_step(int kb, size_t k) {
  return (uint32_t)std::max<size_t>(8, (tree_pieces(kb, k) ? 5 : 3) * k);
}
constexpr size_t kMwMaxRuns = 256;

inline uint32_t sample_stride(int kb, size_t k) {
  return (uint32_t)(piece_cap(kb, k) / (piece_step(kb, k) + k));
}

size_t align_up(size_t x) { return (x + 255) / 256 * 256; }

struct MwLayout {
  size_t status, ptrs, lens, sbase, skeys, skeys2, sid, sid2, sort_temp, splits, bases, total;
  uint64_t ns, pieces;
};

// ns: sample count, exact when lens are known, else the bound for total keys.
MwLayout mw_layout(int kb, size_t k, uint64_t ns) {
  MwLayout L{};
  L.ns = ns;
  L.pieces = ns == 0 ? 0 : (ns - 1) / piece_step(kb, k) + 1;
  size_t o = 0;
  auto take = [&](size_t bytes) {
    const size_t at = o;
    o = align_up(o + bytes);
    return at;
  };
  L.status = take(4);  // first: the call's status word
  L.ptrs = take(k * 8);
  L.lens = take(k * 8);
  L.sbase = take((k + 1) * 8);
  L.skeys = take(ns * kb);
  L.skeys2 = take(ns * kb);
  L.sid = take(ns * 4);
  L.sid2 = take(ns * 4);
  L.sort_temp = take(sort_temp_bytes(kb == 4 ? MGS_KEY_U32 : MGS_KEY_U64, MGS_VAL_U32, ns));
  L.splits = take((L.pieces + 1) * k * 8);
  L.bases = take((L.pieces + 1) * 8);
  L.total = o;
  return L;
}

uint64_t sample_count(const size_t* lens, size_t k, uint32_t S) {
  uint64_t ns = 0;
  for (size_t j = 0; j < k; ++j) ns += (lens[j] + S - 1) / S;
  return ns;
}

// Sample q: run j with sbase[j] <= q < sbase[j+1], index (q - sbase[j]) S.
template <typename Bits>
__global__ void mw_sample_kernel(const Bits* const* __restrict__ runs, const uint64_t* __restrict__ sbase, uint32_t k,
                                 uint32_t S, uint64_t ns, Bits* __restrict__ skeys, uint32_t* __restrict__ sid,
                                 uint32_t* __restrict__ status) {
  const uint64_t q = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q == 0) *status = 0;  // the kernels after this one only OR into it
  if (q >= ns) return;
  uint32_t lo = 0, hi = k;  // last j with sbase[j] <= q
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (sbase[mid] <= q)
      lo = mid;
    else
      hi = mid;
  }
  skeys[q] = runs[lo][(q - sbase[lo]) * S];
  sid[q] = (uint32_t)q;
}

// Keys of run r that precede value e in encoded order, strictly smaller
// (UPPER false) or smaller or equal (UPPER true), searched in [lo, hi].
template <int KT, bool UPPER, typename Bits>
__device__ __forceinline__ uint64_t bound_global(const Bits* r, uint64_t lo, uint64_t hi, Bits e) {
  while (lo < hi) {
    const uint64_t mid = (lo + hi) >> 1;
    const Bits m = Codec<KT>::enc(r[mid]);
    if (UPPER ? (m <= e) : (m < e))
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo;
}

// Boundaries per coarse boundary: the splits of every kMwCoarse-th boundary
// are searched over the whole runs, the others between those of their coarse
// neighbours, about half the dependent loads and on shared cache lines.
constexpr uint64_t kMwCoarse = 16;
// Two levels pay for their second launch where there are searches enough that
// their loads, and not the longest search, bound the split kernel: whole call, one
// level against two, u32: 64 runs of 2^19 313 / 307 us, of 2^22 2005 / 1709;
// 256 of 2^20 4804 / 3424; 32 of 2^21 425 / 432, of 2^22 745 / 730; 16 of 2^23 543 / 553;
// and up to 8 runs at no size (8 of 2^19 126 / 136, of 2^26 1819 / 1836).
inline bool two_levels(uint64_t pieces, size_t k) { return k > 8 && pieces * k > (uint64_t(1) << 19); }

// Thread (b, j'): split of run j' at boundary b (1 <= b < pieces); boundary
// 0 and `pieces` are the runs' ends.  COARSE: the boundaries that are
// multiples of `coarse`, and `pieces`; otherwise the rest, after them.
template <int KT, bool COARSE, typename Bits>
__global__ void mw_split_kernel(const Bits* const* __restrict__ runs, const uint64_t* __restrict__ lens,
                                const uint64_t* __restrict__ sbase, uint32_t k, uint32_t S,
                                const Bits* __restrict__ skeys, const uint32_t* __restrict__ sid, uint64_t pieces,
                                uint32_t step, uint64_t coarse, uint64_t* splits) {
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t q = t / k;
  const uint32_t jj = (uint32_t)(t % k);
  const uint64_t b = COARSE ? std::min(q * coarse, pieces) : q + q / (coarse - 1) + 1;
  if (COARSE ? q > (pieces + coarse - 1) / coarse : b >= pieces) return;
  uint64_t* const out = splits + b * k + jj;
  if (b == 0 || b == pieces) {
    *out = b == 0 ? 0 : lens[jj];
    return;
  }
  const Bits e = Codec<KT>::enc(skeys[b * step]);
  const uint32_t id = sid[b * step];
  uint32_t lo = 0, hi = k;  // run of sample id
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (sbase[mid] <= id)
      lo = mid;
    else
      hi = mid;
  }
  const uint32_t j = lo;
  uint64_t from = 0, to = lens[jj];
  if (!COARSE) {
    const uint64_t c = b / coarse * coarse;
    from = splits[c * k + jj];
    to = std::max(from, splits[std::min(c + coarse, pieces) * k + jj]);
  }
  if (jj == j)
    *out = (id - sbase[j]) * (uint64_t)S;
  else if (jj < j)
    *out = bound_global<KT, true>(runs[jj], from, to, e);
  else
    *out = bound_global<KT, false>(runs[jj], from, to, e);
}

__global__ void mw_base_kernel(const uint64_t* __restrict__ splits, uint32_t k, uint64_t pieces,
                               uint64_t* __restrict__ bases, const uint32_t* __restrict__ sort_status,
                               uint32_t* __restrict__ status) {
  const uint64_t b = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b == 0 && *sort_status) atomicOr(status, *sort_status);  // the sample sort's own status word
  if (b > pieces) return;
  uint64_t s = 0;
  for (uint32_t j = 0; j < k; ++j) s += splits[b * k + j];
  bases[b] = s;
}

// Keys of `a` taken among the first `diag` outputs of the stable merge of
// a (na keys, taken first on ties) and b (nb keys), both in LDS.
template <int KT, typename Bits>
__device__ __forceinline__ uint32_t corank_lds(const Bits* a, uint32_t na, const Bits* b, uint32_t nb, uint32_t diag) {
  uint32_t lo = diag > nb ? diag - nb : 0;
  uint32_t hi = diag < na ? diag : na;
  while (lo < hi) {
    const uint32_t mid = (lo + hi) >> 1;
    if (Codec<KT>::enc(a[mid]) <= Codec<KT>::enc(b[diag - mid - 1]))
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo;
}

// One piece: its slices of the k runs are loaded into LDS back to back (run
// order), then merged in ceil(log2 k) rounds, each merging adjacent slice
// pairs (2i, 2i+1) into the other LDS buffer (earlier runs first on ties, so
// the order stays stable).  In a round every thread writes q consecutive
// outputs (q odd, q * kTreeBlock >= the piece's keys, q <= kTreeCap / kTreeBlock + 1):
// one co-rank search in its pair, then a serial merge.
template <int KT, typename Bits>
__global__ __launch_bounds__(kTreeBlock) void mw_tree_kernel(const Bits* const* __restrict__ runs, uint32_t k,
                                                            const uint64_t* __restrict__ splits,
                                                            const uint64_t* __restrict__ bases, uint64_t first_piece,
                                                            Bits* __restrict__ out, uint32_t* __restrict__ status) {
  // loads per thread: the piece's keys at most
  constexpr uint32_t kLoads = kTreeCap / kTreeBlock;
  __shared__ Bits buf[2][kTreeCap];
  __shared__ uint32_t bnd[kMwMaxRuns + 1];
  __shared__ uint64_t sbeg[kMwMaxRuns];
  __shared__ const Bits* sptr[kMwMaxRuns];
  __shared__ uint32_t sums[4];
  const int tid = threadIdx.x;
  const uint64_t b = first_piece + blockIdx.x;
  // slice j of the piece: runs[j][splits[b][j], splits[b+1][j]); slices that
  // go backwards or more than kTreeCap keys in all (only unsorted runs break the
  // sample bound) leave the piece unmerged and the call reports it;
  // otherwise the piece's keys are exactly [bases[b], bases[b+1]) of the
  // output
  uint32_t len = 0;
  bool bad = false;
  if ((uint32_t)tid < k) {
    const uint64_t lo = splits[b * k + tid], hi = splits[(b + 1) * k + tid];
    bad = hi < lo;
    len = bad ? 0u : (uint32_t)std::min<uint64_t>(hi - lo, kTreeCap + 1);
    sbeg[tid] = lo;
    sptr[tid] = runs[tid];
  }
  const uint32_t excl = block_excl_scan_256((uint32_t)tid < k ? len : 0u, sums, tid);
  if ((uint32_t)tid < k) {
    bnd[tid] = min(excl, kTreeCap);
    if ((uint32_t)tid == k - 1) {
      bad = bad || excl + len > kTreeCap;
      bnd[k] = min(excl + len, kTreeCap);
    }
  }
  if (__syncthreads_or(bad ? 1 : 0)) {
    if (tid == 0) atomicOr(status, kStatusUnsorted);
    return;
  }
  const uint32_t cnt = bnd[k];
  // outputs per thread in a merge round: the fewest that cover the piece, odd
  // so that the lanes' serial merges start in different LDS banks (a piece of
  // 6800 keys, the average for 8 runs, takes 7 per thread)
  const uint32_t q = ((cnt + kTreeBlock - 1) / kTreeBlock) | 1u;
  {
    // every load of the piece issued before the first LDS store
    Bits v[kLoads];
#pragma unroll
    for (uint32_t i = 0; i < kLoads; ++i) {
      const uint32_t e = (uint32_t)tid + i * kTreeBlock;
      v[i] = Bits(0);
      if (e < cnt) {
        uint32_t lo = 0, hi = k;  // the slice of slot e: last j with bnd[j] <= e
        while (hi - lo > 1) {
          const uint32_t mid = (lo + hi) >> 1;
          if (bnd[mid] <= e)
            lo = mid;
          else
            hi = mid;
        }
        v[i] = sptr[lo][sbeg[lo] + (e - bnd[lo])];
      }
    }
#pragma unroll
    for (uint32_t i = 0; i < kLoads; ++i) {
      const uint32_t e = (uint32_t)tid + i * kTreeBlock;
      if (e < cnt) buf[0][e] = v[i];
    }
  }
  int cur = 0;
  for (uint32_t slices = k; slices > 1; slices = (slices + 1) >> 1) {
    __syncthreads();
    const Bits* src = buf[cur];
    Bits* dst = buf[cur ^ 1];
    const uint32_t pairs = (slices + 1) >> 1;
    uint32_t o = (uint32_t)tid * q;
    const uint32_t end = min(o + q, cnt);
    while (o < end) {
      // the last pair i with bnd[2i] <= o: it ends beyond o (a later pair
      // starts beyond o, or it is the last pair, which ends at cnt)
      uint32_t lo = 0, hi = pairs;
      while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (bnd[2 * mid] <= o)
          lo = mid;
        else
          hi = mid;
      }
      const uint32_t a0 = bnd[2 * lo], a1 = bnd[min(2 * lo + 1, slices)], b1 = bnd[min(2 * lo + 2, slices)];
      const uint32_t na = a1 - a0, nb = b1 - a1;
      const uint32_t pend = min(end, b1);
      uint32_t ia = corank_lds<KT>(src + a0, na, src + a1, nb, o - a0);
      uint32_t ib = (o - a0) - ia;
      // the heads of both sides in registers: one LDS load per output
      Bits ka = ia < na ? src[a0 + ia] : Bits(0);
      Bits kb = ib < nb ? src[a1 + ib] : Bits(0);
      for (; o < pend; ++o) {  // branch-free: one LDS store and one load per output
        const bool take_a = ib >= nb || (ia < na && Codec<KT>::enc(ka) <= Codec<KT>::enc(kb));
        dst[o] = take_a ? ka : kb;
        ia += take_a ? 1u : 0u;
        ib += take_a ? 0u : 1u;
        const uint32_t at = take_a ? a0 + ia : a1 + ib;  // the taken side's next key (past its end: ignored)
        const Bits nk = src[min(at, kTreeCap - 1)];
        ka = take_a ? nk : ka;
        kb = take_a ? kb : nk;
      }
    }
    __syncthreads();
    // boundaries of the merged slices: slice i starts where pair i did
    uint32_t nb_val = 0;
    const uint32_t nslices = pairs;
    if ((uint32_t)tid <= nslices) nb_val = bnd[min(2 * (uint32_t)tid, slices)];
    __syncthreads();
    if ((uint32_t)tid <= nslices) bnd[tid] = nb_val;
    cur ^= 1;
  }
  __syncthreads();
  Bits* dst = out + bases[b];
  for (uint32_t e = tid; e < cnt; e += kTreeBlock) dst[e] = buf[cur][e];
}

// One piece: its slices of the k runs, laid end to end in run order, are
// sorted stably by one workgroup (block_sort.hpp), which is their stable
// merge.
template <int KT, typename Bits>
__global__ __launch_bounds__(kMwBlock, MwCfg<Bits>::kWaves) void mw_piece_kernel(const Bits* const* __restrict__ runs, uint32_t k,
                                                            const uint64_t* __restrict__ splits,
                                                            const uint64_t* __restrict__ bases, const Bits* __restrict__ skeys,
                                                            uint64_t pieces, uint32_t step, uint64_t first_piece,
                                                            Bits* __restrict__ out, uint32_t* __restrict__ status) {
  constexpr int kIpt = MwCfg<Bits>::kIpt;
  constexpr uint32_t kCap = MwCfg<Bits>::kCap;
  __shared__ BlockSortSmem<Bits, NoVal, kMwBlock, kIpt> sm;
  __shared__ uint32_t bnd[kMwMaxRuns + 1];
  __shared__ const Bits* sptr[kMwMaxRuns];
  __shared__ uint32_t sums[4];
  const int tid = threadIdx.x;
  const uint64_t b = first_piece + blockIdx.x;
  // slice j of the piece: runs[j][splits[b][j], splits[b+1][j]); slices that
  // go backwards or more than kCap keys in all (only unsorted runs break the
  // sample bound) leave the piece unmerged and the call reports it;
  // otherwise the piece's keys are exactly [bases[b], bases[b+1]) of the
  // output
  uint32_t len = 0;
  bool bad = false;
  // the samples at the piece's ends bound its keys
  const Bits mn = b > 0 ? Codec<KT>::enc(skeys[b * step]) : Bits(0);
  const Bits mx = b + 1 < pieces ? Codec<KT>::enc(skeys[(b + 1) * step]) : ~Bits(0);
  if ((uint32_t)tid < k) {
    const uint64_t lo = splits[b * k + tid], hi = splits[(b + 1) * k + tid];
    bad = hi < lo;
    len = bad ? 0u : (uint32_t)std::min<uint64_t>(hi - lo, kCap + 1);
    sptr[tid] = runs[tid] + lo;
  }
  block_clear_row<kMwBlock>(sm.off);
  const uint32_t excl = block_excl_scan_256((uint32_t)tid < k ? len : 0u, sums, tid);
  if ((uint32_t)tid < k) {
    bnd[tid] = min(excl, kCap);
    if ((uint32_t)tid == k - 1) {
      bad = bad || excl + len > kCap;
      bnd[k] = min(excl + len, kCap);
    }
  }
  if (__syncthreads_or(bad ? 1 : 0)) {
    if (tid == 0) atomicOr(status, kStatusUnsorted);
    return;
  }
  const uint32_t cnt = readfirstlane(bnd[k]);
  if (cnt == 0) return;
  const uint32_t nit = block_items<kMwBlock>(cnt), wb = block_first<kMwBlock>(nit);
  const Bits pad = Codec<KT>::dec(mx);
  Bits key[kIpt];
  uint32_t none[kIpt];
  // the slice of the thread's first slot (last j with bnd[j] <= wb), then on
  // from slice to slice as its slots pass their ends
  uint32_t lo = 0, hi = k;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (bnd[mid] <= wb)
      lo = mid;
    else
      hi = mid;
  }
  uint32_t next = bnd[lo + 1];
  const Bits* src = sptr[lo] - bnd[lo];
  static_for<kIpt>([&](auto i) {
    const uint32_t e = wb + i * kWave;
    key[i] = pad;
    if ((uint32_t)i < nit && e < cnt) {
      if (e >= next) {
        do next = bnd[++lo + 1];
        while (e >= next);
        src = sptr[lo] - bnd[lo];
      }
      key[i] = src[e];
    }
  });
  // (only unsorted runs have keys outside the samples' bounds; block_sort
  // then stays in bounds, but padding may take their place)
  static_for<kIpt>([&](auto i) {
    const Bits x = Codec<KT>::enc(key[i]);
    bad |= x < mn || x > mx;
  });
  if (bad) atomicOr(status, kStatusUnsorted);
  block_sort<KT, NoVal, kMwBlock, kIpt>(sm, key, none, cnt, mn, mx, out + bases[b], (NoVal*)nullptr);
}

// Launches the pieces [first, first + count).
template <int KT, typename Bits>
void launch_pieces(const Bits* const* d_runs, size_t k, const uint64_t* splits, const uint64_t* bases, const Bits* skeys,
                   uint64_t pieces, uint64_t first, uint64_t count, Bits* out, uint32_t* status, hipStream_t s) {
  if constexpr (sizeof(Bits) == 8) {
    if (tree_pieces(8, k)) {
      mw_tree_kernel<KT, Bits><<<(uint32_t)count, kTreeBlock, 0, s>>>(d_runs, (uint32_t)k, splits, bases, first, out,
                                                                     status);
      return;
    }
  }
  mw_piece_kernel<KT, Bits><<<(uint32_t)count, kMwBlock, 0, s>>>(d_runs, (uint32_t)k, splits, bases, skeys, pieces,
                                                                 piece_step(sizeof(Bits), k), first, out, status);
}

uint32_t grid_of(uint64_t threads, int block) { return (uint32_t)((threads + block - 1) / block); }

template <int KT>
int mw_launch(const void* const* runs, const size_t* lens, size_t k, void* out, void* temp, size_t temp_bytes,
              hipStream_t s, size_t portions, size_t* portion_end, hipEvent_t* portion_done) {
  using Bits = typename Codec<KT>::Bits;
  constexpr int KB = sizeof(Bits);
  const uint32_t S = sample_stride(KB, k);
  const uint64_t ns = sample_count(lens, k, S);
  if (ns > 0 && k <= 2)
    return merge_two_runs((mgs_key)KT, runs[0], lens[0], k > 1 ? runs[1] : nullptr, k > 1 ? lens[1] : 0, out, temp,
                          temp_bytes, s, portions, portion_end, portion_done);
  if (ns > (uint64_t)MGS_MAX_KEYS) return MGS_ERR_TOO_LARGE;  // sample ids and the sample sort
  if (ns == 0) {  // no keys: nothing to merge and no tables, the status word says ok
    if (temp == nullptr || temp_bytes < sizeof(uint32_t)) return MGS_ERR_TEMP_TOO_SMALL;
    hipError_t z = hipMemsetAsync(temp, 0, 4, s);
    for (size_t p = 0; z == hipSuccess && p < portions; ++p) {
      portion_end[p] = 0;
      if (portion_done) z = hipEventRecord(portion_done[p], s);
    }
    return record_hip(z);
  }
  const MwLayout L = mw_layout(KB, k, ns);
  if (temp == nullptr || temp_bytes < L.total) return MGS_ERR_TEMP_TOO_SMALL;
  char* t = static_cast<char*>(temp);
  // run table: host arrays copied into temp (pageable sources; the copy
  // has read them when hipMemcpyAsync returns)
  std::vector<uint64_t> h(3 * k + 1);
  uint64_t acc = 0;
  for (size_t j = 0; j < k; ++j) {
    h[j] = reinterpret_cast<uint64_t>(runs[j]);
    h[k + j] = lens[j];
    h[2 * k + j] = acc;
    acc += (lens[j] + S - 1) / S;
  }
  h[3 * k] = acc;
  hipError_t e = hipMemcpyAsync(t + L.ptrs, h.data(), k * 8, hipMemcpyHostToDevice, s);
  if (e == hipSuccess) e = hipMemcpyAsync(t + L.lens, h.data() + k, k * 8, hipMemcpyHostToDevice, s);
  if (e == hipSuccess) e = hipMemcpyAsync(t + L.sbase, h.data() + 2 * k, (k + 1) * 8, hipMemcpyHostToDevice, s);
  if (e != hipSuccess) return record_hip(e);
  const Bits* const* d_runs = reinterpret_cast<const Bits* const*>(t + L.ptrs);
  const uint64_t* d_lens = reinterpret_cast<const uint64_t*>(t + L.lens);
  const uint64_t* d_sbase = reinterpret_cast<const uint64_t*>(t + L.sbase);
  Bits* sk = reinterpret_cast<Bits*>(t + L.skeys);
  Bits* sk2 = reinterpret_cast<Bits*>(t + L.skeys2);
  uint32_t* sid = reinterpret_cast<uint32_t*>(t + L.sid);
  uint32_t* sid2 = reinterpret_cast<uint32_t*>(t + L.sid2);
  uint64_t* splits = reinterpret_cast<uint64_t*>(t + L.splits);
  uint64_t* bases = reinterpret_cast<uint64_t*>(t + L.bases);
  uint32_t* status = reinterpret_cast<uint32_t*>(t + L.status);
  const uint32_t* sort_status = reinterpret_cast<const uint32_t*>(t + L.sort_temp);  // first word of its scratch

  mw_sample_kernel<Bits><<<grid_of(ns, 256), 256, 0, s>>>(d_runs, d_sbase, (uint32_t)k, S, ns, sk, sid, status);
  int rc = check_launch();
  if (rc != MGS_OK) return rc;
  rc = sort_dispatch((mgs_key)KT, MGS_VAL_U32, sk, sk2, sid, sid2, ns, t + L.sort_temp,
                     sort_temp_bytes((mgs_key)KT, MGS_VAL_U32, ns), s);
  if (rc != MGS_OK) return rc;
  const uint64_t coarse = two_levels(L.pieces, k) ? kMwCoarse : 1;
  mw_split_kernel<KT, true, Bits><<<grid_of(((L.pieces + coarse - 1) / coarse + 1) * k, 256), 256, 0, s>>>(
      d_runs, d_lens, d_sbase, (uint32_t)k, S, sk2, sid2, L.pieces, piece_step(KB, k), coarse, splits);
  if (coarse > 1)
    mw_split_kernel<KT, false, Bits><<<grid_of((L.pieces - 1) * k, 256), 256, 0, s>>>(
        d_runs, d_lens, d_sbase, (uint32_t)k, S, sk2, sid2, L.pieces, piece_step(KB, k), coarse, splits);
  mw_base_kernel<<<grid_of(L.pieces + 1, 256), 256, 0, s>>>(splits, (uint32_t)k, L.pieces, bases, sort_status,
                                                            status);
  rc = check_launch();
  if (rc != MGS_OK) return rc;

  Bits* o = static_cast<Bits*>(out);
  if (portions <= 1) {
    launch_pieces<KT, Bits>(d_runs, k, splits, bases, sk2, L.pieces, 0, L.pieces, o, status, s);
    rc = check_launch();
    if (rc == MGS_OK && portions == 1) {
      size_t n = 0;
      for (size_t j = 0; j < k; ++j) n += lens[j];
      portion_end[0] = n;
      if (portion_done) rc = record_hip(hipEventRecord(portion_done[0], s));
    }
    return rc;
  }
  // portions: pieces [P p / portions, P (p+1) / portions); their output ends
  // come from the bases, read back once
  std::vector<uint64_t> first(portions + 1);
  for (size_t p = 0; p <= portions; ++p) first[p] = L.pieces * p / portions;
  std::vector<uint64_t> hb(L.pieces + 1);
  e = hipMemcpyAsync(hb.data(), bases, (L.pieces + 1) * 8, hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) return record_hip(e);
  for (size_t p = 0; p < portions; ++p) {
    const uint64_t np = first[p + 1] - first[p];
    if (np > 0)
      launch_pieces<KT, Bits>(d_runs, k, splits, bases, sk2, L.pieces, first[p], np, o, status, s);
    rc = check_launch();
    if (rc != MGS_OK) return rc;
    portion_end[p] = (size_t)hb[first[p + 1]];
    if (portion_done) {
      rc = record_hip(hipEventRecord(portion_done[p], s));
      if (rc != MGS_OK) return rc;
    }
  }
  return MGS_OK;
}

template <int KB>
size_t mw_bytes(size_t k, size_t total) {
  if (k == 0) return 256;
  if (k <= 2) return merge_two_runs_temp_bytes(total);
  const uint32_t S = sample_stride(KB, k);
  return mw_layout(KB, k, total / S + k).total;
}

}  // namespace

size_t multiway_temp_bytes(mgs_key kt, size_t k, size_t total) {
  const int kb = key_bytes(kt);
  if (kb < 0 || k > kMwMaxRuns) return 0;
  return kb == 4 ? mw_bytes<4>(k, total) : mw_bytes<8>(k, total);
}

int multiway_dispatch(mgs_key kt, const void* const* runs, const size_t* lens, size_t k, void* out, void* temp,
                      size_t temp_bytes, hipStream_t s, size_t portions, size_t* portion_end,
                      hipEvent_t* portion_done) {
  if (k > kMwMaxRuns) return MGS_ERR_INVALID;
  switch (kt) {
    case MGS_KEY_U32: return mw_launch<MGS_KEY_U32>(runs, lens, k, out, temp, temp_bytes, s, portions, portion_end, portion_done);
    case MGS_KEY_U64: return mw_launch<MGS_KEY_U64>(runs, lens, k, out, temp, temp_bytes, s, portions, portion_end, portion_done);
    case MGS_KEY_I32: return mw_launch<MGS_KEY_I32>(runs, lens, k, out, temp, temp_bytes, s, portions, portion_end, portion_done);
    case MGS_KEY_I64: return mw_launch<MGS_KEY_I64>(runs, lens, k, out, temp, temp_bytes, s, portions, portion_end, portion_done);
    case MGS_KEY_F32: return mw_launch<MGS_KEY_F32>(runs, lens, k, out, temp, temp_bytes, s, portions, portion_end, portion_done);
    case MGS_KEY_F64: return mw_launch<MGS_KEY_F64>(runs, lens, k, out, temp, temp_bytes, s, portions, portion_end, portion_done);
  }
  return MGS_ERR_BAD_TYPE;
}

}  // namespace mgs
