// Three-pass hybrid radix sort of 8-byte keys and of keys with payloads
// (msd_wide.hip; the kernels of one record type are in msd_wide_kernels.hpp).
// The LSD passes (radix_sort.hip) move every record sizeof(key) times; this
// path moves it three times whatever the key's width:
//
//   upfront  one read of the keys: a 16-bit window of every encoded key (the
//            16 bits below the leading bits that a sample of 1024 keys
//            shares) is counted per range of the input, as in the path of
//            4-byte keys (msd_sort.hip)
//   scan     sub-bucket (window value) offsets, look-back tables, and the
//            batches of the last step: consecutive sub-buckets of one bucket
//            that one workgroup sorts
//   pass 1   scatter by the window's high byte, 8 chains of tiles
//   pass 2   scatter by its low byte inside each of the 256 buckets
//   local    every batch is sorted in LDS by its bits below the window and
//            those in which its sub-buckets differ (block_sort.hpp: up to three
//            passes over the top 27 of them and a look at the neighbours) and
//            written back in place
//
// A sub-bucket that does not fit a workgroup, a key outside the sample's
// shared leading bits, a window counter that overflowed or one XCD's buckets
// holding more than twice their share turn the path off (MsdCtl::off): the
// LSD passes, launched behind it, then run.  So does the upfront's sample,
// before the read, when too many of its keys share their window value.
#pragma once

#include "msd_sort.hpp"

namespace mgs {

// Geometry of one record type.  The scatter passes take the LSD passes'
// tiles (512 threads, one workgroup per CU: TileCfg); the local sort takes
// the records of two 512-thread workgroups per CU.
template <int KB, int VB>
struct WideCfg {
  static constexpr int kRec = KB + VB;
  static constexpr int kBlock = 512;
  static constexpr int kIpt = kRec <= 8 ? 28 : kRec <= 12 ? 16 : 12;
  static constexpr int kTile = kBlock * kIpt;
  static constexpr int kLocalIpt = kRec <= 8 ? 14 : kRec <= 12 ? 10 : 7;
  static constexpr uint32_t kCap = (uint32_t)kBlock * kLocalIpt;  // records of one batch
};
inline int wide_tile(int rec) { return rec <= 8 ? WideCfg<8, 0>::kTile : rec <= 12 ? WideCfg<8, 4>::kTile : WideCfg<8, 8>::kTile; }
inline uint32_t wide_cap(int rec) { return rec <= 8 ? WideCfg<8, 0>::kCap : rec <= 12 ? WideCfg<8, 4>::kCap : WideCfg<8, 8>::kCap; }

// Integer keys only: the exponents of floats (uniform in [0, 1), normal) put
// whole percents of them into one window value, so the path would always be
// left, and its launches alone cost 5-15% of a sort of 2^22 keys.
template <int KT>
constexpr bool kFloatKey = KT == MGS_KEY_F32 || KT == MGS_KEY_F64;

// Sizes the path is tried for: up to where the sub-buckets of uniform keys
// (n / 65536, Poisson) still fit a workgroup, and from where it beats the
// splits (segmented.hip) for 8-byte keys: u64 2^22 164 us against 155 us, 2^23
// 198 against 251, 2^24 327 against 430; and the LSD passes for 4-byte keys
// with payloads: u32 + u32 2^24 366 -> 311 us.
inline size_t wide_min(int kb) { return size_t(1) << (kb == 8 ? 23 : 24); }
size_t wide_max(int rec);
bool wide_eligible(int kb, int vb, size_t n);

constexpr uint32_t kWideRanges = 256;  // input ranges counted apart

struct WideLayout {
  size_t ctl, desc, slices, range_hist, range_pref, range_bad, xcd_of, sub_off, bucket_tot, bucket_start, leaders,
      batch_cnt, batch_base, batches, tile_base1, tile_base2, counters, end;
};
// Scratch from offset `at` of temp (it may overlap the LSD descriptors), the
// control block at `ctl_at` (which must not).
WideLayout wide_layout(int rec, size_t n, size_t at, size_t ctl_at);

// How the input is cut: ranges of whole tiles counted apart by the upfront,
// kWideRanges / 8 of them to a chain of pass 1.
struct WidePlan {
  uint32_t tiles, tiles_per_range, range_keys, ranges, chains1, ranges_per_chain;
};
WidePlan wide_plan(int rec, size_t n);

// The tables between the upfront and pass 1.
int wide_tables(int rec, size_t n, const WidePlan& P, char* t, const WideLayout& L, hipStream_t s, Marks& mark);

// Enqueues the path: pass 1 from kin into alt, pass 2 and the local sort into
// kout.
template <int KT, int VT>
int wide_launch(const void* kin, void* kout, void* kalt, const void* vin, void* vout, void* valt, size_t n, char* t,
                const WideLayout& L, uint32_t* status, uint32_t spin_limit, hipStream_t s, Marks& mark);

}  // namespace mgs
