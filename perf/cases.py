"""Performance cases of the sorting library: what its users have it do.

Each case goes through the package's public entry points (mgsort.sort,
merge, multiway_merge, segmented_sort, segmented_sort_ranges) with the
buffers that a program keeps between calls: inputs, outputs and scratch.
Sorts are out of place, so a pass can be repeated on the same inputs.

Kinds of case and their fields:
  sort      n keys of type `key` (u32, u64, i32, i64, f32, f64), payload `val`
            ("none", "u32", "u64"), key distribution `dist`
  segments  `nseg` arrays laid end to end, lengths log-uniform in
            [2^lo, 2^hi] (the batched workload); `batch` seeds the lengths
  ranges    the same lengths, each array somewhere in one pool, sorted in
            place (what the serving layer runs); the pool is first refilled
            from the requests' arrival buffer
  merge     two sorted runs of n0 and n1 keys into one (the Tanasic sort's
            local merge)
  multiway  `runs` sorted runs of about n / runs keys each into one (the
            heterogeneous sort's device merge)
"""
import ctypes
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "multi-gpu-sorting_amd"))
import mgsort  # noqa: E402
from mgsort import batched, tuning  # noqa: E402

KEY_DTYPE = {"u32": torch.int32, "i32": torch.int32, "f32": torch.float32,
             "u64": torch.int64, "i64": torch.int64, "f64": torch.float64}
VAL_DTYPE = {"u32": torch.int32, "u64": torch.int64}


def listed():
    return [
        # a request of a few thousand bytes: one launch, all latency
        {"name": "sort_u32_2k", "kind": "sort", "key": "u32", "val": "none", "n": 2000, "dist": "uniform"},
        # a small index build (key + row number): launches count
        {"name": "sort_u32v32_50k", "kind": "sort", "key": "u32", "val": "u32", "n": 50_021, "dist": "uniform"},
        # an ordinary 64-bit column chunk, odd size
        {"name": "sort_u64_1m", "kind": "sort", "key": "u64", "val": "none", "n": 1_000_003, "dist": "uniform"},
        # the reference's smallest benchmark array
        {"name": "sort_u32_16m", "kind": "sort", "key": "u32", "val": "none", "n": 1 << 24, "dist": "uniform"},
        # measured values: floats whose exponents crowd into few digits, ragged size
        {"name": "sort_f32_67m_normal", "kind": "sort", "key": "f32", "val": "none", "n": (1 << 26) + 4321,
         "dist": "normal"},
        # a table sorted by a 64-bit key with row numbers
        {"name": "sort_u64v32_67m", "kind": "sort", "key": "u64", "val": "u32", "n": 1 << 26, "dist": "uniform"},
        # one GPU's share of a large 64-bit sort
        {"name": "sort_u64_268m", "kind": "sort", "key": "u64", "val": "none", "n": 1 << 28, "dist": "uniform"},
        # the headline: 2^30 keys resident in HBM
        {"name": "sort_u32_1g", "kind": "sort", "key": "u32", "val": "none", "n": 1 << 30, "dist": "uniform"},
        # the batched workload's lengths and record, a quarter of its arrays
        {"name": "segments_u64v32_1024", "kind": "segments", "key": "u64", "val": "u32", "nseg": 1024, "lo": 8.0,
         "hi": 22.0, "batch": 2024, "dist": "uniform"},
        # a batch of serving requests
        {"name": "ranges_u32_256", "kind": "ranges", "key": "u32", "val": "none", "nseg": 256, "lo": 10.0, "hi": 18.0,
         "batch": 2024, "dist": "uniform"},
        # local merge step of two sorted partitions
        {"name": "merge_u32_2x134m", "kind": "merge", "key": "u32", "val": "none", "n0": 1 << 27, "n1": 1 << 27},
        # the heterogeneous sort's final merge of 8 sorted chunks
        {"name": "multiway_u32_8x67m", "kind": "multiway", "key": "u32", "runs": 8, "n": 1 << 29},
    ]


def _log_size(rng, lo, hi):
    """An odd-ish size, log-uniform in [lo, hi]."""
    return int(min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng: random.Random):
    kind = rng.choices(["sort", "segments", "ranges", "merge", "multiway"], [10, 2, 2, 2, 3])[0]
    if kind == "sort":
        key = rng.choice(["u32", "u32", "i32", "f32", "u64", "i64", "f64"])
        val = rng.choice(["none", "none", "u32", "u64"])
        rec = (4 if key.endswith("32") else 8) + {"none": 0, "u32": 4, "u64": 8}[val]
        n = _log_size(rng, 500, (1 << 32) // rec if rec == 4 else (1 << 31) // rec)
        dists = ["uniform", "uniform", "normal", "sorted"] + (["zipf"] if key[0] != "f" and n <= 1 << 27 else [])
        return {"kind": kind, "key": key, "val": val, "n": n, "dist": rng.choice(dists)}
    if kind in ("segments", "ranges"):
        key, val = rng.choice([("u64", "u32"), ("u32", "none"), ("u32", "u32"), ("u64", "none"), ("f32", "none")])
        lo = rng.uniform(6.0, 11.0)
        hi = rng.uniform(lo + 2.0, 22.0 if kind == "segments" else 20.0)
        mean = (2.0 ** hi - 2.0 ** lo) / ((hi - lo) * math.log(2.0))
        nseg = _log_size(rng, 16, max(17, min(4096, int((1 << 28) / mean))))
        dist = rng.choice(["uniform", "uniform", "normal" if key[0] == "f" else "zipf"])
        return {"kind": kind, "key": key, "val": val, "nseg": nseg, "lo": lo, "hi": hi,
                "batch": rng.randrange(1 << 20), "dist": dist}
    if kind == "merge":
        key = rng.choice(["u32", "u64", "f32"])
        val = rng.choice(["none", "none", "u32"])
        n = _log_size(rng, 1000, 1 << 28 if key != "u64" else 1 << 27)
        n0 = int(n * rng.uniform(0.2, 0.8))
        return {"kind": kind, "key": key, "val": val, "n0": n0, "n1": n - n0}
    key = rng.choice(["u32", "u32", "u64"])
    return {"kind": kind, "key": key, "runs": rng.choice([2, 3, 4, 8, 8, 16, 32, 64]),
            "n": _log_size(rng, 100_000, 1 << 29 if key == "u32" else 1 << 27)}


def _lengths(case, seed):
    """Array lengths of a batch, round(2^(lo + (hi - lo) U)) with the case's
    own draws of U, in an order of the seed's."""
    r = random.Random(case["batch"])
    lens = [int(round(2.0 ** r.uniform(case["lo"], case["hi"]))) for _ in range(case["nseg"])]
    random.Random(seed).shuffle(lens)
    return np.array(lens, dtype=np.int64)


def _ascending(key, n, g):
    """n sorted keys, uniform over the range (floats: over [-1, 1)), as the
    running sum of exponential gaps (an exact integer sum, so ascending)."""
    if n == 0:
        return torch.empty(0, dtype=KEY_DTYPE[key], device="cuda")
    u = torch.rand(n, dtype=torch.float64, device="cuda", generator=g)
    c = torch.cumsum((-torch.log1p(-u) * 2.0 ** 30).to(torch.int64) + 1, 0)
    x = c.to(torch.float64) / (float(c[-1].item()) + 2.0 ** 30)  # in (0, 1), ascending
    if key in ("f32", "f64"):
        return (2.0 * x - 1.0).to(KEY_DTYPE[key])
    if key in ("u32", "i32"):
        v = (x * 2.0 ** 32).to(torch.int64)  # 0 .. 2^32 - 1
        v = torch.where(v >= 2 ** 31, v - 2 ** 32, v) if key == "u32" else v - 2 ** 31
        return v.to(torch.int32)
    v = ((x - 0.5) * 2.0 ** 63).to(torch.int64) * 2  # the signed range, ascending
    return v ^ (-(2 ** 63)) if key == "u64" else v


def _keys(key, n, dist, seed, g):
    """n keys of one distribution, in the key type's tensor (unsigned keys as
    their bit patterns)."""
    dt = KEY_DTYPE[key]
    if dist == "sorted":
        return _ascending(key, n, g)
    if key in ("f32", "f64"):
        if dist == "normal":
            return torch.randn(n, dtype=dt, device="cuda", generator=g)
        return torch.rand(n, dtype=dt, device="cuda", generator=g)
    if dist == "normal":  # around the middle of the range, deviation a sixteenth of it
        x = torch.randn(n, dtype=torch.float32, device="cuda", generator=g).clamp_(-7.9, 7.9)
        if dt == torch.int32:
            v = (x * 2.0 ** 28).to(torch.int32)
            return v ^ (-(2 ** 31)) if key == "u32" else v
        v = (x * 2.0 ** 60).to(torch.int64)
        v = v ^ torch.randint(0, 2 ** 36, (n,), dtype=torch.int64, device="cuda", generator=g)
        return v ^ (-(2 ** 63)) if key == "u64" else v
    if dist == "zipf":  # 2^20 distinct values, exponent 1.2
        k = batched.make_keys(n, "zipf-1.2", seed, torch.device("cuda"))
        return k if dt == torch.int64 else (k >> 32).to(torch.int32)
    if dt == torch.int32:
        return torch.randint(-(2 ** 31), 2 ** 31, (n,), dtype=torch.int32, device="cuda", generator=g)
    return batched.make_keys(n, "uniform", seed, torch.device("cuda"))


def _vals(val, n):
    """Payload: the position in the input (None without a payload)."""
    return None if val == "none" else torch.arange(n, dtype=VAL_DTYPE[val], device="cuda")


def _inputs(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    kind, key = case["kind"], case["key"]
    if kind == "sort":
        return {"keys": _keys(key, case["n"], case["dist"], seed, g), "vals": _vals(case["val"], case["n"])}
    if kind == "segments":
        lens = _lengths(case, seed)
        n = int(lens.sum())
        return {"lens": lens, "keys": _keys(key, n, case["dist"], seed, g), "vals": _vals(case["val"], n)}
    if kind == "ranges":
        # requests lie in a pool in shuffled order with gaps between them
        lens = _lengths(case, seed)
        order = np.random.default_rng(seed).permutation(len(lens))
        slot = (lens[order] + 63) // 64 * 64 + 64
        at = np.empty(len(lens), dtype=np.int64)
        at[order] = np.cumsum(slot) - slot
        pool = int(slot.sum())
        return {"lens": lens, "at": at, "keys": _keys(key, pool, case["dist"], seed, g),
                "vals": _vals(case["val"], pool)}
    if kind == "merge":
        a, b = _ascending(key, case["n0"], g), _ascending(key, case["n1"], g)
        v = _vals(case["val"], case["n0"] + case["n1"])
        return {"a": a, "b": b, "av": None if v is None else v[:case["n0"]], "bv": None if v is None else v[case["n0"]:]}
    sizes = [case["n"] // case["runs"] + (7 * j) % 64 for j in range(case["runs"])]
    return {"runs": [_ascending(key, m, g) for m in sizes]}


def prepare(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    kt = mgsort.key_type(case["key"])
    vt = mgsort.val_type(case.get("val", "none"))
    s.update(kind=kind, kt=kt)
    if kind in ("sort", "segments", "ranges"):
        s["keys_out"] = torch.empty_like(s["keys"])
        s["vals_out"] = None if s["vals"] is None else torch.empty_like(s["vals"])
    if kind == "sort":
        need = mgsort.lib.mgs_sort_temp_bytes(kt, vt, case["n"])
    elif kind in ("segments", "ranges"):
        lens = s["lens"]
        s["total"] = int(lens.sum())
        # the persisted tuning of this type and size, as the batching and
        # serving layers pass it
        found = tuning.lookup(kt, vt, s["total"])
        s["tuning"] = found[0] if found is not None else mgsort.Tuning()
        s["tuning"].max_segment_keys = int(lens.max())
        if kind == "segments":
            bounds = np.concatenate([[0], np.cumsum(lens)])
        else:
            bounds = np.stack([s["at"], s["at"] + lens], axis=1).reshape(-1)
        s["bounds"] = torch.from_numpy(np.ascontiguousarray(bounds, dtype=np.int64)).cuda()
        need = mgsort.lib.mgs_segmented_sort_temp_bytes_tuned(kt, vt, s["total"], len(lens), ctypes.byref(s["tuning"]))
    elif kind == "merge":
        s["out"] = torch.empty(case["n0"] + case["n1"], dtype=KEY_DTYPE[case["key"]], device="cuda")
        s["out_vals"] = None if s["av"] is None else torch.empty(s["out"].numel(), dtype=s["av"].dtype, device="cuda")
        need = mgsort.lib.mgs_merge_temp_bytes(kt, vt, case["n0"], case["n1"])
    else:
        total = sum(r.numel() for r in s["runs"])
        s["out"] = torch.empty(total, dtype=KEY_DTYPE[case["key"]], device="cuda")
        need = mgsort.lib.mgs_multiway_merge_temp_bytes(kt, len(s["runs"]), total)
    s["temp"] = mgsort.temp_buffer(need, "cuda")
    return s


def run(s):
    kind = s["kind"]
    if kind == "sort":
        mgsort.sort(s["kt"], s["keys"], s["vals"], keys_out=s["keys_out"], vals_out=s["vals_out"], temp=s["temp"])
        return {"keys": s["keys_out"], "vals": s["vals_out"]}
    if kind == "segments":
        mgsort.segmented_sort(s["kt"], s["keys"], s["bounds"], s["vals"], keys_out=s["keys_out"],
                              vals_out=s["vals_out"], max_total=s["total"], tuning=s["tuning"], temp=s["temp"])
        return {"keys": s["keys_out"], "vals": s["vals_out"]}
    if kind == "ranges":
        # the requests' data arrives in the pool, then one call sorts them all
        s["keys_out"].copy_(s["keys"])
        if s["vals"] is not None:
            s["vals_out"].copy_(s["vals"])
        mgsort.segmented_sort_ranges(s["kt"], s["keys_out"], s["bounds"], s["vals_out"], max_total=s["total"],
                                     tuning=s["tuning"], temp=s["temp"])
        return {"keys": s["keys_out"], "vals": s["vals_out"]}
    if kind == "merge":
        mgsort.merge(s["kt"], s["a"], s["b"], s["out"], s["av"], s["bv"], s["out_vals"], temp=s["temp"])
        return {"keys": s["out"], "vals": s["out_vals"]}
    mgsort.multiway_merge(s["kt"], s["runs"], s["out"], temp=s["temp"])
    return {"keys": s["out"]}


def work(case):
    kb = 4 if case["key"].endswith("32") else 8
    vb = {"none": 0, "u32": 4, "u64": 8}[case.get("val", "none")]
    if case["kind"] in ("segments", "ranges"):
        lo, hi = case["lo"], case["hi"]
        n = case["nseg"] * (2.0 ** hi - 2.0 ** lo) / ((hi - lo) * math.log(2.0))  # the mean total
    else:
        n = case["n0"] + case["n1"] if case["kind"] == "merge" else case["n"]
    # every record read once and written once; a sort does no arithmetic
    return {"bytes": 2.0 * n * (kb + vb), "flops": 0.0}


def exact(case, seed):
    """Sorted float keys in 64 bits (integer outputs are compared bit for bit)."""
    if case["key"] not in ("f32", "f64") or case["kind"] not in ("sort", "merge"):
        return None
    n = case["n"] if case["kind"] == "sort" else case["n0"] + case["n1"]
    if n > 1 << 27:
        return None
    s = _inputs(case, seed)
    keys = s["keys"] if case["kind"] == "sort" else torch.cat([s["a"], s["b"]])
    return {"keys": torch.sort(keys.double()).values, "vals": None}
