"""The workgroup sort in LDS (block_sort.hpp) through the entry points that
use it: sizes at the edges of its item slots and pieces, keys whose top
differing bits tie (neighbour fix-up, and the passes over all bits where the
ties are long), bit for bit against the oracle."""
import numpy as np
import pytest

import pyoracle as O
from helpers import KEY_NAME, from_dev, random_keys, random_vals, to_dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mg():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import mgsort
    return mgsort


def tied_keys(kt, n, rng, dist):
    """uniform; pairs: every key about twice; clustered: 5 far apart values
    plus small offsets, so that in 8-byte keys the top 27 differing bits leave
    long groups in disorder; lone: clustered with one key at the bottom of the range."""
    if dist == "uniform":
        return random_keys(kt, n, rng)
    bd = O.BITS_DTYPE[kt]
    nbits = 32 if bd == np.uint32 else 64
    if dist == "pairs":
        pool = random_keys(kt, max(n // 2, 1), rng, "nonneg")
        return pool[rng.integers(0, pool.size, size=n)]
    top = rng.integers(0, 2**16, size=5).astype(np.uint64)[rng.integers(0, 5, size=n)] << np.uint64(nbits - 20)
    k = (top | rng.integers(0, 2**11, size=n).astype(np.uint64)).astype(bd)
    if dist == "lone":
        k[n // 2] = 0
    return k


@pytest.mark.parametrize("kt,k", [(O.K_U32, 3), (O.K_F32, 5), (O.K_I32, 40), (O.K_U64, 4), (O.K_U64, 9), (O.K_F64, 12),
                                  (O.K_I64, 100)], ids=lambda v: str(v))
@pytest.mark.parametrize("dist", ["uniform", "pairs", "clustered", "lone"])
@pytest.mark.parametrize("total", [1, 511, 513, 8191, 8193, 70_001, 400_000])
def test_multiway_pieces(mg, kt, k, dist, total):
    import torch
    rng = np.random.default_rng(total + 11 * k + kt)
    cuts = np.sort(rng.integers(0, total + 1, size=k - 1))
    lens = np.diff(np.concatenate([[0], cuts, [total]]))
    keys = tied_keys(kt, total, rng, dist)
    runs, at = [], 0
    for n in lens:
        r = keys[at:at + n]
        runs.append(np.ascontiguousarray(r[np.argsort(O.encode(kt, r), kind="stable")]))
        at += n
    expect = O.sort(kt, np.concatenate(runs))[0]
    out = torch.empty(total, dtype=to_dev(expect).dtype, device="cuda")
    temp = mg.temp_buffer(mg.lib.mgs_multiway_merge_temp_bytes(kt, k, total), "cuda")
    mg.multiway_merge(KEY_NAME[kt], [to_dev(r) for r in runs], out, temp=temp)
    assert mg.temp_status(temp) == 0
    assert np.array_equal(from_dev(out, expect.dtype), expect)


@pytest.mark.parametrize("lens", [(1,), (3840,), (3841, 0), (0, 3839), (100_003, 77)], ids=str)
@pytest.mark.parametrize("portions", [0, 1, 5])
def test_one_or_two_runs(mg, lens, portions):
    """One or two runs take the merge path, with the stretches' ends on its
    tile boundaries."""
    import torch
    rng = np.random.default_rng(sum(lens))
    runs = [np.sort(random_keys(O.K_U32, n, rng, "lowbits")) for n in lens]
    expect = np.sort(np.concatenate(runs))
    out = torch.empty(expect.size, dtype=torch.int32, device="cuda")
    temp = mg.temp_buffer(mg.lib.mgs_multiway_merge_temp_bytes(O.K_U32, len(lens), expect.size), "cuda")
    ends = mg.multiway_merge("u32", [to_dev(r) for r in runs], out, temp=temp, portions=portions)
    assert mg.temp_status(temp) == 0
    assert portions == 0 or (len(ends) == portions and ends[-1] == expect.size and ends == sorted(ends))
    assert np.array_equal(from_dev(out, np.uint32), expect)


@pytest.mark.parametrize("kt,k,total", [(O.K_U32, 256, 12_500_000), (O.K_U32, 256, 12_900_000),
                                        (O.K_U64, 200, 14_000_000), (O.K_F32, 8, 13_000_000)], ids=lambda v: str(v))
@pytest.mark.parametrize("dist", ["uniform", "pairs"])
def test_multiway_split_levels(mg, kt, k, total, dist):
    """Around 2^19 searches for the pieces' bounds, from where these take two levels."""
    import torch
    rng = np.random.default_rng(total + kt)
    cuts = np.sort(rng.integers(0, total + 1, size=k - 1))
    cuts = np.concatenate([[0], cuts, [total]])
    keys = tied_keys(kt, total, rng, dist)
    runs = [O.sort(kt, np.ascontiguousarray(keys[a:b]))[0] for a, b in zip(cuts[:-1], cuts[1:])]
    expect = O.sort(kt, np.concatenate(runs))[0]
    out = torch.empty(total, dtype=to_dev(expect).dtype, device="cuda")
    temp = mg.temp_buffer(mg.lib.mgs_multiway_merge_temp_bytes(kt, k, total), "cuda")
    mg.multiway_merge(KEY_NAME[kt], [to_dev(r) for r in runs], out, temp=temp)
    assert mg.temp_status(temp) == 0
    assert np.array_equal(from_dev(out, expect.dtype), expect)


@pytest.mark.parametrize("kt", [O.K_U32, O.K_F64], ids=str)
@pytest.mark.parametrize("k", [1, 2, 3, 9])
def test_empty_runs(mg, kt, k):
    """Runs that are all empty merge with the scratch that their size asks for."""
    import torch
    runs = [torch.empty(0, dtype=torch.int32 if kt == O.K_U32 else torch.int64, device="cuda") for _ in range(k)]
    out = torch.empty(1, dtype=runs[0].dtype, device="cuda")
    temp = mg.temp_buffer(mg.lib.mgs_multiway_merge_temp_bytes(kt, k, 0), "cuda")
    assert mg.multiway_merge(KEY_NAME[kt], runs, out, temp=temp, portions=3) == [0, 0, 0]
    assert mg.temp_status(temp) == 0


RECORDS = [(O.K_U64, None), (O.K_I64, np.uint32), (O.K_U64, np.uint64), (O.K_U32, np.uint32), (O.K_I32, np.uint64)]


def run_sort(mg, kt, vdt, keys, rng, inplace):
    """Sorts on the device, checks status and oracle, returns the path."""
    import torch
    n = keys.size
    vals = None if vdt is None else random_vals(vdt, n, rng)
    ek, ev = O.sort(kt, keys, vals)
    vt = mg.VAL_NONE if vdt is None else (mg.VAL_U32 if vdt == np.uint32 else mg.VAL_U64)
    temp = mg.temp_buffer(mg.lib.mgs_sort_temp_bytes(kt, vt, n), "cuda")
    dk, dv = to_dev(keys), to_dev(vals)
    ok = dk if inplace else torch.empty_like(dk)
    ov = dv if inplace or dv is None else torch.empty_like(dv)
    mg.sort(KEY_NAME[kt], dk, dv, keys_out=ok, vals_out=ov, temp=temp)
    assert mg.temp_status(temp) == 0
    path = mg.lib.mgs_sort_path(kt, vt, n, mg._ptr(temp), temp.numel(), None)
    assert np.array_equal(from_dev(ok, keys.dtype), ek)
    if vdt is not None:
        assert np.array_equal(from_dev(ov, vals.dtype), ev)
    if not inplace:
        assert np.array_equal(from_dev(dk, keys.dtype), keys)
    return path


@pytest.mark.parametrize("kt,vdt", RECORDS, ids=lambda v: str(v))
@pytest.mark.parametrize("n", [8195, 100_003, (1 << 20) + 77])
@pytest.mark.parametrize("dist", ["uniform", "sorted", "reverse", "few", "lowbits", "runs", "nonneg", "stray",
                                  "clustered", "pairs"])
def test_three_pass_wide_forced(mg, kt, vdt, n, dist, monkeypatch):
    """The three-pass path of wider records, tried at any size: uniform keys
    take it, keys that crowd its sub-buckets or leave the sample's shared
    bits hand over to the LSD passes; the result is the oracle's either way,
    in place and out of place."""
    monkeypatch.setenv("MGS_MSD_MIN", "0")
    rng = np.random.default_rng(n + 5 * kt)
    keys = tied_keys(kt, n, rng, dist) if dist in ("clustered", "pairs") else random_keys(kt, n, rng, dist)
    path = run_sort(mg, kt, vdt, keys, rng, inplace=bool(n & 1))
    assert path in (2, 3)
    if dist in ("uniform", "nonneg"):
        assert path == 3


@pytest.mark.parametrize("kt,vdt", RECORDS, ids=lambda v: str(v))
@pytest.mark.parametrize("dist", ["uniform", "sorted", "skewed", "nonneg"])
def test_three_pass_wide_default(mg, kt, vdt, dist):
    """Without environment: 8-byte keys from 2^23 records on, 4-byte keys
    with payloads from 2^24."""
    rng = np.random.default_rng(3 + kt)
    keys = random_keys(kt, (1 << (23 if O.BITS_DTYPE[kt] == np.uint64 else 24)) + 4321, rng, dist)
    path = run_sort(mg, kt, vdt, keys, rng, inplace=False)
    assert path in (2, 3)
    if dist == "uniform":
        assert path == 3


def test_three_pass_wide_small_scratch(mg):
    """Scratch that only fits the LSD passes still sorts."""
    rng = np.random.default_rng(8)
    n = (1 << 23) + 9
    keys = random_keys(O.K_U64, n, rng)
    temp = mg.temp_buffer(n * 8 + (4 << 20), "cuda")
    assert temp.numel() < mg.lib.mgs_sort_temp_bytes(O.K_U64, mg.VAL_NONE, n)
    dk = to_dev(keys)
    mg.sort("u64", dk, temp=temp)
    assert mg.temp_status(temp) == 0
    assert mg.lib.mgs_sort_path(O.K_U64, mg.VAL_NONE, n, mg._ptr(temp), temp.numel(), None) == 2
    assert np.array_equal(from_dev(dk, np.uint64), np.sort(keys))


def scaled_keys(kt, n, rng, dist):
    """heavy: one value in 60% of the places; nested: a third each uniform
    over the whole range, over its 2^-20th and its 2^-40th (4-byte keys: 2^-10th,
    2^-20th), which outlasts two levels of splits; edge: the range's ends and
    254 to 256 consecutive values."""
    bd = O.BITS_DTYPE[kt]
    nbits = 32 if bd == np.uint32 else 64
    k = random_keys(kt, n, rng).view(bd) if dist != "edge" else None
    if dist == "heavy":
        k[rng.random(n) < 0.6] = k[0]
    elif dist == "nested":
        if kt in (O.K_F32, O.K_F64):
            k = random_keys(kt, n, rng, "nonneg").view(bd)
        k = k >> (rng.integers(0, 3, size=n) * (nbits // 3 - 1)).astype(bd)
    elif dist == "edge":
        k = (bd(1) << bd(nbits - 3)) + rng.integers(0, 254 + n % 3, size=n).astype(bd)
        k[n // 2], k[n // 3] = 0, bd(1) << bd(nbits - 2)
    return k


@pytest.mark.parametrize("kt,vdt", [(O.K_U32, None), (O.K_F32, np.uint32), (O.K_I64, None), (O.K_U64, np.uint32),
                                    (O.K_F64, np.uint64)], ids=lambda v: str(v))
@pytest.mark.parametrize("dist", ["uniform", "heavy", "nested", "edge", "sorted"])
def test_splits(mg, kt, vdt, dist):
    """Segments at the edges of what one workgroup sorts (512 x 7, 10, 14, 16
    records), of the scatter's tiles, and long enough for two and three
    levels of splits."""
    import torch
    rng = np.random.default_rng(kt + 17)
    lens = [0, 1, 256, 257] + [512 * i + d for i in (7, 10, 14, 16, 20, 32) for d in (-1, 0, 1)]
    lens += [70_001, 300_002] + ([1_100_003] if dist in ("uniform", "nested") else [])
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    make = scaled_keys if dist in ("heavy", "nested", "edge") else random_keys
    parts = [make(kt, n, rng, dist).view(O.BITS_DTYPE[kt]) if n else np.zeros(0, O.BITS_DTYPE[kt]) for n in lens]
    keys = np.concatenate(parts).view(random_keys(kt, 1, rng).dtype)
    vals = None if vdt is None else random_vals(vdt, keys.size, rng)
    ek, ev = O.segmented_sort(kt, keys, off, vals)
    dk, dv = to_dev(keys), to_dev(vals)
    mg.segmented_sort(KEY_NAME[kt], dk, torch.from_numpy(off.view(np.int64)).cuda(), dv)
    torch.cuda.synchronize()
    assert np.array_equal(from_dev(dk, O.BITS_DTYPE[kt]), ek.view(O.BITS_DTYPE[kt]))
    if vdt is not None:
        assert np.array_equal(from_dev(dv, vdt), ev)


@pytest.mark.parametrize("kt,vdt,most", [(O.K_U32, None, 24576), (O.K_F32, np.uint32, 15360), (O.K_I64, None, 15360),
                                         (O.K_U64, np.uint32, 10240), (O.K_F64, np.uint64, 7168)], ids=lambda v: str(v))
@pytest.mark.parametrize("dist", ["uniform", "heavy", "nested"])
def test_middle_sizes(mg, kt, vdt, most, dist):
    """One array around the longest that one workgroup sorts, and by splits."""
    rng = np.random.default_rng(kt + most)
    for n in (2047, 2049, 4095, 4097, most - 1, most, most + 1, 200_003):
        keys = scaled_keys(kt, n, rng, dist).view(random_keys(kt, 1, rng).dtype)
        assert run_sort(mg, kt, vdt, keys, rng, inplace=bool(n & 1)) == (1 if n <= most else 4)


@pytest.mark.parametrize("kt,vdt,end", [(O.K_F32, None, 23), (O.K_U32, None, 22), (O.K_U32, np.uint32, 23),
                                        (O.K_I64, np.uint32, 23)], ids=lambda v: str(v))
def test_splits_end(mg, kt, vdt, end):
    """Splits below 2^23 records (4-byte integers alone: 2^22; not doubles),
    the passes from there on."""
    rng = np.random.default_rng(kt)
    for n in (1 << end) - 1, 1 << end:
        path = run_sort(mg, kt, vdt, random_keys(kt, n, rng), rng, inplace=False)
        assert (path == 4) == (n < 1 << end)


@pytest.mark.parametrize("kt,vdt", [(O.K_U32, None), (O.K_F64, np.uint32)], ids=lambda v: str(v))
@pytest.mark.parametrize("dist", ["uniform", "heavy", "nested"])
def test_splits_chunks(mg, kt, vdt, dist):
    """Segments of more than 1024 tiles (of 4096 and 6144 records), whose
    tiles are counted in chunks of 64, beside short ones."""
    import torch
    rng = np.random.default_rng(kt + 23)
    long = 4096 * 1100 if kt == O.K_U32 else 6144 * 1100
    lens = [9, long + 1, 70_001, long // 3, 20_000, 20_000, long - 64 * 4096 - 1]
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    keys = np.concatenate([scaled_keys(kt, n, rng, dist) for n in lens]).view(random_keys(kt, 1, rng).dtype)
    vals = None if vdt is None else random_vals(vdt, keys.size, rng)
    ek, ev = O.segmented_sort(kt, keys, off, vals)
    dk, dv = to_dev(keys), to_dev(vals)
    mg.segmented_sort(KEY_NAME[kt], dk, torch.from_numpy(off.view(np.int64)).cuda(), dv, tuning=mg.Tuning(2, 0, 0, 0))
    torch.cuda.synchronize()
    assert np.array_equal(from_dev(dk, O.BITS_DTYPE[kt]), ek.view(O.BITS_DTYPE[kt]))
    if vdt is not None:
        assert np.array_equal(from_dev(dv, vdt), ev)


@pytest.mark.parametrize("dist", ["uniform", "sorted", "few"])
def test_doubles_take_splits(mg, dist):
    rng = np.random.default_rng(6)
    keys = random_keys(O.K_F64, (1 << 24) + 77, rng, dist)
    assert run_sort(mg, O.K_F64, None, keys, rng, inplace=True) == 4


def skewed_keys(kt, n, rng, dist):
    """Keys that even steps do not divide: log: every binary order of
    magnitude equally often; zipf: small counts, 1 in 87% of the places (10%
    in 4-byte keys); near: 1 - eps over 50 orders of eps; four: four values
    2^-30, 2^-20 and 2^-10 apart; shares: 55% 0, 25% 1, 12% 2, the rest
    spread; geometric: counts, halving; single: one value; ends: 40% the lowest
    and 30% the highest key that sorts, the rest log."""
    bd = O.BITS_DTYPE[kt]
    fd = np.float32 if bd == np.uint32 else np.float64
    u = rng.random(n)
    if dist == "ends":
        k = skewed_keys(kt, n, rng, "log")
        top = bd(~bd(0)) if kt in (O.K_U32, O.K_U64) else bd(~bd(0)) >> bd(1)
        k[u < 0.3] = top  # (of floats the NaN that sorts last)
        k[u > 0.6] = ~top
        return k
    if dist == "log":
        x = np.exp2(u * (31 if bd == np.uint32 else 63))
    elif dist == "zipf":
        x = np.minimum(np.maximum(u, 1e-9) ** (-5 if bd == np.uint64 else -2), 2.0**20)
    elif dist == "near":
        x = 1 - np.exp2(-50 * u)
    elif dist == "four":
        x = np.array([1, 1 + 2.0**-30, 1 + 2.0**-20, 1 + 2.0**-10])[rng.integers(0, 4, n)]
    elif dist == "shares":
        x = np.where(u < 0.55, 0, np.where(u < 0.8, 1, np.where(u < 0.92, 2, rng.random(n) * 1000)))
    elif dist == "geometric":
        x = np.floor(-np.log2(1 - u)) + 1
    else:
        x = np.full(n, 3.0)
    return x.astype(fd).view(bd) if kt in (O.K_F32, O.K_F64) else x.astype(bd)


def left_to_one_workgroup(temp):
    """How many ranges the last level of splits left to a workgroup each (the
    fourth word of the scratch)."""
    return int(from_dev(temp[12:16], np.uint32)[0])


SKEWED = [(kt, vdt, d) for kt, vdt, ds in ((O.K_U64, None, "log zipf single ends"), (O.K_I32, np.uint32, "log zipf ends"),
                                           (O.K_U64, np.uint64, "log zipf"), (O.K_F32, None, "near shares geometric ends"),
                                           (O.K_F64, np.uint32, "near four shares geometric log single ends"))
          for d in ds.split()]


@pytest.mark.parametrize("kt,vdt,dist", SKEWED, ids=lambda v: str(v))
@pytest.mark.parametrize("n", [200_003, 1 << 20, (1 << 23) - 1])
def test_splits_divide_skewed_keys(mg, kt, vdt, dist, n):
    """However the keys are distributed, the levels bring the children to what
    one workgroup sorts in LDS: none is left to one that streams it."""
    import torch
    rng = np.random.default_rng(n + kt)
    keys = skewed_keys(kt, n, rng, dist)
    vals = None if vdt is None else random_vals(vdt, n, rng)
    vt = mg.VAL_NONE if vdt is None else (mg.VAL_U32 if vdt == np.uint32 else mg.VAL_U64)
    for inplace in (False, True):
        temp = mg.temp_buffer(mg.lib.mgs_sort_temp_bytes(kt, vt, n), "cuda")
        dk, dv = to_dev(keys), to_dev(vals)
        ok = dk if inplace else torch.empty_like(dk)
        ov = dv if inplace or dv is None else torch.empty_like(dv)
        mg.sort(KEY_NAME[kt], dk, dv, keys_out=ok, vals_out=ov, temp=temp)
        path = mg.lib.mgs_sort_path(kt, vt, n, mg._ptr(temp), temp.numel(), None)
        assert path == (2 if kt == O.K_I32 and n < 3 << 17 else 4)
        assert mg.temp_status(temp) == 0
        assert path == 2 or left_to_one_workgroup(temp) == 0
        ek, ev = O.sort(kt, keys, vals)
        assert np.array_equal(from_dev(ok, keys.dtype), ek)
        if vdt is not None:
            assert np.array_equal(from_dev(ov, vdt), ev)


@pytest.mark.parametrize("kt,vdt,dist", [v for v in SKEWED if v[1] != np.uint64], ids=lambda v: str(v))
def test_segments_of_skewed_keys(mg, kt, vdt, dist):
    """The same for segments of all lengths, each variant of the scatter."""
    import torch
    rng = np.random.default_rng(kt + 31)
    lens = [0, 3, 300, 5119, 8193, 70_001, 300_002, 20_000, 1_100_003, 9000]
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    keys = np.concatenate([skewed_keys(kt, n, rng, dist) for n in lens])
    vals = None if vdt is None else random_vals(vdt, keys.size, rng)
    vt = mg.VAL_NONE if vdt is None else mg.VAL_U32
    ek, ev = O.segmented_sort(kt, keys, off, vals)
    for variant in range(mg.lib.mgs_segmented_variant_count()):
        dk, dv = to_dev(keys), to_dev(vals)
        temp = mg.temp_buffer(mg.lib.mgs_segmented_sort_temp_bytes(kt, vt, keys.size, len(lens)) * 2, "cuda")
        mg.segmented_sort(KEY_NAME[kt], dk, torch.from_numpy(off.view(np.int64)).cuda(), dv,
                          tuning=mg.Tuning(variant, 0, 0, 0), temp=temp)
        assert mg.temp_status(temp) == 0
        assert left_to_one_workgroup(temp) == 0
        assert np.array_equal(from_dev(dk, keys.dtype), ek)
        if vdt is not None:
            assert np.array_equal(from_dev(dv, vdt), ev)


@pytest.mark.parametrize("vdt", [np.uint32, np.uint64], ids=str)
@pytest.mark.parametrize("dist", ["uniform", "nested", "heavy"])
def test_doubles_with_payloads_take_splits(mg, vdt, dist):
    rng = np.random.default_rng(16)
    n = (1 << 23) + 12_345
    keys = scaled_keys(O.K_F64, n, rng, dist) if dist != "uniform" else random_keys(O.K_F64, n, rng)
    assert run_sort(mg, O.K_F64, vdt, keys, rng, inplace=False) == 4


@pytest.mark.parametrize("n,path", [(3584 * (254 * 254 // 8 * 7) - 1, 4), (3584 * (254 * 254 // 8 * 7), 2)], ids=str)
def test_doubles_end_of_splits(mg, n, path):
    """16-byte records on both sides of the longest that sorts by splits,
    checked on the device: ascending, the payloads (places) with their keys, in
    order where keys are equal."""
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    k = torch.floor(torch.randn(n, dtype=torch.float64, device="cuda", generator=g) * 2.0**20)
    v = torch.arange(n, dtype=torch.int64, device="cuda")
    temp = mg.temp_buffer(mg.lib.mgs_sort_temp_bytes(O.K_F64, mg.VAL_U64, n), "cuda")
    ko, vo = torch.empty_like(k), torch.empty_like(v)
    mg.sort("f64", k, v, keys_out=ko, vals_out=vo, temp=temp)
    assert mg.lib.mgs_sort_path(O.K_F64, mg.VAL_U64, n, mg._ptr(temp), temp.numel(), None) == path
    assert mg.temp_status(temp) == 0
    assert path != 4 or left_to_one_workgroup(temp) == 0
    same = ko[1:] == ko[:-1]
    assert bool(((ko[1:] > ko[:-1]) | (same & (vo[1:] > vo[:-1]))).all())
    assert torch.equal(k[vo], ko)


@pytest.mark.parametrize("kt,dist", [(O.K_U64, "log"), (O.K_U32, "log"), (O.K_F64, "near"), (O.K_U64, "zipf")],
                         ids=lambda v: str(v))
@pytest.mark.parametrize("n", [2000, 6999])
def test_crowded_windows(mg, kt, dist, n):
    """Keys of which many share a window value: right, and by the passes over
    all bits (at most three times the window's, so five times a sort of uniform
    keys leaves room for the clock) instead of walks through long groups."""
    import torch
    rng = np.random.default_rng(n + kt)
    us = {}
    for d in ("uniform", dist):
        keys = random_keys(kt, n, rng) if d == "uniform" else skewed_keys(kt, n, rng, d)
        dk = to_dev(keys)
        ok = torch.empty_like(dk)
        temp = mg.temp_buffer(mg.lib.mgs_sort_temp_bytes(kt, mg.VAL_NONE, n), "cuda")
        begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        best = float("inf")
        for _ in range(8):
            begin.record()
            for _ in range(50):
                mg.sort(KEY_NAME[kt], dk, keys_out=ok, temp=temp)
            end.record()
            end.synchronize()
            best = min(best, begin.elapsed_time(end))
        us[d] = best * 20
        assert np.array_equal(from_dev(ok, keys.dtype), O.sort(kt, keys)[0])
    assert us[dist] < 5 * us["uniform"], us


@pytest.mark.parametrize("kt,vdt,n,path", [(O.K_U32, np.uint32, (1 << 16) - 1, 4), (O.K_I32, np.uint32, 1 << 16, 2),
                                           (O.K_I32, np.uint64, (3 << 17) - 1, 2), (O.K_U32, np.uint64, 3 << 17, 4),
                                           (O.K_U32, np.uint64, (9 << 17) - 1, 4), (O.K_I32, np.uint64, 9 << 17, 2),
                                           (O.K_U32, np.uint32, 9 << 17, 4), (O.K_F32, np.uint32, (13 << 15) - 1, 4),
                                           (O.K_F32, np.uint64, 13 << 15, 2), (O.K_F32, np.uint32, (5 << 18) - 1, 2),
                                           (O.K_F32, np.uint64, 5 << 18, 4),
                                           (O.K_U32, None, 1 << 16, 4)], ids=lambda v: str(v))
def test_pairs_between_splits(mg, kt, vdt, n, path):
    """4-byte keys with payloads on both sides of the sizes that the LSD passes
    sort faster than splits."""
    rng = np.random.default_rng(n)
    assert run_sort(mg, kt, vdt, random_keys(kt, n, rng), rng, inplace=False) == path


def sample_places(n):
    """Where a range of n records is sampled (sort_sample in segmented.hip)."""
    m = np.uint64(0xFFFFFFFF)
    t = np.arange(255, dtype=np.uint64)
    a, b = np.uint64(n) * t // np.uint64(255), np.uint64(n) * (t + np.uint64(1)) // np.uint64(255)
    h = ((t + np.uint64(1)) * np.uint64(0x9E3779B9) & m) ^ np.uint64(n)
    h = (h ^ (h >> np.uint64(16))) * np.uint64(0x85EBCA6B) & m
    h = (h ^ (h >> np.uint64(13))) * np.uint64(0xC2B2AE35) & m
    return (a + ((h ^ (h >> np.uint64(16))) * (b - a) >> np.uint64(32))).astype(np.int64)


@pytest.mark.parametrize("kt,vdt", [(O.K_U32, None), (O.K_I32, np.uint64), (O.K_U64, np.uint32), (O.K_I64, None),
                                    (O.K_U64, np.uint64)], ids=lambda v: str(v))
@pytest.mark.parametrize("values", [1, 2000])
def test_long_children(mg, kt, vdt, values):
    """Keys made against the sample: on both levels it sees evenly spread keys
    only, and all others lie close together, so that one child (or two, across a
    step) is left to a workgroup that streams it; of one value, or not."""
    import torch
    n, bd = 90_001, O.BITS_DTYPE[kt]
    nbits = 32 if bd == np.uint32 else 64
    rng = np.random.default_rng(kt + values)
    mid = np.uint64(3 << (nbits - 3))
    k = mid + rng.integers(0, values, size=n).astype(np.uint64)
    first = sample_places(n)
    rest = np.setdiff1d(np.arange(n), first)
    # the second level's range is the first's fullest step: all but its sample
    k[rest[sample_places(rest.size)]] = mid - np.uint64(1 << 20) + np.arange(255, dtype=np.uint64) * np.uint64(1 << 13)
    spread = np.arange(255, dtype=np.uint64) * np.uint64((1 << nbits) // 255)
    near = np.abs(spread.astype(np.float64) - float(mid)) < 2.0**nbits / 100  # (not in that step)
    k[first] = np.where(near, np.uint64(7), spread)
    keys = k.astype(bd) ^ (bd(1) << bd(nbits - 1) if kt in (O.K_I32, O.K_I64) else bd(0))
    vals = None if vdt is None else random_vals(vdt, n, rng)
    off = np.array([0, n], dtype=np.uint64)
    ek, ev = O.segmented_sort(kt, keys, off, vals)
    dk, dv = to_dev(keys), to_dev(vals)
    vt = mg.VAL_NONE if vdt is None else (mg.VAL_U32 if vdt == np.uint32 else mg.VAL_U64)
    temp = mg.temp_buffer(mg.lib.mgs_segmented_sort_temp_bytes(kt, vt, n, 1), "cuda")
    mg.segmented_sort(KEY_NAME[kt], dk, torch.from_numpy(off.view(np.int64)).cuda(), dv, temp=temp)
    assert mg.temp_status(temp) == 0
    assert left_to_one_workgroup(temp) in (1, 2)
    assert np.array_equal(from_dev(dk, bd), ek.view(bd))
    if vdt is not None:
        assert np.array_equal(from_dev(dv, vdt), ev)
