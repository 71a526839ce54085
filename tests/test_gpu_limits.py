"""Calls at the limits of a dispatch: more features than a packed node holds,
small and uneven shapes that a rule made for average ones must still take."""
import ctypes as C

import numpy as np
import pytest

import hessboost_amd as hb

pytestmark = pytest.mark.gpu


def _walked(trees, x, base):
    """The margins of finite rows x by the trees' own thresholds, one f32
    addition a tree."""
    out = np.full(len(x), base, np.float32)
    for t in trees:
        at = np.zeros(len(x), np.int64)
        for _ in range(len(t["left"])):
            left = t["left"][at]
            inner = left != -1
            if not inner.any():
                break
            go = x[np.arange(len(x)), t["split_feature"][at]] < t["split_cond"][at]
            at = np.where(inner, np.where(go, left, t["right"][at]), at)
        out = out + t["leaf_value"][at]
    return out


# the informative features are the last of more than a packed node's 2^15, and
# the features that those numbers' low 15 bits name hold something else; bins
# of u8 and of u16, trees decided on the device, by the host and best-first
@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("grow", ["device", "host", "lossguide"])
def test_trees_over_more_than_32768_features_walk_their_own_features(monkeypatch, wide, grow):
    rng = np.random.default_rng(7)
    n, f = 700, 33_000
    x = rng.integers(0, 2, (n, f)).astype(np.float32)
    x[:, 32_770:32_775] = rng.standard_normal((n, 5), dtype=np.float32)
    y = x[:, 32_770] + 2.0 * (x[:, 32_771] > 0.3) * x[:, 32_772] + 0.5 * x[:, 32_800]
    params = {"objective": "reg:squarederror", "max_depth": 3, "eta": 0.3, "max_bin": 500 if wide else 64}
    if grow == "lossguide":
        params.update(grow_policy="lossguide", max_leaves=6, max_depth=0)
    if grow == "host":
        monkeypatch.setenv("HBROCM_DEVICE_GROW", "0")
    engine = hb.DMatrix(x, label=y).engine(params["max_bin"])
    t = hb.Trainer(engine, params, y)
    t.boost(3)
    trees = t.trees()
    assert max(int(k["split_feature"].max()) for k in trees) >= 32_768
    assert np.array_equal(t.margins(), _walked(trees, x, t.base_score()[0]))


def _free_bytes():
    """The device's free memory, from the HIP runtime the library has loaded."""
    hip = C.CDLL("libamdhip64.so.7")
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def _fit(monkeypatch, x, y, params, device):
    monkeypatch.setenv("HBROCM_DEVICE_GROW", "1" if device else "0")
    engine = hb.DMatrix(x, label=y).engine(params["max_bin"])
    t = hb.Trainer(engine, params, y)
    free = _free_bytes()
    t.boost(2)
    return t.trees(), t.margins(), free - _free_bytes()


# few bins a feature beside one of many (a tile's sums take 128 KiB for every
# feature then), and many features of two bins (128 KiB for every 32): a deep
# level's nodes may not each take that much
@pytest.mark.parametrize("f,depth,widest,max_bin,nan", [
    (300, 10, 5_000, 5_000, 0.0), (2_000, 11, 2, 256, 0.0), (2_000, 12, 2, 256, 0.0), (33, 10, 2, 256, 0.0),
    (200, 10, 2, 256, 0.1)])
def test_deep_levels_of_few_bins_take_little_memory(monkeypatch, f, depth, widest, max_bin, nan):
    rng = np.random.default_rng(f + depth)
    n = 6_000
    x = rng.integers(0, 2, (n, f)).astype(np.float32)
    if widest > 2:
        x[:, 5] = rng.permutation(n).astype(np.float32)
    y = (x[:, :12] @ rng.standard_normal(12) + 0.1 * rng.standard_normal(n)).astype(np.float32)
    x[rng.random(x.shape) < nan] = np.nan
    params = {"objective": "reg:squarederror", "max_depth": depth, "eta": 0.3, "max_bin": max_bin}
    trees, margins, used = _fit(monkeypatch, x, y, params, True)
    want, want_margins, _ = _fit(monkeypatch, x, y, params, False)
    for a, b in zip(trees, want):
        for key in a:
            assert np.array_equal(a[key], b[key]), key
    assert np.array_equal(margins, want_margins)
    # slots, records and the tiles' partials; a partial a node would take 4 to 10 GB
    assert used <= 1 << 30, used


def _best_first(x, y, leaves, depth, rounds=2, max_bin=256):
    engine = hb.DMatrix(x, label=y).engine(max_bin)
    params = {"grow_policy": "lossguide", "max_depth": depth, "max_leaves": leaves, "eta": 0.3, "min_child_weight": 2.0}
    t = hb.Trainer(engine, params, y)
    free = _free_bytes()
    before = engine.counters()
    t.boost(rounds)
    after = engine.counters()
    return t, free - _free_bytes(), {k: after[k] - before[k] for k in after}


# 1,000 features of 256 bins: 4 MB a histogram slot. A depth limit of 4 leaves
# no more than 16; where the pops cannot be foreseen the unused splits stay
# within the leaves, and most pops then split nothing ahead
@pytest.mark.parametrize("leaves,depth,slots", [(0, 4, 2 * 16), (100, 0, 2 * 100), (3, 0, 2 * 3)])
def test_best_first_slots_stay_within_twice_the_leaves(leaves, depth, slots):
    rng = np.random.default_rng(leaves)
    x = rng.standard_normal((3_000, 1_000), dtype=np.float32)
    y = rng.standard_normal(3_000).astype(np.float32)
    t, used, counters = _best_first(x, y, leaves, depth)
    # 272 partials of 128 KiB a tile and 32 features, of 2 x 256 workgroups at most, and small records
    assert used <= slots * 1_000 * 256 * 16 + (160 << 20), used / 2**20
    taken = sum(int(np.sum(k["left"] >= 0)) for k in t.trees())
    # splits made: a root histogram a tree, then one for each split
    assert counters["hist_nodes"] - 2 <= 2 * taken


# a pool that holds a tree's leaves but not the splits ahead beside them: the
# same trees, none refused, and the counters of what the kept growth did
@pytest.mark.parametrize("noise", [0.1, 3.0])
@pytest.mark.parametrize("leaves,pool", [(60, 64), (127, 128), (32, 32)])
def test_a_full_slot_pool_grows_the_oracles_best_first_trees(monkeypatch, noise, leaves, pool):
    from oracle import oracle as O
    from tests.test_gpu_train import compare_trees

    monkeypatch.setenv("HBROCM_HIST_SLOTS", str(pool))
    rng = np.random.default_rng(leaves)
    x = rng.standard_normal((2_500, 20), dtype=np.float32)
    y = (x[:, 0] - x[:, 1] * x[:, 2] + noise * rng.standard_normal(2_500)).astype(np.float32)
    ref = O.Model(O.Dataset(x), y, O.params(grow_policy=O.GROW_LOSSGUIDE, max_depth=0, max_leaves=leaves,
                                            min_child_weight=2.0), 3)
    t, _, counters = _best_first(x, y, leaves, 0, rounds=3)
    compare_trees(t.trees(), ref.trees())
    assert np.max(np.abs(t.margins() - ref.margins().reshape(-1))) <= 1e-5
    assert counters["trees"] == 3


# rows of a few entries among which some are long: a wave of rows with none,
# with one, with as many long ones as short, ends of waves and of entries
@pytest.mark.parametrize("f,values", [(300, 3), (4_000, 2), (5_000, 9)])
@pytest.mark.parametrize("share", [0.0, 0.0005, 0.05, 0.6])
def test_uneven_sparse_rows_sum_every_entry(f, values, share):
    rng = np.random.default_rng(f + int(share * 1e4))
    n = 3_001
    lens = rng.integers(0, 6, n)
    lens[rng.random(n) < share] = f - rng.integers(0, 3)
    lens[-1] = f
    ptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    cols = np.concatenate([np.sort(rng.choice(f, k, replace=False)) for k in lens]).astype(np.int32)
    vals = rng.integers(0, values, ptr[-1]).astype(np.float32)
    data = hb.DMatrix((ptr, cols, vals), n_cols=f)
    engine = data.engine()
    pairs = rng.integers(-8, 9, (n, 2)).astype(np.float32)  # every sum exact
    engine.prepare(pairs)
    row_ptr, row_bins = data.index().row_bins()
    counts = np.diff(row_ptr.astype(np.int64))
    for rows in (np.arange(n), np.flatnonzero(rng.random(n) < 0.3), np.array([n - 1]), np.arange(n - 65, n)):
        hist = engine.build(rows)
        inside = np.isin(np.repeat(np.arange(n), counts), rows)
        for c in (0, 1):
            want = np.bincount(row_bins[inside], weights=np.repeat(pairs[:, c], counts)[inside].astype(np.float64),
                               minlength=len(hist))
            assert np.array_equal(hist[:, c], want)


def test_the_reorders_second_copy_of_the_rows_is_given_back(monkeypatch):
    """After a reordered fit the copy stays for the next such trainer, and
    goes with the first call of another kind."""
    monkeypatch.setenv("HBROCM_ROW_ORDER_MIN_ROWS", "1000")
    rng = np.random.default_rng(4)
    n = 1_000_000
    x = rng.standard_normal((n, 20), dtype=np.float32)
    y = (x[:, 0] + x[:, 1] * x[:, 2] > 0).astype(np.float32)
    engine = hb.DMatrix(x, label=y).engine()
    params = {"objective": "binary:logistic", "max_depth": 4}
    copies = n * (32 + 20 + 4 * 2)  # the rows, the columns, and each row's two places, at least

    def fit(**more):
        t = hb.Trainer(engine, dict(params, **more), y)
        t.boost(3)
        return t.trees(), t.margins()

    first = fit()
    assert engine.counters()["row_orders"] == 1
    free = _free_bytes()
    again = fit()
    assert abs(_free_bytes() - free) < copies // 4
    for call in (lambda: engine.load_margins(np.zeros(n, np.float32), 1),
                 lambda: fit(grow_policy="lossguide", max_leaves=7, max_depth=0)):
        last = fit()
        free = _free_bytes()
        call()
        assert _free_bytes() - free > copies, (_free_bytes() - free) / 2**20
    for a, b in zip(first[0] + first[0], again[0] + last[0]):
        for key in a:
            assert np.array_equal(a[key], b[key])
    assert np.array_equal(first[1], last[1]) and np.array_equal(first[1], again[1])
