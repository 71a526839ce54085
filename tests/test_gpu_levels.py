"""The kernels of a device-grown level at the sizes where they can go wrong
(edges of tiles, remainders, the smallest and largest of their ranges): trees
and margins against growth decided by the host, level by level, whose
kernels share none of them, bit for bit."""
import numpy as np
import pytest

import hessboost_amd as hb

pytestmark = pytest.mark.gpu


def _fit(x, y, params, rounds, weight=None):
    engine = hb.DMatrix(x, label=y).engine(params.get("max_bin", 256))
    t = hb.Trainer(engine, params, y, weight)
    engine.set_profiling(True)
    t.boost(rounds)
    launches = {k: v[1] for k, v in engine.kernel_stats().items()}
    engine.set_profiling(False)
    return t.trees(), t.margins(), launches


def _same(a, b):
    (ta, ma, _), (tb, mb, _) = a, b
    assert len(ta) == len(tb)
    for i, (p, q) in enumerate(zip(ta, tb)):
        for key in p:
            assert np.array_equal(p[key], q[key]), (i, key)
    assert np.array_equal(ma.view(np.uint32), mb.view(np.uint32))


def _data(n, f, nan, seed, classes=0):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((n, f), dtype=np.float32)
    s = x[:, 0] - 0.5 * x[:, 1 % f] * x[:, 2 % f]
    if classes:
        y = np.clip(np.floor(s * 0.7 + classes / 2), 0, classes - 1)
    else:
        y = s > 0
    if nan:
        x[rng.random(x.shape) < nan] = np.nan
    return x, y.astype(np.float32)


def _both(monkeypatch, x, y, params, rounds, weight=None):
    device = _fit(x, y, params, rounds, weight)
    monkeypatch.setenv("HBROCM_DEVICE_GROW", "0")
    host = _fit(x, y, params, rounds, weight)
    return device, host


# tiles of 2,048, 4,096 and 8,192 rows (up to 2^19 and 2^21 rows, and beyond)
@pytest.mark.parametrize("n,f,nan,classes", [
    (1, 3, 0.0, 0), (63, 3, 0.0, 0), (2047, 5, 0.1, 0), (2048, 5, 0.0, 0), (2049, 33, 0.1, 0), (4097, 4, 0.0, 3),
    (2**19 + 1, 4, 0.0, 0), (2**19 + 4095, 4, 0.1, 0), (2**21 + 8191, 3, 0.0, 0), (700_001, 3, 0.0, 3),
])
def test_one_pass_partition_gives_the_host_levels_trees(monkeypatch, n, f, nan, classes):
    x, y = _data(n, f, nan, seed=n, classes=classes)
    params = {"objective": "multi:softprob" if classes else "binary:logistic", "max_depth": 5, "eta": 0.3,
              "base_score": 0.5}
    if classes:
        params["num_class"] = classes
    device, host = _both(monkeypatch, x, y, params, 2)
    assert device[2].get("hbr_part_move", 0) > 0 and "hbr_part_count" not in device[2]
    _same(device, host)


# few rows (one tile), about one tile's worth, one wave of tiles and beyond,
# dense groups of 32 features (one and several), 16-bit bins and sparse rows
@pytest.mark.parametrize("n", [1, 255, 257, 5_000, 60_001, 300_000])
@pytest.mark.parametrize("f,bins,density", [(7, 256, 1.0), (40, 256, 1.0), (20, 400, 1.0), (60, 256, 0.1)])
def test_histogram_tiles_sum_every_row(n, f, bins, density):
    rng = np.random.default_rng(n + f)
    x = rng.standard_normal((n, f), dtype=np.float32)
    if density < 1.0:
        x[rng.random(x.shape) >= density] = np.nan
    engine = hb.DMatrix(x).engine(bins)
    pairs = rng.integers(-8, 9, (n, 2)).astype(np.float32)  # every sum exact
    engine.prepare(pairs)
    hist = engine.build(np.arange(n))
    index = hb.DMatrix(x).index(bins)
    row_ptr, row_bins = index.row_bins()
    rows = np.repeat(np.arange(n), np.diff(row_ptr.astype(np.int64)))
    for c in (0, 1):
        want = np.bincount(row_bins, weights=pairs[rows, c].astype(np.float64), minlength=len(hist))
        assert np.array_equal(hist[:, c], want)


@pytest.mark.parametrize("n", [1, 2, 63, 64, 1025, 300_001])
def test_intercepts_from_counted_labels(n):
    """The trainer's intercept from the device's label counts equals the
    host's chain of additions over the labels, and labels that are not
    classes are refused."""
    rng = np.random.default_rng(n)
    engine = hb.DMatrix(rng.standard_normal((n, 2), dtype=np.float32)).engine()
    for y in ((rng.random(n) < 0.37).astype(np.float32), np.zeros(n, np.float32), np.full(n, -0.0, np.float32),
              np.ones(n, np.float32), rng.standard_normal(n).astype(np.float32)):
        mean = np.add.accumulate(y.astype(np.float64) / n)[-1]
        for objective in ("reg:squarederror", "binary:logitraw"):
            got = hb.Trainer(engine, {"objective": objective}, y).base_score()
            assert got.view(np.uint32)[0] == np.float32(mean).view(np.uint32) or got[0] == np.float32(mean) == 0
    k = 5
    y = rng.integers(0, k, n).astype(np.float32)
    t = hb.Trainer(engine, {"objective": "multi:softprob", "num_class": k}, y)
    prior = np.log(np.float32(np.bincount(y.astype(int), minlength=k) / np.float32(n)) + np.float32(1e-6))
    assert np.allclose(t.base_score(), prior - prior.mean(dtype=np.float32), rtol=0, atol=1e-5)
    assert np.array_equal(t.margins().reshape(n, k), np.broadcast_to(t.base_score(), (n, k)))
    for bad in (-1.0, float(k), 1.5, np.nan, np.inf):
        y[n // 2] = bad
        with pytest.raises(hb.HbrError):
            hb.Trainer(engine, {"objective": "multi:softprob", "num_class": k}, y)


# one to several groups of features and tiles, narrow and constant features,
# missing cells (the backward pass), with and without the guard, monotone
@pytest.mark.parametrize("n,f,nan,params", [
    (300, 1, 0.0, {}), (5_000, 3, 0.2, {}), (40_000, 33, 0.0, {"gamma": 0.1, "monotone_constraints": [1, -1]}),
    (40_000, 33, 0.1, {"monotone_constraints": [1, -1], "min_child_weight": 3.0}), (120_000, 70, 0.05, {"alpha": 0.2}),
    (9_000, 4, 0.3, {"max_bin": 17}), (9_000, 5, 0.0, {"max_delta_step": 0.4}),
])
def test_level_reduce_and_search_give_the_host_levels_trees(monkeypatch, n, f, nan, params):
    x, y = _data(n, f, nan, seed=n + f)
    x[:, -1] = 3.0  # one bin: no candidate
    x[:, f // 2] = np.round(x[:, f // 2])
    params = dict(params, objective="binary:logistic", max_depth=7, eta=0.3)
    device, host = _both(monkeypatch, x, y, params, 2)
    assert device[2].get("hbr_reduce_scan", 0) > 0
    _same(device, host)


# best-first trees whose nodes are split ahead of their pops: budgets that end
# before, inside and after a batch, more leaves than the rows allow; dense
# rows (margins by the walk) and sparse ones (margins by each leaf's rows)
@pytest.mark.parametrize("sparse", [False, True])
@pytest.mark.parametrize("leaves,depth", [(2, 0), (3, 0), (6, 0), (40, 0), (41, 5), (200, 0), (0, 4), (5000, 0)])
def test_best_first_trees_split_ahead_match_the_oracle(sparse, leaves, depth):
    from oracle import oracle as O
    from tests.test_gpu_train import compare_trees

    rng = np.random.default_rng(leaves + 7 * depth)
    n, f = 3_000, 30
    x = rng.exponential(1.0, (n, f)).astype(np.float32)
    if sparse:
        x[rng.random(x.shape) < 0.85] = np.nan
    y = (np.nan_to_num(x[:, 0]) - np.nan_to_num(x[:, 1]) * np.nan_to_num(x[:, 2]) + rng.standard_normal(n) * 0.1)
    y = y.astype(np.float32)
    params = {"grow_policy": "lossguide", "max_depth": depth, "max_leaves": leaves, "eta": 0.3, "min_child_weight": 2.0}
    ref = O.Model(O.Dataset(x), y, O.params(grow_policy=O.GROW_LOSSGUIDE, max_depth=depth, max_leaves=leaves,
                                            min_child_weight=2.0), 3)
    engine = hb.DMatrix(x, label=y).engine()
    t = hb.Trainer(engine, params, y)
    before = engine.counters()
    t.boost(3)
    compare_trees(t.trees(), ref.trees())
    assert np.max(np.abs(t.margins() - ref.margins().reshape(-1))) <= 1e-5
    assert engine.counters()["near_ties"] - before["near_ties"] <= sum(len(k["left"]) for k in t.trees())


# sparse rows: most bins of a node empty (few rows) and none (many), features
# of one bin, of at most 64, of up to 256 and of more (several chunks a pass)
@pytest.mark.parametrize("n", [40, 3_000, 12_000])
@pytest.mark.parametrize("bins", [20, 256, 700])
@pytest.mark.parametrize("lossguide", [False, True])
def test_sparse_search_and_siblings_match_the_oracle(n, bins, lossguide):
    from oracle import oracle as O
    from tests.test_gpu_train import compare_trees

    rng = np.random.default_rng(n + bins)
    f = 260  # more than masked rows take
    x = rng.standard_normal((n, f)).astype(np.float32)
    x[rng.random(x.shape) < 0.7] = np.nan
    x[:, 3] = np.where(np.isnan(x[:, 3]), np.nan, 2.0)  # one bin
    x[:, 4] = np.round(x[:, 4] * 3)
    y = np.nan_to_num(x[:, 0]) - np.nan_to_num(x[:, 1]) * np.nan_to_num(x[:, 4]) + 0.5 * np.isnan(x[:, 3])
    y = (y + 0.1 * rng.standard_normal(n)).astype(np.float32)
    grow = dict(max_depth=0, max_leaves=30) if lossguide else dict(max_depth=6)
    params = dict(grow, max_bin=bins, eta=0.3, min_child_weight=2.0, grow_policy="lossguide" if lossguide else "depthwise")
    more = dict(grow_policy=O.GROW_LOSSGUIDE) if lossguide else {}
    ref = O.Model(O.Dataset(x, max_bin=bins), y, O.params(min_child_weight=2.0, **grow, **more), 2)
    trees, margins, launches = _fit(x, y, params, 2)
    assert launches.get("hbr_scan_sparse", 0) > 0 and "hbr_subtract" not in launches
    compare_trees(trees, ref.trees())
    assert np.max(np.abs(margins - ref.margins().reshape(-1))) <= 1e-5  # f32 sums of two leaves each


# rows of u16 bins: each width of a feature group, one group and several, one
# tile and many, class trees in a batch
@pytest.mark.parametrize("n,f,bins,depth,classes", [
    (1, 2, 300, 3, 0), (600, 17, 512, 1, 0), (5_000, 16, 300, 6, 0), (5_000, 5, 1000, 8, 0), (30_000, 33, 600, 5, 0),
    (40_000, 3, 8000, 4, 0), (600_001, 2, 512, 4, 0), (20_000, 6, 400, 4, 3), (9_000, 4, 2000, 10, 0),
])
def test_device_growth_over_u16_bins_gives_the_host_levels_trees(monkeypatch, n, f, bins, depth, classes):
    x, y = _data(n, f, 0.0, seed=n + bins, classes=classes)
    params = {"objective": "multi:softprob" if classes else "binary:logistic", "max_depth": depth, "eta": 0.3,
              "base_score": 0.5, "max_bin": bins}
    if classes:
        params["num_class"] = classes
    device, host = _both(monkeypatch, x, y, params, 3)
    if n > 1 and depth > 1:
        assert device[2].get("hbr_part_move", 0) > 0 and device[2].get("hbr_walk_leaves16", 0) > 0
    _same(device, host)
