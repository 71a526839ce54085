"""The pair walk's ways of sharing a row block (a wave a block, a workgroup's
waves sharing one) against the one-level mirror walk, margins and leaf ids
bit for bit: rows around a block and around the block counts where the way
changes, trees around a wave's sixteen, one and several outputs."""
import numpy as np
import pytest

import hessboost_amd as hb

pytestmark = pytest.mark.gpu


def _forest(rng, trees, depth, f, outputs):
    inner, nodes = (1 << depth) - 1, (2 << depth) - 1
    i = np.arange(nodes)
    leaf = i >= inner
    return dict(tree_offset=np.arange(trees + 1, dtype=np.uint64) * nodes,
                split_feature=rng.integers(0, f, trees * nodes).astype(np.uint32),
                split_cond=rng.standard_normal(trees * nodes).astype(np.float32),
                default_left=rng.integers(0, 2, trees * nodes).astype(np.uint8),
                left=np.tile(np.where(leaf, -1, 2 * i + 1), trees).astype(np.int32),
                right=np.tile(np.where(leaf, -1, 2 * i + 2), trees).astype(np.int32),
                leaf_value=rng.standard_normal(trees * nodes).astype(np.float32),
                tree_weight=rng.random(trees).astype(np.float32),
                tree_output=rng.integers(0, outputs, trees).astype(np.uint32),
                base_score=rng.standard_normal(outputs).astype(np.float32))


@pytest.mark.parametrize("n", [1, 63, 64, 65, 256 * 64, 256 * 64 + 1, 512 * 64 + 7, 1024 * 64 + 65])
@pytest.mark.parametrize("trees,depth,f,outputs", [(1, 3, 3, 1), (16, 2, 30, 1), (17, 5, 126, 3), (300, 3, 20, 1),
                                                   (270, 4, 60, 4)])
def test_shared_blocks_equal_the_mirror_walk(monkeypatch, n, trees, depth, f, outputs):
    rng = np.random.default_rng(n + trees)
    forest = hb.Forest(_forest(rng, trees, depth, f, outputs), outputs)
    x = rng.standard_normal((n, f), dtype=np.float32)
    x[rng.random(x.shape) < 0.05] = np.nan
    init = rng.standard_normal((n, outputs)).astype(np.float32)

    def all_of():
        small = x[:2_000]
        return [forest.predict_margin(x), forest.predict_margin(x, init_margins=init),
                forest.predict_margin(np.nan_to_num(x, nan=-7.0), missing=-7.0),
                forest.predict_leaf(small).astype(np.float32)]

    pairs = all_of()
    monkeypatch.setenv("HBROCM_PRED_KERNEL", "mirror")
    for got, want in zip(pairs, all_of()):
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))



# host rows read in place (up to 256 KiB), in one copy (up to 8 MiB), in chunks
@pytest.mark.parametrize("n", [1, 700, 1_250, 2_180, 2_200, 8_700, 8_800, 20_011, 69_905, 69_906, 150_001])
@pytest.mark.parametrize("outputs", [1, 3])
def test_host_rows_of_every_size_equal_device_rows(n, outputs):
    rng = np.random.default_rng(n + outputs)
    f = 30
    forest = hb.Forest(_forest(rng, 40, 5, f, outputs), outputs)
    x = rng.standard_normal((n, f), dtype=np.float32)
    x[rng.random(x.shape) < 0.05] = np.nan
    dx, dout = hb.DeviceBuffer(x.nbytes), hb.DeviceBuffer(4 * n * outputs)
    dx.upload(x)
    forest.predict_margin_device(dx.ptr, n, f, dout.ptr)
    want = dout.download(np.float32, n * outputs)
    init = np.tile(forest.arrs["base_score"], (n, 1))
    for _ in range(2):
        assert np.array_equal(forest.predict_margin(x).view(np.uint32), want.view(np.uint32))
        assert np.array_equal(forest.predict_margin(x, init_margins=init).view(np.uint32), want.view(np.uint32))


def test_forests_in_several_threads_share_the_device():
    """Each its own forest, sizes that are read in place, copied and staged in
    turn: every thread gets what it gets alone."""
    import threading

    rng = np.random.default_rng(3)
    k, f = 4, 30
    forests = [hb.Forest(_forest(rng, 20 + 9 * i, 4, f, 1 + i % 2), 1 + i % 2) for i in range(k)]
    rows = [[rng.standard_normal((n, f), dtype=np.float32) for n in (1, 900, 3_000, 12_000, 75_000)] for _ in range(k)]
    alone = [[forests[i].predict_margin(x) for x in rows[i]] for i in range(k)]
    wrong, gate = [], threading.Barrier(k)

    def work(i):
        gate.wait()
        for turn in range(12):
            for j in range(len(rows[i])):
                at = (j + i + turn) % len(rows[i])
                if not np.array_equal(forests[i].predict_margin(rows[i][at]), alone[i][at]):
                    wrong.append((i, at, turn))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(k)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
