"""Calls at the limits of a dispatch: more features than a packed node holds,
small and uneven shapes that a rule made for average ones must still take."""
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
