"""The work that users of this package have it do, as measurable cases.

Every case goes through the public Python entry points (`train`, `Engine`,
`Trainer`, `RowEngineRounds`, `Forest`) on seeded inputs. Feature values lie
on a grid of as many normal quantiles as the case has bins, so the cuts are
the grid's steps and a value's bin is its rank: `exact` can then grow the
same trees in 64 bits from the ranks alone.

Kinds (`case["kind"]`):

- "predict": margins of a batch of rows by an uploaded forest, from host rows
  (a service's request) or from rows already on the GPU (a scoring job);
- "call": one whole `train` call on host arrays, with an evaluation set;
- "fit": boosting rounds over an index resident on the GPU, dense rows
  (with or without missing cells, weights, several classes, more than 256
  bins) or sparse ones;
- "rounds": the same rounds driven call for call through the row engine.
"""
import math

import numpy as np
import torch

import hessboost_amd as hb
from hessboost_amd import _capi
from hessboost_amd.rowengine import RowEngineRounds, as_tree

_FIELDS = ("left", "split_feature", "split_cond", "default_left", "leaf_value")
_DEV = "cuda:0"


def _fit(name, objective, n, f, depth, rounds, **more):
    case = dict(name=name, kind="fit", objective=objective, n=n, f=f, depth=depth, rounds=rounds, classes=1,
                bins=256, nan=0.0, weighted=False, density=1.0, leaves=0, eta=0.1)
    case.update(more)
    return case


def _predict(name, n, f, trees, depth, where, nan=0.0, outputs=1):
    return dict(name=name, kind="predict", n=n, f=f, trees=trees, depth=depth, where=where, nan=nan, outputs=outputs)


def listed():
    return [
        # a service scoring a handful of rows per request: latency alone
        _predict("predict_request", 32, 28, 100, 6, "host"),
        # a batch scoring job handing over host rows (the copy is part of it)
        _predict("predict_batch_host", 500_000, 30, 100, 6, "host"),
        # a multi-class model over rows on the GPU, an odd row count
        _predict("predict_classes", 200_003, 50, 1000, 6, "device", outputs=10),
        # the large ensemble over a large resident table with missing cells
        _predict("predict_resident", 10_000_000, 100, 1000, 8, "device", nan=0.02),
        # a small table trained from scratch in one call, with an evaluation
        # set: sketch, binning, launches and readbacks all count
        dict(name="train_call_small", kind="call", objective="binary:logistic", n=4_000, f=8, depth=4, rounds=20,
             classes=1, bins=256, nan=0.0, weighted=False, density=1.0, leaves=0, eta=0.3, evals=1_000),
        # a mid-size regression fit: many small launches per round
        _fit("fit_regression", "reg:squarederror", 100_000, 32, 6, 100),
        # the large binary fit: ten million rows, deep trees
        _fit("fit_logistic_large", "binary:logistic", 10_500_000, 28, 8, 100),
        # a weighted table with missing cells and an odd row count
        _fit("fit_missing_weighted", "binary:logistic", 1_000_003, 50, 8, 20, nan=0.02, weighted=True),
        # ten classes: ten trees a round
        _fit("fit_classes", "multi:softprob", 2_000_000, 50, 6, 5, classes=10, eta=0.3),
        # a wide sparse table grown best-first
        _fit("fit_sparse_lossguide", "reg:squarederror", 100_000, 1_000, 0, 4, density=0.1, leaves=255, eta=0.3),
        # finer bins than a byte holds
        _fit("fit_fine_bins", "binary:logistic", 500_000, 28, 7, 10, bins=512),
        # an outside builder driving each level through the row engine
        _fit("rounds_row_engine", "binary:logistic", 1_000_000, 30, 8, 3, kind="rounds"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("predict", "predict", "call", "dense", "dense", "classes", "sparse", "fine", "rounds"))
    if kind == "predict":
        where = rng.choice(("host", "device"))
        trees, depth = _log(rng, 20, 1000), rng.randint(3, 8)
        outputs = rng.choice((1, 1, 3, 10))
        trees = max(outputs, trees // outputs * outputs)
        n = _log(rng, 1, 500_000) if where == "host" else _log(rng, 1_000, 4_000_000)
        return dict(kind="predict", n=n, f=_log(rng, 4, 100), trees=trees, depth=depth, where=where,
                    nan=rng.choice((0.0, 0.02)), outputs=outputs)
    if kind == "call":
        return dict(kind="call", objective=rng.choice(("binary:logistic", "reg:squarederror")),
                    n=_log(rng, 4_000, 50_000), f=rng.randint(4, 33), depth=rng.randint(3, 7),
                    rounds=rng.randint(10, 50), classes=1, bins=256, nan=rng.choice((0.0, 0.02)), weighted=False,
                    density=1.0, leaves=0, eta=0.3, evals=_log(rng, 500, 5_000))
    case = _fit("", rng.choice(("binary:logistic", "reg:squarederror")), 0, 0, 0, 0, eta=rng.choice((0.1, 0.3)))
    del case["name"]
    if kind == "dense":
        case.update(n=_log(rng, 3_000, 4_000_000), f=rng.randint(5, 100), depth=rng.randint(4, 9),
                    rounds=rng.randint(5, 30), nan=rng.choice((0.0, 0.02)), weighted=rng.random() < 0.3)
    elif kind == "classes":
        case.update(objective="multi:softprob", classes=rng.choice((2, 3, 4, 7, 10)), n=_log(rng, 10_000, 1_000_000),
                    f=rng.randint(8, 64), depth=rng.randint(3, 7), rounds=rng.randint(3, 8))
    elif kind == "sparse":
        case.update(objective="reg:squarederror", n=_log(rng, 10_000, 100_000), f=_log(rng, 200, 1_000), density=0.1,
                    leaves=rng.randint(15, 255), rounds=rng.randint(2, 4))
    elif kind == "fine":
        case.update(n=_log(rng, 20_000, 500_000), f=rng.randint(8, 40), depth=rng.randint(4, 8),
                    rounds=rng.randint(5, 10), bins=rng.choice((300, 512, 1000)))
    else:
        case.update(kind="rounds", n=_log(rng, 20_000, 1_000_000), f=rng.randint(8, 32), depth=rng.randint(4, 8),
                    rounds=rng.randint(2, 4))
    return case


# ---- inputs --------------------------------------------------------------------------

def _grid(case):
    """The feature values: normal quantiles, ascending, fewer than the bins."""
    q = (torch.arange(case["bins"] - 6, dtype=torch.float64) + 0.5) / (case["bins"] - 6)
    return (torch.erfinv(2 * q - 1) * math.sqrt(2)).to(torch.float32)


def _table(case, seed, n=None):
    """(ranks [n][f] int16 with -1 for a missing cell, labels, weights) on the GPU."""
    n, f = case["n"] if n is None else n, case["f"]
    gen = torch.Generator(device=_DEV).manual_seed(seed)
    levels = case["bins"] - 6
    k = torch.randint(0, levels, (n, f), generator=gen, device=_DEV, dtype=torch.int16)
    v = _grid(case).to(_DEV)
    if case["density"] < 1.0:
        # a sparse row's absent cells count as 0 for its label
        chunk = max(1, (1 << 26) // f)
        for s in range(0, n, chunk):
            part = k[s:s + chunk]
            part[torch.rand(part.shape, generator=gen, device=_DEV) >= case["density"]] = -1
    col = lambda c: torch.where(k[:, c % f] < 0, 0.0, v[k[:, c % f].long().clamp_min(0)])  # noqa: E731
    s = 0.8 * col(0) - 0.5 * col(1) * col(2) + torch.tanh(col(3)) + 0.3 * (col(4) * col(5)).abs()
    if case["objective"] == "multi:softprob":
        w = torch.randn((case["classes"], f), generator=gen, device=_DEV) / math.sqrt(f)
        score = torch.empty((n, case["classes"]), device=_DEV)
        for b in range(0, n, 1 << 20):
            score[b:b + (1 << 20)] = v[k[b:b + (1 << 20)].long()] @ w.T
        gumbel = -torch.log(-torch.log(torch.rand(score.shape, generator=gen, device=_DEV).clamp(1e-7, 1 - 1e-7)))
        y = (2 * score + gumbel).argmax(1).float()
    elif case["objective"] == "binary:logistic":
        y = (torch.rand(n, generator=gen, device=_DEV) < torch.sigmoid(s)).float()
    else:
        y = s + 0.1 * torch.randn(n, generator=gen, device=_DEV)
    wt = 0.5 + torch.rand(n, generator=gen, device=_DEV) if case["weighted"] else None
    if case["nan"] > 0:
        chunk = max(1, (1 << 26) // f)
        for b in range(0, n, chunk):
            part = k[b:b + chunk]
            part[torch.rand(part.shape, generator=gen, device=_DEV) < case["nan"]] = -1
    return k, y, wt


def _values(case, k):
    v = torch.cat([_grid(case).to(k.device), torch.full((1,), math.nan, device=k.device)])
    x = torch.empty(k.shape, dtype=torch.float32, device=k.device)
    chunk = max(1, (1 << 26) // k.shape[1])
    for s in range(0, k.shape[0], chunk):
        x[s:s + chunk] = v[k[s:s + chunk].long()]  # rank -1 is the last entry, NaN
    return x


class _Memory:
    """A tensor's memory as DeviceBuffer.copy_from reads it."""

    def __init__(self, t):
        self.ptr, self.nbytes, self.tensor = t.data_ptr(), t.numel() * t.element_size(), t


def _resident_engine(case, k):
    """The engine over rows already on the GPU, cuts from the first rows."""
    x = _values(case, k)
    cuts = hb.Cuts.from_dense(x[:65_536].cpu().numpy(), max_bin=case["bins"])
    torch.cuda.synchronize()
    buf = hb.DeviceBuffer(x.numel() * 4)
    buf.copy_from(_Memory(x))
    return hb.Engine.from_dense(buf, cuts, n_rows=case["n"], n_cols=case["f"])


def _params(case):
    p = {"objective": case["objective"], "eta": case["eta"], "max_depth": case["depth"], "max_bin": case["bins"]}
    if case["classes"] > 1:
        p["num_class"] = case["classes"]
    if case["leaves"]:
        p.update(grow_policy="lossguide", max_leaves=case["leaves"], max_depth=64)
    return p


def _forest_tables(case, seed):
    """Complete trees as a [trees][nodes] table: features, thresholds,
    default directions, leaf values."""
    rng = np.random.default_rng(seed)
    inner, nodes = (1 << case["depth"]) - 1, (2 << case["depth"]) - 1
    shape = (case["trees"], nodes)
    leaf = np.arange(nodes)[None, :] >= inner
    feature = np.where(leaf, 0, rng.integers(0, case["f"], shape)).astype(np.uint32)
    cond = np.where(leaf, 0.0, rng.standard_normal(shape)).astype(np.float32)
    default = rng.integers(0, 2, shape).astype(np.uint8)
    value = np.where(leaf, rng.normal(0.0, 0.05, shape), 0.0).astype(np.float32)
    return feature, cond, default, value


def _predict_rows(case, seed):
    gen = torch.Generator(device=_DEV).manual_seed(seed)
    x = torch.randn((case["n"], case["f"]), generator=gen, device=_DEV)
    if case["nan"] > 0:
        chunk = max(1, (1 << 26) // case["f"])
        for s in range(0, case["n"], chunk):
            part = x[s:s + chunk]
            part[torch.rand(part.shape, generator=gen, device=_DEV) < case["nan"]] = math.nan
    return x


def prepare(case, seed):
    if case["kind"] == "predict":
        feature, cond, default, value = _forest_tables(case, seed)
        trees, nodes = feature.shape
        i = np.arange(nodes)
        leaf = i >= nodes // 2
        every = lambda v, dt: np.broadcast_to(v.astype(dt), feature.shape).reshape(-1)  # noqa: E731
        arrs = dict(tree_offset=np.arange(trees + 1, dtype=np.uint64) * nodes, split_feature=feature.reshape(-1),
                    split_cond=cond.reshape(-1), default_left=default.reshape(-1),
                    left=every(np.where(leaf, -1, 2 * i + 1), np.int32),
                    right=every(np.where(leaf, -1, 2 * i + 2), np.int32), leaf_value=value.reshape(-1),
                    tree_weight=np.ones(trees, np.float32),
                    tree_output=(np.arange(trees) % case["outputs"]).astype(np.uint32),
                    base_score=np.zeros(case["outputs"], np.float32))
        x = _predict_rows(case, seed)
        state = dict(kind="predict", where=case["where"], forest=hb.Forest(arrs, case["outputs"]), n=case["n"],
                     f=case["f"], outputs=case["outputs"])
        state["x"] = x.cpu().numpy() if case["where"] == "host" else x
        torch.cuda.synchronize()
        return state
    params = _params(case)
    if case["kind"] == "call":
        k, y, _ = _table(case, seed)
        ke, ye, _ = _table(case, seed + 7_919, case["evals"])
        return dict(kind="call", params=params, rounds=case["rounds"], nodes=_most_nodes(case),
                    x=_values(case, k).cpu().numpy(), y=y.cpu().numpy(), xe=_values(case, ke).cpu().numpy(),
                    ye=ye.cpu().numpy())
    k, y, wt = _table(case, seed)
    state = dict(kind=case["kind"], params=params, rounds=case["rounds"], nodes=_most_nodes(case), y=y.cpu().numpy(),
                 wt=None if wt is None else wt.cpu().numpy())
    if case["density"] < 1.0:
        present = k >= 0
        ptr = torch.zeros(case["n"] + 1, dtype=torch.int64, device=_DEV)
        ptr[1:] = torch.cumsum(present.sum(1), 0)
        cols = torch.nonzero(present)[:, 1].to(torch.int32)
        vals = _grid(case).to(_DEV)[k[present].long()]
        data = hb.DMatrix((ptr.cpu().numpy(), cols.cpu().numpy(), vals.cpu().numpy()), label=state["y"],
                          n_cols=case["f"])
        state["engine"] = data.engine(case["bins"])
    elif case["bins"] > 256:
        state["engine"] = hb.DMatrix(_values(case, k).cpu().numpy(), label=state["y"]).engine(case["bins"])
    else:
        state["engine"] = _resident_engine(case, k)
    if case["kind"] == "rounds":
        state["fo"], state["cuts"] = state["engine"].index.feature_offset(), state["engine"].index.cut_values()
        state["engine"].set_sums("fixed_point")
    return state


# ---- one pass ----------------------------------------------------------------------------

def _model(trees, nodes):
    """A model's trees as one [trees][nodes] table a field, each tree padded
    to the most nodes it can have, and each tree's node count."""
    out = {"nodes": np.array([len(t["left"]) for t in trees], np.int64)}
    for key in _FIELDS:
        table = np.zeros((len(trees), nodes), np.asarray(trees[0][key]).dtype)
        for row, t in zip(table, trees):
            row[:len(t[key])] = t[key]
        out[key] = table
    return out


def _most_nodes(case):
    return 2 * case["leaves"] - 1 if case["leaves"] else (2 << case["depth"]) - 1


def run(state):
    kind = state["kind"]
    if kind == "predict":
        if state["where"] == "host":
            return state["forest"].predict_margin(state["x"])
        out = torch.empty(state["n"] * state["outputs"], dtype=torch.float32, device=_DEV)
        state["forest"].predict_margin_device(state["x"].data_ptr(), state["n"], state["f"], out.data_ptr())
        return out
    nodes = state["nodes"]
    if kind == "call":
        b = hb.train(state["params"], hb.DMatrix(state["x"], label=state["y"]), state["rounds"],
                     evals=[(hb.DMatrix(state["xe"], label=state["ye"]), "eval")])
        return {**_model(b.trees, nodes), "eval_margins": b.eval_margins["eval"]}
    if kind == "rounds":
        driver = RowEngineRounds(state["engine"], state["fo"], state["cuts"], state["params"],
                                 _capi.LOSS_LOGISTIC if state["params"]["objective"] == "binary:logistic"
                                 else _capi.LOSS_SQUARED_ERROR)
        margins = np.zeros(len(state["y"]), np.float32)
        return _model([as_tree(driver.device_round(margins, state["y"])) for _ in range(state["rounds"])], nodes)
    t = hb.Trainer(state["engine"], state["params"], state["y"], state["wt"])
    t.boost(state["rounds"])
    return _model(t.trees(), nodes)


# ---- what a pass cannot do without ------------------------------------------------------------

def work(case):
    if case["kind"] == "predict":
        # each cell read once, each node once, each margin written; a step of
        # the walk is a comparison, a leaf an addition
        return {"bytes": 4.0 * case["n"] * (case["f"] + case["outputs"]) + 16.0 * case["trees"] * (2 << case["depth"]),
                "flops": float(case["n"]) * case["trees"] * (case["depth"] + 1)}
    # per tree the root's histogram reads every row's bins, and each further
    # level (eight of them for a leaf-bounded tree of 255 leaves) the rows of
    # the smaller children, a half at most and a third taken; the pairs and
    # margins are read and written once; two additions a binned cell
    width = 1 if case["bins"] <= 256 else 2
    cells = case["n"] * case["f"] * case["density"]
    levels = case["depth"] or max(1.0, math.log2(case["leaves"] + 1))
    passes = 1 + (levels - 1) / 3
    trees = case["rounds"] * case["classes"]
    entry = 4 if case["density"] < 1.0 else width
    once = 4.0 * case["n"] * case["f"] if case["kind"] == "call" else 0.0
    return {"bytes": once + trees * (passes * cells * entry + 16.0 * case["n"]), "flops": trees * passes * cells * 2.0}


# Prediction sums a tree's leaf per f32 addition in tree order: another order
# shows about 1e-7 of the result for 100 trees and 4e-7 for 1,000. A fit's
# histograms are integer sums of quantised pairs, so its splits are whole
# numbers that do not depend on an order; its leaf values and thresholds are
# single f32 roundings of f64 quotients, and its evaluation margins f32 sums.
def tolerance(case):
    if case["kind"] == "predict":
        return {"rel": 2e-6, "max": 2e-5}
    return {"rel": 1e-6, "max": 1e-5, "differ": 0.0}


# ---- the same in 64 bits -------------------------------------------------------------------------

def _exact_predict(case, seed):
    if float(case["n"]) * case["trees"] * case["depth"] > 4e10:
        return None
    feature, cond, default, value = (torch.from_numpy(t.astype(np.int64) if t.dtype.kind == "u" else t).to(_DEV)
                                     for t in _forest_tables(case, seed))
    x = _predict_rows(case, seed)
    out = torch.zeros((case["n"], case["outputs"]), dtype=torch.float64, device=_DEV)
    for s in range(0, case["n"], 1 << 20):
        part = x[s:s + (1 << 20)]
        rows = torch.arange(part.shape[0], device=_DEV)
        for t in range(case["trees"]):
            at = torch.zeros(part.shape[0], dtype=torch.int64, device=_DEV)
            for _ in range(case["depth"]):
                v = part[rows, feature[t][at]]
                left = torch.where(torch.isnan(v), default[t][at] != 0, v < cond[t][at])
                at = 2 * at + torch.where(left, 1, 2)
            out[s:s + (1 << 20), t % case["outputs"]] += value[t][at].double()
    out = out.reshape(-1)
    return out.cpu().numpy() if case["where"] == "host" else out


def _weight(g, h):
    """A node's weight at lambda 1, with the search's floor of h > 0."""
    return torch.where(h > 0, -g / (h + 1.0), torch.zeros_like(g))


def _gain32(g, h):
    """A child's gain as the split score defines it: the weight rounded to
    f32 (its square too), the gain in f64 rounded to f32."""
    w = _weight(g, h).float()
    return torch.where(h > 0, -(2.0 * g * w.double() + (h + 1.0) * (w * w).double()), torch.zeros_like(g)).float()


def _search(hist, total):
    """The best split of each node from hist [m][f][b][2] and total [m][2],
    in the order candidates are defined: features ascending, per feature the
    forward pass over its bins, then the backward one; the first best wins."""
    m, f, b, _ = hist.shape
    pre = torch.cumsum(hist, 2)
    suf = torch.flip(torch.cumsum(torch.flip(hist, (2,)), 2), (2,))
    t = total[:, None, None, :]
    left = torch.cat([pre, t - torch.flip(suf, (2,))], 2)  # [m][f][2b][2]
    right = torch.cat([t - pre, torch.flip(suf, (2,))], 2)
    ok = (left[..., 1] >= 1.0) & (right[..., 1] >= 1.0)
    loss = (_gain32(left[..., 0], left[..., 1]) + _gain32(right[..., 0], right[..., 1])) - _gain32(
        total[:, 0], total[:, 1])[:, None, None]
    # without missing cells the backward pass repeats the forward one
    full = (pre[:, :, -1, 1] - total[:, None, 1]).abs() <= 1e-9 * total[:, None, 1].abs() + 1e-12
    ok[:, :, b:] &= ~full[:, :, None]
    loss = torch.where(ok, loss, torch.full_like(loss, -1.0)).reshape(m, -1)
    best = loss.max(1).values
    at = (loss == best[:, None]).int().argmax(1)
    pick = at[:, None, None].expand(-1, 1, 2)
    left, right = left.reshape(m, -1, 2).gather(1, pick)[:, 0], right.reshape(m, -1, 2).gather(1, pick)[:, 0]
    feat, pos = at // (2 * b), at % (2 * b)
    limit = torch.where(pos < b, pos + 1, 2 * b - 1 - pos)  # bins below it go left
    return best, feat, limit, pos >= b, left, right


class _Grower:
    """A tree over ranks [n][f] (-1: missing) in 64 bits."""

    def __init__(self, case, k):
        self.case, self.k = case, k
        self.f, self.b = case["f"], case["bins"] - 6

    def hist(self, rows, node, m, g, h):
        """[m][f][b][2] sums over rows (node: each row's node below m)."""
        out = torch.zeros((2, m * self.f * self.b), dtype=torch.float64, device=_DEV)
        first = torch.arange(self.f, device=_DEV) * self.b
        chunk = max(1, (1 << 27) // self.f)
        for s in range(0, rows.shape[0], chunk):
            r = rows[s:s + chunk]
            k = self.k[r].long()
            at = node[s:s + chunk, None] * (self.f * self.b) + first + k
            some = k >= 0
            at = at[some]
            for c, v in ((0, g), (1, h)):
                out[c].index_add_(0, at, v[r][:, None].expand(-1, self.f)[some])
        return out.reshape(2, m, self.f, self.b).permute(1, 2, 3, 0)

    def depthwise(self, g, h):
        n = g.shape[0]
        rows = torch.arange(n, device=_DEV)
        node = torch.zeros(n, dtype=torch.int64, device=_DEV)  # the frontier node of each row, -1: in a leaf
        total = torch.stack([g.sum(), h.sum()])[None]
        ids = torch.zeros(1, dtype=torch.int64, device=_DEV)
        value = [0.0]
        tree, leaf_of = [], torch.zeros(n, dtype=torch.int64, device=_DEV)
        for level in range(self.case["depth"]):
            if not ids.numel():
                break
            live = rows[node >= 0]
            best, feat, limit, dleft, left, right = _search(self.hist(live, node[live], len(ids), g, h), total)
            split = best > 1e-6
            slot = torch.cumsum(split.long(), 0) - 1
            base = len(value)
            count = int(split.sum())
            kids = torch.stack([left[split], right[split]], 1).reshape(-1, 2)
            weights = _weight(kids[:, 0], kids[:, 1])
            for i in torch.nonzero(~split)[:, 0].tolist():
                value[int(ids[i])] = float(self.case["eta"] * _weight(total[i, 0], total[i, 1]))
            for i in torch.nonzero(split)[:, 0].tolist():
                tree.append((int(ids[i]), int(feat[i]), int(limit[i]), bool(dleft[i]), base + 2 * int(slot[i])))
            last = level + 1 == self.case["depth"]
            value += ((self.case["eta"] if last else 1.0) * weights).tolist()
            c = self.k[live, feat[node[live]]].long()
            goes = torch.where(c < 0, dleft[node[live]], c < limit[node[live]])
            at = node[live]
            kid = torch.where(split[at], 2 * slot[at] + torch.where(goes, 0, 1), torch.full_like(at, -1))
            leaf_of[live] = torch.where(kid >= 0, base + kid, leaf_of[live])
            node[live] = -1 if last else kid
            ids, total = torch.arange(2 * count, device=_DEV) + base, kids
            if last:
                ids = ids[:0]
        return tree, value, leaf_of

    def best_first(self, g, h):
        n = g.shape[0]
        leaf_of = torch.zeros(n, dtype=torch.int64, device=_DEV)
        value, tree = [0.0], []

        def opened(i, rows, total):
            found = _search(self.hist(rows, torch.zeros_like(rows), 1, g, h), total[None])
            best, feat, limit, dleft = float(found[0][0]), int(found[1][0]), int(found[2][0]), bool(found[3][0])
            return (best, i, rows, total, feat, limit, dleft, found[4][0], found[5][0])

        heap, done = [opened(0, torch.arange(n, device=_DEV), torch.stack([g.sum(), h.sum()]))], []
        leaves = 1
        while heap and leaves < self.case["leaves"]:
            top = max(range(len(heap)), key=lambda j: heap[j][0])
            best, i, rows, total, feat, limit, dleft, left, right = heap.pop(top)
            if best <= 1e-6:
                done.append((i, total))
                continue
            base = len(value)
            tree.append((i, feat, limit, dleft, base))
            value[i] = float(_weight(total[0], total[1])) if i else 0.0
            value += [0.0, 0.0]
            c = self.k[rows, feat].long()
            goes = (c < limit) & (c >= 0) | (c < 0) & dleft
            leaves += 1
            for j, r, s in ((base, rows[goes], left), (base + 1, rows[~goes], right)):
                leaf_of[r] = j
                heap.append(opened(j, r, s))
        for i, total in done + [(o[1], o[3]) for o in heap]:
            value[i] = float(self.case["eta"] * _weight(total[0], total[1]))
        return tree, value, leaf_of


def _route(tree, k):
    """The node each row of ranks k ends in."""
    at = torch.zeros(k.shape[0], dtype=torch.int64, device=_DEV)
    for i, feat, limit, dleft, base in tree:  # parents come before their children
        here = torch.nonzero(at == i)[:, 0]
        c = k[here, feat].long()
        at[here] = base + torch.where(torch.where(c < 0, torch.full_like(c, dleft) != 0, c < limit), 0, 1)
    return at


def exact(case, seed):
    """The trees' leaf values (and evaluation margins) in 64 bits. Splits are
    taken by the score's own definition, whose f32 roundings decide ties."""
    if case["kind"] == "predict":
        return _exact_predict(case, seed)
    levels = case["depth"] or 12
    cells = float(case["n"]) * case["f"] * case["rounds"] * case["classes"] * levels
    if cells > (1.2e10 if case["density"] == 1.0 else 6e9):
        return None
    k, y, wt = _table(case, seed)
    y, n, classes = y.double(), case["n"], case["classes"]
    w = torch.ones(n, dtype=torch.float64, device=_DEV) if wt is None else wt.double()
    margins = torch.zeros((n, classes), dtype=torch.float64, device=_DEV)
    start = torch.zeros(classes, dtype=torch.float64, device=_DEV)
    if case["kind"] != "rounds":
        mean = (y * w).sum() / w.sum()
        if case["objective"] == "binary:logistic":
            start[0] = torch.log(mean / (1 - mean))
        elif case["objective"] == "reg:squarederror":
            start[0] = mean
        else:
            prior = torch.bincount(y.long(), weights=w, minlength=classes) / w.sum()
            start = torch.log(prior + 1e-6)
            start = start - start.mean()
    margins += start
    grower = _Grower(case, k)
    values, trees = [], []
    for _ in range(case["rounds"]):
        if case["objective"] == "binary:logistic":
            p = torch.sigmoid(margins[:, 0])
            pairs = [((p - y) * w, (p * (1 - p)).clamp_min(1e-16) * w)]
        elif case["objective"] == "reg:squarederror":
            pairs = [((margins[:, 0] - y) * w, w)]
        else:
            p = torch.softmax(margins, 1)
            pairs = [((p[:, c] - (y == c).double()) * w, (2 * p[:, c] * (1 - p[:, c])).clamp_min(1e-16) * w)
                     for c in range(classes)]
        for c, (g, h) in enumerate(pairs):
            tree, value, leaf_of = grower.best_first(g, h) if case["leaves"] else grower.depthwise(g, h)
            trees.append(tree)
            values.append(np.array(value))
            margins[:, c] += torch.tensor(value, dtype=torch.float64, device=_DEV)[leaf_of]
    out = {key: None for key in _FIELDS}
    out["leaf_value"] = np.zeros((len(values), _most_nodes(case)))
    for row, value, tree in zip(out["leaf_value"], values, trees):
        row[:len(value)] = value
        if case["kind"] == "rounds":  # its trees keep no weights at inner nodes
            row[[i for i, *_ in tree]] = 0.0
    out["nodes"] = np.array([len(v) for v in values], np.int64)
    if case["kind"] == "call":
        ke, _, _ = _table(case, seed + 7_919, case["evals"])
        m = start[0].repeat(case["evals"])
        for tree, value in zip(trees, values):
            m = m + torch.from_numpy(value).to(_DEV)[_route(tree, ke)]
        out["eval_margins"] = m[:, None].cpu().numpy()
    return out
