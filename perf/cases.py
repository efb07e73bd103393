"""The work a user has this framework do, as cases that can be timed and compared.

Six kinds of case, each through public entry points:

- ``boost``: boosting iterations of a loaded ``Trainer`` (gradients, quantization, tree growth, leaf renewal, score
  update), the run restarted from its initial score before each pass;
- ``train``: the whole ``silvic_amd.train`` call on host data, the upload included;
- ``learner``: a tree grown split by split over the trait's calls, as a binding with its own learner does (several
  ranks, or more leaves than the device's learner takes), with the histograms on the host or in device slots;
- ``histogram``: one leaf's histogram into a device buffer;
- ``histogram_host``: one leaf's histogram to the host, as a rank that sums histograms over ranks takes it;
- ``rows``: the calls of a learner's iteration that pass over all rows (score update by a tree, gradients,
  quantization, bag, leaf sums, scores back).

Trees, histograms and scores are results of exact integer or fixed-order arithmetic, so outputs are compared exactly.
"""

import ctypes as C
import heapq
import math

import numpy as np
import torch

import silvic_amd
from silvic_amd import _abi
from silvic_amd.backend import bin_split, device_node, wide_bin_split
from silvic_amd.dataset import BinnedDataset, FeatureGroup, layout

OBJECTIVES = {"regression": _abi.OBJ_REGRESSION, "binary": _abi.OBJ_BINARY, "lambdarank": _abi.OBJ_LAMBDARANK}


def listed():
    return [
        # a small table, as in a test or a parameter search: latency and launches are all there is
        dict(name="boost 5k x 13", kind="boost", rows=5003, features=13, max_bin=63, leaves=31, objective="regression",
             rounds=20),
        # the first benchmark configuration: a mid-sized regression table
        dict(name="boost 100k x 28", kind="boost", rows=100_000, features=28, max_bin=255, leaves=31,
             objective="regression", rounds=20),
        # options in earnest: weights, categorical features, bagging, feature sampling and a validation set, odd sizes
        dict(name="boost 300k x 77 mixed", kind="boost", rows=300_007, features=77, max_bin=255, leaves=63,
             objective="binary", rounds=10, weighted=True, categorical=9, bagging=0.8, feature_fraction=0.7,
             valid_rows=60_001),
        # the headline benchmark's shape
        dict(name="boost 10M x 128", kind="boost", rows=10_000_000, features=128, max_bin=255, leaves=255,
             objective="binary", rounds=2),
        # learning to rank, half the ranking benchmark's documents
        dict(name="boost 1M x 136 rank", kind="boost", rows=1_000_000, features=136, max_bin=255, leaves=127,
             objective="lambdarank", rounds=4),
        # many mostly-zero features of few bins
        dict(name="boost 400k x 2000 sparse", kind="boost", rows=400_000, features=2000, max_bin=63, leaves=63,
             objective="binary", rounds=3, sparse=True),
        # two-byte bins, 2047 leaves and 16-bit gradient units
        dict(name="boost 6M x 32 wide", kind="boost", rows=6_000_000, features=32, max_bin=1023, leaves=2047,
             objective="regression", rounds=1, quant_bins=32766),
        # the train() call as a program makes it: the table on the host, a validation set, 30 rounds
        dict(name="train 60k x 40", kind="train", rows=60_000, features=40, max_bin=255, leaves=63,
             objective="binary", rounds=30, valid_rows=9001),
        # a binding's own learner with host histograms (several ranks add theirs up between the calls)
        dict(name="learner host 100k x 28", kind="learner", rows=100_000, features=28, max_bin=255, leaves=16,
             slots=False),
        # the same learner with the histograms in device slots, on a larger table
        dict(name="learner slots 1M x 64", kind="learner", rows=1_000_000, features=64, max_bin=255, leaves=32,
             slots=True),
        # one leaf's histogram, the hot operation by itself: a mid-sized leaf whose rows are scattered over the table
        dict(name="histogram 200k of 1M x 100", kind="histogram", rows=1_000_003, features=100, max_bin=255, share=0.2),
        # the passes over all rows that surround a tree
        dict(name="rows 3M x 40", kind="rows", rows=3_000_000, features=40, max_bin=255, leaves=127,
             objective="binary", bagging=0.75),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["boost", "boost", "boost", "boost", "train", "learner", "histogram", "histogram_host", "rows"])
    case = dict(kind=kind, max_bin=rng.choice([15, 63, 127, 255]))
    if kind == "boost":
        style = rng.choice(["dense", "dense", "options", "rank", "sparse", "wide"])
        case["rows"] = _log_int(rng, 2000, 4_000_000) | 1
        case["features"] = _log_int(rng, 4, 300)
        case["leaves"] = _log_int(rng, 7, 511)
        case["objective"] = rng.choice(["regression", "binary"])
        case["quant_bins"] = rng.choice([4, 4, 4, 16, 64, 1024])
        if style == "options":
            case.update(weighted=rng.random() < 0.5, categorical=rng.randint(0, 6), bagging=round(rng.uniform(0.5, 1.0), 2),
                        feature_fraction=round(rng.uniform(0.5, 1.0), 2), valid_rows=_log_int(rng, 500, 100_000),
                        quant_bins=4)
        elif style == "rank":
            case.update(objective="lambdarank", rows=_log_int(rng, 5000, 1_000_000), leaves=_log_int(rng, 15, 127),
                        quant_bins=4)
        elif style == "sparse":
            case.update(sparse=True, max_bin=63, features=_log_int(rng, 300, 2000), rows=_log_int(rng, 2000, 300_000),
                        leaves=_log_int(rng, 15, 127), quant_bins=4)
        elif style == "wide":
            case.update(max_bin=rng.choice([511, 1023]), features=_log_int(rng, 4, 64), leaves=_log_int(rng, 31, 1023),
                        quant_bins=rng.choice([4, 32766]))
        case["features"] = max(4, min(case["features"], 600_000_000 // case["rows"]))
        case["rounds"] = 10 if case["rows"] < 100_000 else 3 if case["rows"] < 1_000_000 else 1
    elif kind == "train":
        case.update(rows=_log_int(rng, 2000, 300_000), features=_log_int(rng, 5, 120), leaves=_log_int(rng, 15, 127),
                    objective=rng.choice(["regression", "binary"]), rounds=rng.randint(5, 40),
                    valid_rows=_log_int(rng, 500, 20_000))
    elif kind == "learner":
        case.update(rows=_log_int(rng, 2000, 2_000_000), features=_log_int(rng, 4, 128), leaves=rng.randint(8, 40),
                    slots=rng.random() < 0.5, max_bin=rng.choice([15, 63, 255, 1023]))
        if case["max_bin"] > 255:
            case["features"] = min(case["features"], 48)
    elif kind in ("histogram", "histogram_host"):
        case.update(rows=_log_int(rng, 1000, 4_000_000) | 1, features=_log_int(rng, 4, 160),
                    share=round(math.exp(rng.uniform(math.log(0.02), 0.0)), 3), max_bin=rng.choice([15, 63, 255, 1023]))
        if case["max_bin"] > 255:
            case["features"] = min(case["features"], 64)
        case["features"] = min(case["features"], 400_000_000 // case["rows"])
    else:
        case.update(rows=_log_int(rng, 2000, 4_000_000) | 1, features=_log_int(rng, 4, 60), leaves=_log_int(rng, 7, 511),
                    objective=rng.choice(["regression", "binary"]), bagging=round(rng.uniform(0.5, 1.0), 2))
    return case


# ---- tables ---------------------------------------------------------------------------------------------------


def _columns(case):
    """Bins, kinds and NaN bins of the case's features: three quarters continuous features in equal-count bins and a
    quarter integers of few values, 10% of both missing; or mostly-zero features; categorical ones last."""
    f, top = case["features"], case["max_bin"]
    r = np.random.default_rng(1000 * f + top)
    if case.get("sparse"):
        bins = [int(r.integers(17, top + 1)) if j % 8 == 0 else int(r.integers(2, 17)) for j in range(f)]
        return bins, [_abi.BINS_NUMERICAL] * f, [False] * f
    cat = min(case.get("categorical", 0), f - 1)
    bins = [top if j < 3 * f // 4 else int(r.integers(4, min(40, top) + 1)) for j in range(f)]
    kinds = [_abi.BINS_NUMERICAL] * (f - cat) + [_abi.BINS_CATEGORICAL] * cat
    return bins, kinds, [k == _abi.BINS_NUMERICAL for k in kinds]


def _table(case, rows, seed):
    """A binned dataset of the case's shape, its bins and labels drawn on the GPU."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rnd = lambda *s: torch.rand(*s, generator=gen, device="cuda")
    bins, kinds, nan_bins = _columns(case)
    wide = case["max_bin"] > 256
    features, members, total = layout(bins, kinds, nan_bins)
    informative = set(range(0, len(bins), max(1, len(bins) // 12)))
    signal = torch.zeros(rows, device="cuda")
    held, groups = None, []
    for mem in members:
        value_bins = torch.tensor([bins[j] - int(nan_bins[j]) for j in mem], device="cuda", dtype=torch.float32)
        u = rnd(rows, len(mem))
        if case.get("sparse"):  # 2% of a feature's values are not zero (bin 0)
            x = torch.where(u < 0.02, u * 50.0, torch.full_like(u, -1.0))
            b = torch.where(u < 0.02, 1 + (x * (value_bins - 1)).floor(), torch.zeros_like(u))
        else:
            x = (u - 0.1) / 0.9  # below zero: missing
            skew = torch.tensor([2.0 if j >= 3 * len(bins) // 4 else 1.0 for j in mem], device="cuda")
            b = (x.clamp_min(0) ** skew * value_bins).floor()
            missing = torch.tensor([bins[j] - 1 if nan_bins[j] else 0 for j in mem], device="cuda", dtype=torch.float32)
            b = torch.where(x < 0, missing.expand_as(b), torch.minimum(b, value_bins - 1))
        b = torch.minimum(b, torch.tensor([bins[j] - 1 for j in mem], device="cuda", dtype=torch.float32))
        for c, j in enumerate(mem):
            if j not in informative:
                continue
            v, k = x[:, c], len([i for i in informative if i < j])
            term = (v > 0.3 + 0.05 * k).float() if k % 3 == 0 else (v - 0.5).abs() if k % 3 == 1 else v
            signal += (1.5 if k % 2 else -1.2) * term / (1 + 0.15 * k)
            if held is not None and k % 4 == 3:
                signal += 0.8 * ((v > 0.5) & (held > 0.5)).float()
            held = v
        if wide:
            stride = (2 * len(mem) + 3) // 4 * 4
            data = torch.zeros(rows, stride // 2, dtype=torch.int16, device="cuda")
            data[:, : len(mem)] = b.to(torch.int16)
            data = data.view(torch.uint8)
        else:
            stride = (len(mem) + 3) // 4 * 4
            data = torch.zeros(rows, stride, dtype=torch.uint8, device="cuda")
            data[:, : len(mem)] = b.to(torch.uint8)
        groups.append(FeatureGroup(list(mem), stride, features[mem[0]].hist_offset, sum(bins[j] for j in mem),
                                   data.reshape(-1).cpu().numpy(), 16 if wide else 8))
        del u, x, b, data
    if wide:
        for m in features:
            m.column *= 2  # a two-byte bin's column is its byte offset in the row
    signal = (signal - signal.mean()) / signal.std().clamp_min(1e-6)
    objective, queries, weight = case.get("objective", "regression"), None, None
    noise = torch.randn(rows, generator=gen, device="cuda")
    if objective == "binary":
        label = (rnd(rows) < torch.sigmoid(1.5 * signal - 0.5)).float()
    elif objective == "lambdarank":  # labels 0-4, most of them low; queries of 10 to 200 documents, short ones common
        s = signal + 0.7 * noise
        label = sum((s > t).float() for t in (0.3, 0.9, 1.5, 2.2))
        r = np.random.default_rng(seed)
        sizes = (10.0 * 20.0 ** (r.random(rows // 10 + 1) ** 1.5)).astype(np.int64)
        ends = np.cumsum(sizes)
        queries = np.concatenate([[0], ends[ends < rows], [rows]]).astype(np.uint32)
    else:
        label = 2.0 * signal + 0.5 * noise
    if case.get("weighted"):
        weight = (0.5 + rnd(rows)).cpu().numpy()
    return BinnedDataset(rows, features, groups, total, label.cpu().numpy(), weight, query_boundaries=queries)


def _split(data, feature, threshold):
    """The split of a numerical feature at ``threshold``, missing values to the right."""
    m = data.features[feature]
    if data.groups[m.group].bin_bits == 16:
        return wide_bin_split(m.group, m.column, threshold)
    return bin_split(m.group, m.column, range(threshold + 1))


def _config(min_data=20):
    return _abi.SplitConfig(min_data, 1e-3, 0.0, 0.0, 0.0, 4, 32, 10.0, 10.0, 100)


def _custom_gradients(data, seed):
    """Gradients of a program's own objective, as the host hands them to the backend."""
    r = np.random.default_rng(seed + 5)
    label = np.asarray(data.label, np.float32)
    g = (r.standard_normal(data.num_rows).astype(np.float32) * np.float32(0.5) - (label - label.mean())).astype(np.float32)
    h = (0.05 + 0.2 * r.random(data.num_rows)).astype(np.float32)
    return g, h


def _quant_spec(max_grad, max_hess, quant_bins=4):
    gs, hs = max_grad / (quant_bins // 2), max_hess / quant_bins
    return _abi.QuantSpec(np.float32(1.0 / gs), np.float32(1.0 / hs), gs, hs, quant_bins // 2, quant_bins, 0, 0,
                          (C.c_uint8 * 2)(), 1, 0)


def _random_tree(case, data, seed):
    """A tree of the case's leaves over random numerical splits, children after their parent, and its leaf values."""
    r = np.random.default_rng(seed + 9)
    numeric = [j for j, m in enumerate(data.features) if m.kind == _abi.BINS_NUMERICAL and m.num_bins > 2]
    left, right, rule, ends = [], [], [], [(-1, False)]
    for k in range(case["leaves"] - 1):
        leaf = int(r.integers(0, min(len(ends), 24)))
        parent, went_right = ends[leaf]
        if parent >= 0:
            (right if went_right else left)[parent] = k
        left.append(~leaf)
        right.append(~len(ends))
        ends[leaf] = (k, False)
        ends.append((k, True))
        j = numeric[int(r.integers(0, len(numeric)))]
        rule.append((j, int(r.integers(0, data.features[j].num_bins - 2))))
    values = (0.1 * r.standard_normal(case["leaves"])).astype(np.float32)
    return left, right, rule, values


# ---- prepare ----------------------------------------------------------------------------------------------------


def _params(case):
    p = dict(objective=case["objective"], num_leaves=case["leaves"], num_grad_quant_bins=case.get("quant_bins", 4),
             num_iterations=case["rounds"])
    if case.get("bagging", 1.0) < 1.0:
        p.update(bagging_fraction=case["bagging"], bagging_freq=1)
    if case.get("feature_fraction", 1.0) < 1.0:
        p["feature_fraction"] = case["feature_fraction"]
    return p


def prepare(case, seed):
    kind = case["kind"]
    data = _table(case, case["rows"], seed)
    valid = (_table(case, case["valid_rows"], seed + 500_009),) if case.get("valid_rows") else ()
    state = dict(case=case, data=data, valid=valid)
    if kind == "train":
        state["params"] = _params(case)
        return state
    if kind == "boost":
        state["trainer"] = silvic_amd.Trainer(_params(case), data, valid_sets=valid)
        return state
    be = silvic_amd.RocmBackend()
    be.load(data, objective=OBJECTIVES[case.get("objective", "regression")])
    state["backend"] = be
    if kind == "rows":
        left, right, rule, values = _random_tree(case, data, seed)
        state["nodes"] = [device_node(_split(data, j, t), lc, rc) for lc, rc, (j, t) in zip(left, right, rule)]
        state["values"] = values
        return state
    g, h = _custom_gradients(data, seed)
    max_grad, max_hess = be.set_gradients(g, h)
    state["spec"] = _quant_spec(max_grad, max_hess)
    be.quantize(state["spec"])
    if kind == "learner":
        if case["slots"]:
            be.hist_slots(case["leaves"])
        return state
    rows = be.reset_partition()
    left = be.partition((0, rows), _split(data, 0, _threshold(case, data)))
    state["leaf"] = (0, left)
    state["out"] = torch.empty(2 * data.total_bins, dtype=torch.int64, device="cuda")
    return state


def _threshold(case, data):
    """The threshold of feature 0 that sends about ``share`` of the rows left."""
    values = data.features[0].num_bins - 1
    return max(0, min(values - 1, int(case["share"] / 0.9 * values)))


# ---- run ---------------------------------------------------------------------------------------------------------

TREE_KEYS = ("split_feature", "threshold_bin", "default_left", "left_child", "right_child", "split_gain",
             "internal_value", "internal_weight", "internal_count", "leaf_value", "leaf_weight", "leaf_count",
             "leaf_parent", "leaf_depth", "leaf_range", "left_bins")


def _trees(trees):
    out = {k: np.concatenate([t[k].reshape(-1) for t in trees]) for k in TREE_KEYS}
    out["num_leaves"] = np.array([t["num_leaves"] for t in trees])
    return out


def run(state):
    return {"boost": _run_boost, "train": _run_train, "learner": _run_learner, "histogram": _run_histogram,
            "histogram_host": _run_histogram_host, "rows": _run_rows}[state["case"]["kind"]](state)


def _run_boost(state):
    t = state["trainer"]
    for d in range(1 + len(state["valid"])):  # the run starts over
        t.backend.init_scores(d, t.init_score)
    t.iteration, t.finished = 0, False
    t.trees.clear()
    out = _trees(t.step(state["case"]["rounds"]))
    if state["data"].num_rows <= 500_000:  # the training metric of a run this short
        out["scores"] = t.backend.scores(0)
    if state["valid"]:
        out["valid_scores"] = t.backend.scores(1)
    return out


def _run_train(state):
    booster = silvic_amd.train(state["params"], state["data"], valid_sets=state["valid"])
    return _trees(booster.trees)


def _run_learner(state):
    """Best-first growth, one split at a time: the smaller child's histogram is built, the other is the difference."""
    be, data, spec, slots = state["backend"], state["data"], state["spec"], state["case"]["slots"]
    cfg, feats, limit = _config(), data.features, state["case"]["leaves"]
    every = np.ones(len(feats), bool)
    built = []
    rows = be.reset_partition()
    first = feats[0]
    if slots:
        be.histogram_slot((0, rows), 0)
        root, free = 0, 1
        head = be.read_slot(0)
    else:
        root = head = be.histogram((0, rows))
    built.append(head)
    pairs = head.reshape(-1, 2)[first.hist_offset : first.hist_offset + first.num_bins]

    def search(hist, sums, evaluate):
        find = be.find_best_split_slot if slots else be.find_best_split
        return find(hist, feats, evaluate, sums, spec.grad_scale, spec.hess_scale, cfg)

    leaves, heap = [(0, rows)], []

    def queue(leaf, hist, sums, evaluate):
        info, splittable = search(hist, sums, evaluate)
        if info.found and info.gain > 0:
            heapq.heappush(heap, (-info.gain, leaf, hist, info, splittable))

    queue(0, root, (float(pairs[:, 0].sum()), float(pairs[:, 1].sum()), rows), every)
    picked = []
    while heap and len(leaves) < limit:
        _, leaf, hist, info, splittable = heapq.heappop(heap)
        begin, count = leaves[leaf]
        m = feats[info.feature]
        if data.groups[m.group].bin_bits == 16:
            split = wide_bin_split(m.group, m.column, info.threshold, m.num_bins - 1 if info.default_left else None)
        else:
            split = bin_split(m.group, m.column, list(range(info.threshold + 1)) + [m.num_bins - 1] * int(info.default_left))
        side = 0 if info.left.count <= info.right.count else 1
        if slots:
            left = be.partition_and_histogram_slot((begin, count), split, side, free)
            child, free = free, free + 1
        else:
            left, child = be.partition_and_histogram((begin, count), split, side)
            built.append(child)
        picked.append((leaf, info.feature, info.threshold, info.default_left, left, count - left, info.gain,
                       info.left_output, info.right_output))
        new = len(leaves)
        leaves[leaf] = (begin, left)
        leaves.append((begin + left, count - left))
        if len(leaves) == limit:
            break
        if slots:
            be.subtract(hist, child)
            other = hist
        else:
            other = hist - child
        for at, s, k in ((leaf, info.left, 0), (new, info.right, 1)):
            queue(at, child if k == side else other, (s.grad, s.hess, leaves[at][1]), splittable)
    return {"splits": np.array(picked, np.float64), "leaves": np.array(leaves, np.int64), "root": built[0],
            "built": np.concatenate(built[1:]) if len(built) > 1 else built[0], "rows": be.partition_rows()}


def _run_histogram(state):
    be, out = state["backend"], state["out"]
    rc = _abi.load_rocm().srocm_histogram_noalloc(be._h, _abi.LeafRange(*state["leaf"]), out.data_ptr(), out.numel(), 0)
    if rc != _abi.OK:
        raise RuntimeError("srocm_histogram_noalloc failed")
    return out


def _run_histogram_host(state):
    return state["backend"].histogram(state["leaf"])


def _run_rows(state):
    be, case = state["backend"], state["case"]
    be.init_scores(0, 0.25)
    be.add_tree(state["nodes"], state["values"])
    max_grad, max_hess = be.compute_gradients()
    spec = _quant_spec(max_grad, max_hess)
    be.quantize(spec)
    kept = be.reset_partition(_abi.Bag(_abi.BAG_BERNOULLI, 3, 0, 0, case["bagging"]))
    edges = [kept * i // 16 for i in range(17)]
    sums = be.leaf_sums([(a, b - a) for a, b in zip(edges, edges[1:])], float(2**20), float(2**20))
    return {"maxima": np.array([max_grad, max_hess]), "kept": kept, "sums": sums, "scores": be.scores(0)}


# ---- work, tolerance, exact -----------------------------------------------------------------------------------------


def work(case):
    """A pass reads the binned rows it is about once for each histogram from scratch (a tree's root) and, below the
    root, the bins of the smaller children: about a third of the parent's rows at each of log2(leaves) levels."""
    rows, width = case["rows"], case["features"] * (2 if case["max_bin"] > 256 else 1)
    cells = rows * case["features"]
    kind = case["kind"]
    if kind in ("histogram", "histogram_host"):
        n = case["share"] * rows
        total = sum(_columns(case)[0])
        return dict(bytes=n * (width + 8) + 16 * total, flops=2 * case["share"] * cells)
    levels = math.log2(max(2, case["leaves"]))
    if kind == "rows":  # tree walk, scores, gradients, quantized words, the bag's rows and their sums
        return dict(bytes=rows * (levels + 8 + 12 + 12 + 4 + 12 + 4), flops=rows * (2 * levels + 40))
    trees = 1 if kind == "learner" else case["rounds"]
    if case.get("bagging", 1.0) < 1.0:
        rows, cells = rows * case["bagging"], cells * case["bagging"]
    per = rows * (width + 8) + levels * rows * (9 + (width + 4) / 3) + 24 * rows
    upload = case["rows"] * width if kind == "train" else 0
    return dict(bytes=trees * per + upload, flops=trees * 2 * cells * (1 + levels / 3))


def tolerance(case):
    """Histograms and leaf sums are integers; split gains, leaf values and scores are the reference's f64 and f32
    operations in its order."""
    return "exact"


def _bin_columns(data):
    """Every feature's bins on the GPU, one at a time."""
    for j, m in enumerate(data.features):
        yield j, m, torch.from_numpy(np.ascontiguousarray(data.bin(j)).astype(np.int64)).cuda()


def _integer_histogram(data, g, h, rows):
    out = torch.zeros(data.total_bins, 2, dtype=torch.float64, device="cuda")
    for _, m, bins in _bin_columns(data):
        b = bins[rows]
        for k, w in enumerate((g, h)):
            out[m.hist_offset : m.hist_offset + m.num_bins, k] = torch.bincount(b, weights=w[rows], minlength=m.num_bins)
    return out.reshape(-1)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("boost", "train"):
        return None  # whole training runs: seconds to minutes in plain torch
    data = _table(case, case["rows"], seed)
    if kind == "rows":
        left, right, rule, values = _random_tree(case, data, seed)
        node = torch.zeros(case["rows"], dtype=torch.int64, device="cuda")
        bins = {j: torch.from_numpy(np.ascontiguousarray(data.bin(j)).astype(np.int64)).cuda() for j in {j for j, _ in rule}}
        for k, (lc, rc, (j, t)) in enumerate(zip(left, right, rule)):
            here = node == k
            node = torch.where(here, torch.where(bins[j] <= t, lc, rc), node)
        score = 0.25 + torch.from_numpy(values.astype(np.float64)).cuda()[~node]
        label = torch.from_numpy(data.label.astype(np.float64)).cuda()
        if case["objective"] == "binary":
            p = torch.sigmoid(score)
            g, h = p - (label > 0).double(), p * (1 - p)
        else:
            g, h = score - label, torch.ones_like(score)
        return {"maxima": torch.stack([g.abs().max(), h.max()]), "kept": None, "sums": None, "scores": score}
    g, h = _custom_gradients(data, seed)
    spec = _quant_spec(float(np.abs(g).max()), float(h.max()))
    units = [torch.from_numpy(np.rint(a * np.float32(s)).astype(np.float64)).cuda()
             for a, s in ((g, spec.inv_grad_scale), (h, spec.inv_hess_scale))]
    if kind == "learner":
        every = torch.arange(case["rows"], device="cuda")
        return {"splits": None, "leaves": None, "root": _integer_histogram(data, *units, every), "built": None, "rows": None}
    first = torch.from_numpy(np.ascontiguousarray(data.bin(0)).astype(np.int64)).cuda()
    rows = torch.nonzero(first <= _threshold(case, data)).reshape(-1)
    hist = _integer_histogram(data, *units, rows)
    return hist.to(torch.int64) if kind == "histogram" else hist
