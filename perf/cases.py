"""The work this package is used for, as cases that can be timed and compared.

Five kinds, all through the public operators (`tensornet_amd.core`, `tensornet_amd.ops`):

  step    one training step of an embedding layer whose combiner runs elsewhere: SparseTablePush of the gradients of
          the batch in hand, SparseTablePull of the batch again (the rows the next step computes with)
  pooled  the same step with the combiner on the device: push of the pooled gradients, pull, embedding_lookup_sparse
  serve   inference: pull, embedding_lookup_sparse
  shard   a server's share of a remote worker's step: SparseTable::Push of a request's records, SparseTable::Pull
  dense   DenseTablePushPull of a network's variables

A pass starts with the backward half of a step and ends with the forward half of the next one, so that what it returns
shows the updated rows.  A state is one table (two for "wide and deep") that holds its resident signs, one batch and
the gradients of it.
"""
import math

import numpy as np
import torch

import tensornet_amd as tn
import tensornet_amd.ops
from tensornet_amd import synth

LOOKUPS_MAX = 5_000_000   # lookups of one batch
FLOATS_MAX = 80_000_000   # lookups x row length: what the gradients and variables of a batch take at most
DENSE_MAX = 200_000_000   # parameters of a dense table


def listed():
    return [
        # the plumbing configuration of the benchmark: the smallest training step, where launches and waits count
        dict(name="step 1024x8 AdaGrad 8", kind="step", rows=1024, slots=8, ids=1.0, zipf=1.1, vocab=10**6,
             resident=10**6, fresh=0.0, opt="AdaGrad", dim=8, wide=False, cvm=False),
        # wide & deep with single-valued categorical features under Adam
        dict(name="step 4096x26 Adam 16", kind="step", rows=4096, slots=26, ids=1.0, zipf=1.05, vocab=10**8,
             resident=2 * 10**7, fresh=0.0, opt="Adam", dim=16, wide=False, cvm=False),
        # two tables per step, dim-1 Ftrl weights and dim-64 AdaGrad embeddings of the same signs, many of them rare
        dict(name="step 8192x40 wide+deep 64", kind="step", rows=8192, slots=40, ids=1.0, zipf=1.1, vocab=10**8,
             resident=10**7, fresh=0.2, opt="AdaGrad", dim=64, wide=True, cvm=False),
        # a large batch of single-valued features on a large table
        dict(name="step 32768x64 AdaGrad 16", kind="step", rows=32768, slots=64, ids=1.0, zipf=1.2, vocab=10**9,
             resident=10**8, fresh=0.0, opt="AdaGrad", dim=16, wide=False, cvm=False),
        # the headline configuration of the benchmark: multi-valued features, five million lookups a batch
        dict(name="step 16384x100x3 AdaGrad 16", kind="step", rows=16384, slots=100, ids=3.0, zipf=1.1, vocab=10**9,
             resident=10**8, fresh=0.0, opt="AdaGrad", dim=16, wide=False, cvm=False),
        # rows with the two show / click columns, a batch of no round size
        dict(name="step 3001x47x2 cvm 8", kind="step", rows=3001, slots=47, ids=2.0, zipf=1.1, vocab=10**8,
             resident=10**7, fresh=0.01, opt="AdaGrad", dim=8, wide=False, cvm=True),
        # a model with more slots than the slot masks have bits, combiner on the device
        dict(name="pooled 2039x211x2 sqrtn", kind="pooled", rows=2039, slots=211, ids=2.0, zipf=1.1, vocab=10**8,
             resident=10**7, fresh=0.0, opt="AdaGrad", dim=16, combiner="sqrtn"),
        # the headline configuration with the combiner on the device
        dict(name="pooled 16384x100x3 mean", kind="pooled", rows=16384, slots=100, ids=3.0, zipf=1.1, vocab=10**9,
             resident=10**8, fresh=0.0, opt="AdaGrad", dim=16, combiner="mean"),
        # a request of a ranking service: a few hundred candidates
        dict(name="serve 256x26x3 sum", kind="serve", rows=256, slots=26, ids=3.0, zipf=1.1, vocab=10**8,
             resident=10**7, fresh=0.0, opt="AdaGrad", dim=16, combiner="sum"),
        # what one worker's step sends to a server: a record per distinct sign of each of its slots
        dict(name="shard 40x1500 AdaGrad 16", kind="shard", slots=40, records=1500, vocab=10**8, resident=10**7,
             fresh=0.0, opt="AdaGrad", dim=16),
        # the dense part of a wide & deep model: three hidden layers over concatenated embeddings
        dict(name="dense mlp 3x512 Adam", kind="dense", inputs=429, width=512, layers=3, opt="Adam"),
        # a flat array that only bandwidth bounds
        dict(name="dense flat 2e8 Adam", kind="dense", inputs=2 * 10**8, width=1, layers=0, opt="Adam"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step"] * 5 + ["pooled"] * 3 + ["serve", "shard", "shard", "dense", "dense"])
    if kind == "dense":
        opt = rng.choice(["Adam", "Adam", "AdaGrad"])
        if rng.random() < 0.3:
            return dict(kind=kind, inputs=_log(rng, 1000, DENSE_MAX * (1.0 if opt == "Adam" else 0.8)), width=1, layers=0, opt=opt)
        return dict(kind=kind, inputs=_log(rng, 16, 4000), width=_log(rng, 16, 2048), layers=rng.randint(1, 8), opt=opt)
    vocab = _log(rng, 10**5, 10**9)
    case = dict(kind=kind, vocab=vocab, resident=min(vocab, _log(rng, 10**5, 2 * 10**7)),
                fresh=round(rng.choice([0.0, 0.0, rng.uniform(0.0, 0.05), rng.uniform(0.0, 0.3)]), 3))
    dim = rng.choice([1, 4, 8, 8, 10, 12, 16, 16, 16, 32, 64])
    if kind == "shard":
        slots = _log(rng, 1, 300)
        records = _log(rng, 500, min(1_500_000, FLOATS_MAX // (4 * dim))) // slots
        return dict(case, slots=slots, records=max(1, min(records, vocab // 2)), opt=rng.choice(["AdaGrad", "Adam", "Ftrl"]), dim=dim)
    case["zipf"] = round(rng.uniform(1.02, 1.3), 3)
    ids = rng.choice([1.0, 1.0, round(rng.uniform(1.2, 6.0), 1)])
    if kind == "serve":
        rows, slots = _log(rng, 1, 4096), _log(rng, 4, 300)
    else:
        rows, slots = _log(rng, 60, 40000), _log(rng, 1, 300)
    most = min(LOOKUPS_MAX // 2, FLOATS_MAX // (2 * dim))
    rows = max(1, min(rows, int(most / (slots * ids))))
    case.update(rows=rows, slots=slots, ids=ids, dim=dim)
    if kind == "step":
        opt = rng.choice(["AdaGrad", "AdaGrad", "Adam", "Ftrl"])
        return dict(case, opt=opt, wide=rng.random() < 0.15, cvm=opt == "AdaGrad" and rng.random() < 0.3)
    # (sums of a sign's gradients may be associated differently; Adam divides by their magnitude)
    return dict(case, opt=rng.choice(["AdaGrad", "AdaGrad", "Ftrl"]), combiner=rng.choice(["sum", "mean", "sqrtn"]))


HYPER = {
    "AdaGrad": dict(learning_rate=0.01, initial_g2sum=0.1, epsilon=1e-8),
    "Adam": dict(learning_rate=1e-3, beta1=0.9, beta2=0.999, epsilon=1e-8),
    "Ftrl": dict(learning_rate=0.05, beta=1.0, lambda1=1.0, lambda2=1.0),
}
CLICK_RATE = 0.2  # share of lookups whose example was clicked
LOAD_CHUNK = 1 << 23


class Table:
    """A sparse table with its resident signs splitmix64(1 .. resident); gives its memory back when it goes."""

    def __init__(self, opt, dim, cvm, resident, room, seed):
        self.handle = tn.core.create_sparse_table(getattr(tn.core, opt)(**HYPER[opt]), "", dim, cvm, "")
        self.width = dim + (2 if cvm else 0)
        tn.core.reserve_sparse_table(self.handle, resident + room)
        tn.core.set_sparse_table_seed(self.handle, seed)
        for lo in range(1, resident + 1, LOAD_CHUNK):
            signs = synth.splitmix64_torch(torch.arange(lo, min(resident + 1, lo + LOAD_CHUNK), device="cuda"))
            rows = synth.snapshot_rows_torch(signs, self.width, seed=seed)
            rows[:, dim:] = 0
            tn.ops.table_load_rows(self.handle, signs, rows)

    def __del__(self):
        tn.core.clear_sparse_table(self.handle)


def _signs(case, n, gen):
    """n signs: splitmix64 of bounded Zipf ids; a share `fresh` of them uniform, unlikely to be resident."""
    a = 1.0 - case["zipf"]
    u = torch.rand(n, dtype=torch.float64, device="cuda", generator=gen)
    ids = (1.0 + u * (float(case["vocab"]) ** a - 1.0)) ** (1.0 / a)
    return _some_fresh(case, synth.splitmix64_torch(ids.long().clamp_(1, case["vocab"])), gen)


def _some_fresh(case, signs, gen):
    if case["fresh"] == 0:
        return signs
    uniform = torch.randint(-(1 << 62), 1 << 62, signs.shape, device="cuda", generator=gen)
    return torch.where(torch.rand(signs.shape, device="cuda", generator=gen) < case["fresh"], uniform, signs)


def _request(case, gen):
    """The signs of a request, slot by slot and distinct within a slot: the ids of a slot lie evenly on a logarithmic
    scale (about what is left of Zipf draws without their repeats), so the frequent ones are in every slot."""
    slots, records = case["slots"], case["records"]
    at = torch.arange(records, device="cuda")
    u = torch.rand((slots, records), dtype=torch.float64, device="cuda", generator=gen)
    ids = (float(case["vocab"]) ** ((at + u) / records)).long()
    ids = (ids - at).cummax(1).values + at  # strictly ascending
    ids = ids.gather(1, torch.rand((slots, records), device="cuda", generator=gen).argsort(1))
    signs = synth.splitmix64_torch(ids.reshape(-1))
    return _some_fresh(case, signs, gen)


def _rows_per_slot(flat, counts):
    """Per-slot matrices of the given numbers of rows out of one allocation; every slot starts at a multiple of eight rows."""
    out, at = [], 0
    for c in counts:
        out.append(flat[at:at + c])
        at += -(-c // 8) * 8
    return out


def _total_rows(counts):
    return sum(-(-c // 8) * 8 for c in counts)


def _joined(views, shape):
    """The whole buffer behind the per-slot tensors an operator returns (it hands out views of one allocation)."""
    stride = [1] * len(shape)
    for i in range(len(shape) - 2, -1, -1):
        stride[i] = stride[i + 1] * shape[i + 1]
    return torch.as_strided(views[0], shape, stride)


class Batch:
    """One batch as a data loader leaves it on the device: per slot the signs, the labels and the lookups' examples."""

    def __init__(self, case, gen):
        rows, slots = case["rows"], case["slots"]
        if case["ids"] == 1.0:
            lens = torch.ones((slots, rows), dtype=torch.int64, device="cuda")
        else:
            # multi-valued features: at most twenty values; a list may be empty where the combiner can say so.  The
            # slots' totals are those of the case, which example has how many values is the seed's.
            fixed = torch.Generator(device="cuda")
            fixed.manual_seed(20)
            mean = torch.full((slots, rows), case["ids"], device="cuda")
            lens = torch.poisson(mean, generator=fixed).long().clamp_(1 if case["kind"] == "step" else 0, 20)
            lens = lens.gather(1, torch.rand((slots, rows), device="cuda", generator=gen).argsort(1))
        self.counts = [int(c) for c in lens.sum(1).cpu()]
        self.lookups = sum(self.counts)
        self.values = list(_signs(case, self.lookups, gen).split(self.counts))
        labels = (torch.rand(self.lookups, device="cuda", generator=gen) < CLICK_RATE).long()
        self.labels = list(labels.split(self.counts))
        example = torch.arange(rows, device="cuda").repeat(slots).repeat_interleave(lens.reshape(-1))
        self.examples = list(example.split(self.counts))


class State:
    pass


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    s = State()
    s.case = case
    kind = case["kind"]
    if kind == "dense":
        s.vars = [(torch.rand(shape, device="cuda", generator=gen) - 0.5) * 0.1 for shape in _dense_shapes(case)]
        s.grads = [torch.randn(v.shape, device="cuda", generator=gen) * 1e-4 for v in s.vars]
        s.handle = tn.core.create_dense_table(getattr(tn.core, case["opt"])())
        tn.ops.dense_table_init(s.vars, s.handle)
        return s
    if kind == "shard":
        n, dim = case["slots"] * case["records"], case["dim"]
        s.table = Table(case["opt"], dim, False, case["resident"], n, seed)
        s.signs = _request(case, gen)
        shows = torch.randint(1, 4, (n,), device="cuda", generator=gen)
        s.infos = tn.ops.make_sign_infos(s.signs, shows, (torch.rand(n, device="cuda", generator=gen) < CLICK_RATE).long())
        s.grads = torch.randn((n, dim), device="cuda", generator=gen) * 1e-2
        tn.ops.table_pull(s.table.handle, s.signs, dim)
        return s
    s.batch = b = Batch(case, gen)
    rows, slots = case["rows"], case["slots"]
    tables = [(case["opt"], case["dim"])]
    if kind == "step" and case["wide"]:
        tables.insert(0, ("Ftrl", 1))
    s.parts = []
    for opt, dim in tables:
        p = State()
        cvm = kind == "step" and case["cvm"] and opt == "AdaGrad"
        p.table = Table(opt, dim, cvm, case["resident"], b.lookups, seed)
        width = p.table.width
        # a variable has a row for every distinct sign there can be, and one more
        var_rows = [c + 1 for c in b.counts]
        p.flat = torch.zeros((_total_rows(var_rows), width), device="cuda")
        p.vars = _rows_per_slot(p.flat, var_rows)
        if kind == "step":
            p.grads = _rows_per_slot(torch.randn((_total_rows(b.counts), width), device="cuda", generator=gen) * 1e-2, b.counts)
        elif kind == "pooled":
            p.grads = list((torch.randn((slots, rows, width), device="cuda", generator=gen) * 1e-2).unbind(0))
        # single-valued features come in tensors of fixed shape: the operators are bound to them once
        p.pull = p.push = None
        if kind == "step" and case["ids"] == 1.0:
            p.pull = tn.ops.BoundSparseTablePull(p.vars, b.values, p.table.handle)
            p.push = tn.ops.BoundSparseTablePush(b.values, p.grads, b.labels, p.table.handle)
        if kind != "serve":
            _pull(b, p)
        s.parts.append(p)
    return s


def _pull(b, p):
    return p.pull() if p.pull else tn.ops.sparse_table_pull(p.vars, b.values, p.table.handle)


def run(s):
    case = s.case
    kind = case["kind"]
    if kind == "dense":
        tn.ops.dense_table_push_pull(s.vars, s.grads, 1e-3, s.handle)
        return s.vars
    if kind == "shard":
        tn.ops.table_push(s.table.handle, s.infos, s.grads)
        return tn.ops.table_pull(s.table.handle, s.signs, case["dim"])
    b = s.batch
    out = []
    for p in s.parts:
        h = p.table.handle
        if kind == "pooled":
            tn.ops.sparse_table_push_pooled(b.values, b.examples, p.grads, b.labels, h, case["combiner"])
        elif kind == "step":
            if p.push:
                p.push()
            else:
                tn.ops.sparse_table_push(b.values, p.grads, b.labels, h)
        mapped = _pull(b, p)
        out += [_joined(mapped, (b.lookups,)), p.flat]
        if kind != "step":
            pooled = tn.ops.embedding_lookup_sparse(p.vars, mapped, b.examples, case["rows"], h, case["combiner"])
            out.append(_joined(pooled, (case["slots"], case["rows"], p.table.width)))
    return out


def _dense_shapes(case):
    if case["layers"] == 0:
        return [(case["inputs"],)]
    shapes, fan_in = [], case["inputs"]
    for _ in range(case["layers"]):
        shapes += [(fan_in, case["width"]), (case["width"],)]
        fan_in = case["width"]
    return shapes + [(fan_in, 1), (1,)]


def _distinct(case, n):
    """Expected distinct signs among n draws."""
    a, vocab = 1.0 - case["zipf"], float(case["vocab"])
    drawn = n * (1.0 - case["fresh"])
    edges = np.unique(np.concatenate([np.arange(1.0, 2001.0), np.geomspace(2001.0, max(vocab, 2002.0), 4000)]))
    edges = edges[edges <= vocab]
    cdf = (edges ** a - 1.0) / (vocab ** a - 1.0)
    ids, share = np.diff(edges), np.diff(cdf)
    return float(np.sum(ids * -np.expm1(-drawn * share / ids))) + n * case["fresh"]


def _state_floats(opt, dim):
    return 4 if opt == "AdaGrad" else 2 * dim + 2


def work(case):
    kind = case["kind"]
    if kind == "dense":
        n = sum(math.prod(shape) for shape in _dense_shapes(case))
        # gradient in; weights and optimizer state in and out; variable out
        states = 2 if case["opt"] == "Adam" else 3
        return {"bytes": (4 + 8 + 8 * states + 4) * n, "flops": 12 * n}
    if kind == "shard":
        n, dim = case["slots"] * case["records"], case["dim"]
        edges = np.unique(np.geomspace(1.0, float(case["vocab"]), 4000).astype(np.int64)).astype(np.float64)
        share = np.minimum(1.0, case["records"] * np.log(edges[1:] / edges[:-1]) / math.log(case["vocab"]) / np.diff(edges))
        keys = min(n, float(np.sum(np.diff(edges) * (1.0 - (1.0 - share) ** case["slots"]))) * (1.0 - case["fresh"]) + n * case["fresh"])
        # records, gradients, signs in, rows out; per distinct sign its key, its row and its state in and out
        return {"bytes": n * (16 + 4 * dim + 8 + 4 * dim) + keys * (8 + 8 * dim + 8 * _state_floats(case["opt"], dim)),
                "flops": 8 * n * dim}
    ids = case["ids"] if case["ids"] == 1.0 or kind != "step" else case["ids"] + math.exp(-case["ids"])
    lookups = case["rows"] * case["slots"] * ids
    records = case["slots"] * _distinct(case, case["rows"] * ids)
    keys = _distinct(case, lookups)
    total = flops = 0.0
    for opt, dim in ([("Ftrl", 1)] if kind == "step" and case["wide"] else []) + [(case["opt"], case["dim"])]:
        width = dim + (2 if kind == "step" and case["cvm"] and opt == "AdaGrad" else 0)
        # signs in, mapped ids out; a variable row per record out; key and row of every distinct sign in
        total += 16 * lookups + 4 * width * records + keys * (8 + 4 * width)
        if kind != "step":  # example ids in, one row per example and slot out
            total += 8 * lookups + 4 * width * case["rows"] * case["slots"]
            flops += lookups * width
        if kind != "serve":  # labels in; row out, state in and out
            total += 8 * lookups + keys * (4 * width + 8 * _state_floats(opt, dim))
            flops += 8 * records * width
            # gradients in: a row per record, or one per example and slot
            total += 4 * width * (records if kind == "step" else case["rows"] * case["slots"])
            flops += 0 if kind == "step" else lookups * width
    return {"bytes": total, "flops": flops}


def tolerance(case):
    # whole numbers (mapped ids) are the same; rows are 32-bit sums
    return {"rel": 1e-5, "max": 1e-3}
