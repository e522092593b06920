"""The workloads the engine's speed is judged on, through its public calls.

A case is a dict of plain values; `prepare` builds what a program holds before
the call (instance context, node batch, trained selector), `run` makes one
pass.  Five paths:

host    Engine.bound on host buffers: a CPU explorer hands over one pool of
        nodes and waits for the bounds.
device  Engine.bound_device on a batch resident in HBM: bulk evaluation.
solve   Engine.solve, the device-resident search, to proven optimum or to a
        budget of decomposed parents.
mixed   Multi.run: the nodes of many instances of uneven size in one call.
train   Engine.selector_train on logged records, the learned selector's
        forward and backward pass, optimiser included.

Instances are drawn by the Taillard generator (times in [1, 99]) or, for
mixed batches, by the job-correlated one; nodes have prefix and suffix
lengths spread uniformly over a random permutation.
"""
import itertools
import random

import numpy as np
import torch

import wsbb_amd

MIXED_SHAPES = tuple(itertools.product((20, 50, 100), (5, 10, 20)))
RECORDS_STRIDE = 16  # every 16th child of a logging solve becomes a record


def listed():
    return [
        # one wavefront of nodes of the smallest Taillard class: the call's latency
        dict(name="host_20x5_64", path="host", n=20, m=5, nodes=64, kind="lb2"),
        # the reference's launch shape: pools of 4096 nodes, 20x10
        dict(name="host_20x10_4096", path="host", n=20, m=10, nodes=4096, kind="lb2"),
        # an ordinary resident batch of an odd size, the class learned selection targets
        dict(name="device_20x20_100k", path="device", n=20, m=20, nodes=100_003, kind="lb2"),
        # the headline batch: 2^20 nodes, 50x20
        dict(name="device_50x20_1m", path="device", n=50, m=20, nodes=1 << 20, kind="lb2"),
        # four job-mask words per node
        dict(name="device_100x10_64k", path="device", n=100, m=10, nodes=65_521, kind="lb2"),
        # 20x5 to proven optimum with the one-machine bound, one pool per round
        dict(name="solve_20x5_lb1", path="solve", n=20, m=5, kind="lb1", pool=4096, batches=1,
             budget=100_000),
        # 20x10 with the reference's ring of ten 4096-child pools
        dict(name="solve_20x10", path="solve", n=20, m=10, kind="lb2", pool=4096, batches=10,
             budget=200_000),
        # 20x20 at the widest measured pool shape
        dict(name="solve_20x20_wide", path="solve", n=20, m=20, kind="lb2", pool=65536, batches=8,
             budget=4_000_000),
        # 50x20 at the fastest measured pool shape, stopped by its budget
        dict(name="solve_50x20", path="solve", n=50, m=20, kind="lb2", pool=4096, batches=4,
             budget=100_000),
        # the same search as solve_20x20_wide with a selector trained on its instance
        dict(name="learned_20x20_wide", path="solve", n=20, m=20, kind="learned", pool=65536,
             batches=8, budget=4_000_000),
        # 64 instances of nine sizes in one launch
        dict(name="mixed_64", path="mixed", instances=64, nodes=4099),
        # one epoch of the online protocol's training
        dict(name="train_20x20", path="train", n=20, m=20, records=1 << 16, batch=2048),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng: random.Random):
    """One more case of the ranges above, odd sizes among them."""
    path = rng.choice(["host", "device", "device", "solve", "solve", "mixed", "train"])
    n = rng.choice([20, 50, 100, rng.randint(11, 101)])
    m = rng.choice([5, 10, 20, rng.randint(3, 20)])
    if path == "host":
        return dict(path=path, n=n, m=m, nodes=_log_int(rng, 1, 16384),
                    kind=rng.choice(["lb2", "lb2", "lb1"]))
    if path == "device":
        # up to the headline batch's work
        top = min(1 << 20, int((1 << 20) * 50 * 190 / (n * max(1, m * (m - 1) // 2))))
        return dict(path=path, n=n, m=m, nodes=_log_int(rng, 1000, top),
                    kind=rng.choice(["lb2", "lb2", "lb2", "lb1"]))
    if path == "solve":
        n = rng.choice([20, 20, 50, rng.randint(15, 60)])
        kind = rng.choice(["lb2", "lb2", "lb1", "learned"])
        if kind == "learned":
            m = max(m, 10)
        pool, batches = rng.choice([(4096, 1), (4096, 4), (4096, 10), (16384, 4), (65536, 4)])
        return dict(path=path, n=n, m=m, kind=kind, pool=pool, batches=batches,
                    budget=_log_int(rng, 2000, 100_000))
    if path == "mixed":
        return dict(path=path, instances=rng.randint(2, 64), nodes=_log_int(rng, 65, 4099))
    return dict(path=path, n=20, m=rng.choice([10, 15, 20]), records=_log_int(rng, 4096, 1 << 16),
                batch=rng.choice([512, 1024, 2048]))


KINDS = {"lb2": wsbb_amd.LB2, "lb1": wsbb_amd.LB1, "learned": wsbb_amd.LEARNED}


def _instance(case, seed):
    return wsbb_amd.generate(case["n"], case["m"], 1 + (seed * 7919 + 12345) % 2147483000)


def _nodes(n, count, seed):
    """Random nodes on the GPU: position-major permutations and limits."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    perm = torch.rand(count, n, generator=g, device="cuda").argsort(dim=1)
    d1 = (torch.rand(count, generator=g, device="cuda") * n).long().clamp_(max=n - 1)
    d2 = (torch.rand(count, generator=g, device="cuda") * (n - d1)).long()
    d2 = torch.minimum(d2, n - 1 - d1)
    return (perm.to(torch.uint8).t().contiguous(), (d1 - 1).to(torch.int32), (n - d2).to(torch.int32))


def _train_on_own_records(eng, records, epochs):
    """Logs records of a short plain solve and keeps `records` of them at most."""
    eng.selector_init(seed=1)
    eng.selector_config(topk=24, margin=-1, parents=True)
    eng.selector_log(stride=RECORDS_STRIDE, capacity=records)
    eng.solve(pool_size=65536, max_batches=4, budget=max(2000, records))
    feat, label = eng.selector_records()
    eng.selector_log(stride=0, capacity=0)
    eng.selector_set_records(feat, label)
    if epochs:
        eng.selector_train(epochs=epochs, batch=2048, lr=2e-3, seed=2)
    return label.shape[0]


def prepare(case, seed):
    path = case["path"]
    if path == "mixed":
        ps = [wsbb_amd.generate_correlated(*MIXED_SHAPES[i % len(MIXED_SHAPES)], seed * 1009 + i)
              for i in range(case["instances"])]
        per, maxn = case["nodes"], max(p.shape[1] for p in ps)
        total = per * len(ps)
        perm = np.zeros((maxn, total), np.uint8)
        l1, l2 = np.zeros(total, np.int32), np.zeros(total, np.int32)
        for i, p in enumerate(ps):
            a, b, c = _nodes(p.shape[1], per, seed * 1013 + i)
            at = slice(i * per, (i + 1) * per)
            perm[:p.shape[1], at], l1[at], l2[at] = a.cpu().numpy(), b.cpu().numpy(), c.cpu().numpy()
        multi = wsbb_amd.Multi(ps)
        multi.load(perm, l1, l2, np.arange(len(ps) + 1, dtype=np.int32) * per)
        return dict(case=case, multi=multi)
    eng = wsbb_amd.Engine(_instance(case, seed))
    state = dict(case=case, eng=eng)
    if path in ("host", "device"):
        perm, l1, l2 = _nodes(case["n"], case["nodes"], seed)
        if path == "host":
            perm, l1, l2 = perm.cpu().numpy(), l1.cpu().numpy(), l2.cpu().numpy()
        else:
            state["out"] = torch.empty(case["nodes"], dtype=torch.int32, device="cuda")
        state.update(perm=perm, l1=l1, l2=l2)
    elif path == "train":
        _train_on_own_records(eng, case["records"], epochs=0)
    elif case["kind"] == "learned":
        _train_on_own_records(eng, 1 << 14, epochs=2)
    return state


def run(state):
    case = state["case"]
    path = case["path"]
    if path == "mixed":
        out, stats, _ = state["multi"].run(kind=wsbb_amd.LB2)
        return dict(bound=out, nodes=stats["nodes"], pairs=stats["pairs"])
    eng = state["eng"]
    if path == "host":
        return eng.bound(state["perm"], state["l1"], state["l2"], kind=KINDS[case["kind"]])
    if path == "device":
        eng.bound_device(state["perm"].data_ptr(), state["l1"].data_ptr(), state["l2"].data_ptr(),
                         case["nodes"], state["out"].data_ptr(), kind=KINDS[case["kind"]])
        return state["out"]
    if path == "train":
        eng.selector_init(seed=1)
        losses = eng.selector_train(epochs=1, batch=case["batch"], lr=2e-3, seed=2)
        return dict(losses=losses, **eng.selector_params())
    res = eng.solve(kind=KINDS[case["kind"]], pool_size=case["pool"], max_batches=case["batches"],
                    budget=case["budget"])
    return dict(best=res["best"], perm=res["perm"], proven=res["proven"],
                stats=np.array([res["stats"][k] for k in wsbb_amd.STAT_NAMES], np.int64))


def _node_ops(n, m, kind):
    """Integer operations of one node's bound at the mean prefix and suffix:
    heads and tails, then per machine pair a step per free job (LB1: per
    machine a sum over the free jobs)."""
    d1, d2 = (n - 1) / 2, (n - 1) / 4
    u = n - d1 - d2
    base = 2 * m * (d1 + d2)
    return base + (m * (u + 3) if kind == "lb1" else m * (m - 1) // 2 * (4 * u + 4))


def work(case):
    path = case["path"]
    if path == "mixed":
        b = f = 0.0
        for i in range(case["instances"]):
            n, m = MIXED_SHAPES[i % len(MIXED_SHAPES)]
            b += case["nodes"] * (n + 12.0)
            f += case["nodes"] * _node_ops(n, m, "lb2")
        return dict(bytes=b, flops=f)
    n, m = case["n"], case["m"]
    if path in ("host", "device"):
        return dict(bytes=case["nodes"] * (n + 12.0), flops=case["nodes"] * _node_ops(n, m, case["kind"]))
    if path == "train":
        feat, hidden, pairs = 5 * m, 128, m * (m - 1) // 2
        weights = feat * hidden + hidden + hidden * pairs + pairs
        steps = -(-case["records"] // case["batch"])
        return dict(bytes=case["records"] * 4.0 * (feat + 1) + steps * 24.0 * weights,
                    flops=6.0 * case["records"] * weights)
    # per decomposed parent: its node in and out of the pool, its children's
    # descriptors and bounds; about n children each
    kids = case["budget"] * float(n)
    pairs = 24 / (m * (m - 1) / 2) if case["kind"] == "learned" else 1.0
    return dict(bytes=case["budget"] * 2.0 * (n + 16) + kids * 8.0,
                flops=kids * _node_ops(n, m, "lb1" if case["kind"] == "lb1" else "lb2") * min(1.0, pairs))


def exact(case, seed):
    """Bounds and search results are whole numbers and have to stay equal;
    the training's result depends on its own shuffling, which plain torch
    does not reproduce."""
    return None
