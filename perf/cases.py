"""The work that programs on this framework have it do, as measurable cases.

A case is a dict of plain values.  Five kinds of call cover the public entry points on the
probe path:

  lookup     Index.lookup over an index that the program keeps: every index kind, 4- and
             8-byte keys, the plain, blockwise-sorting, partitioned and hash-join drivers
  build      Index construction over a sorted column, a lookup, and the index dropped again
             (a query that indexes its build side for itself)
  partition  gj_partition, the radix partitioner on its own, into buffers the program keeps
  aggregate  join_aggregate, the filter / lookup / sum over a fact table
  train      mlp_loss_grad, one training step's loss and gradients of the MLP root

Sizes follow bench.py and bench_suite.py (2^20 and 2^26 keys, 2^24 to 2^28 probes, a
2e6-row dimension under 6e7 fact rows, minibatches of 65536) and the tests' odd sizes.
Inputs live in torch tensors on the GPU and are handed over by pointer; torch's default
stream and the framework's default stream are the same one.
"""
import ctypes
import math

import numpy as np
import torch

import gpujoin_amd as gj

KEY_SPACE = 1 << 63  # 8-byte keys are drawn from [0, 2^63), 4-byte keys from [0, 2^32)


class View:
    """A torch tensor with the attributes that the framework's calls read of a buffer."""

    def __init__(self, tensor, dtype):
        self.tensor = tensor
        self.dtype = np.dtype(dtype)
        self.count = tensor.numel()
        self.ptr = ctypes.c_void_p(tensor.data_ptr())

    def offset(self, elements):
        return ctypes.c_void_p(self.tensor.data_ptr() + int(elements) * self.dtype.itemsize)


# ---- the cases ---------------------------------------------------------------------------

def listed():
    return [
        # a point query's or a small batch's probes against a resident index: latency
        dict(name="lookup_small", op="lookup", approach="plain", kind="learned_plr", key_bytes=8, n=1 << 20, m=1000,
             keys="uniform", probes="uniform", miss=0.0),
        # the 4-byte key configuration: a column that the caches hold
        dict(name="lookup_u32", op="lookup", approach="plain", kind="learned_plr", key_bytes=4, n=1 << 20, m=1 << 24,
             keys="uniform", probes="uniform", miss=0.0),
        # the headline configuration: the default learned index far beyond the caches
        dict(name="lookup_large", op="lookup", approach="plain", kind="learned_plr", key_bytes=8, n=1 << 26, m=1 << 28,
             keys="uniform", probes="uniform", miss=0.0),
        # the comparison index of every run, with the misses of a selective join
        dict(name="lookup_btree_misses", op="lookup", approach="plain", kind="btree", key_bytes=8, n=1 << 26,
             m=(1 << 26) - 77, keys="uniform", probes="uniform", miss=0.1),
        # a spline over skewed keys, an ordinary odd-sized batch
        dict(name="lookup_spline_skewed", op="lookup", approach="plain", kind="radix_spline", key_bytes=8, n=4_000_037,
             m=10_000_019, keys="lognormal", probes="uniform", miss=0.1),
        # the radix-partitioned driver at its default fan-out, eight windows
        dict(name="lookup_partitioned", op="lookup", approach="partitioning", kind="btree", key_bytes=8, n=1 << 25,
             m=1 << 25, keys="uniform", probes="uniform", miss=0.0, radix_bits=10, passes=1, window=1 << 22),
        # the blockwise-sorting driver over the column alone
        dict(name="lookup_sorted_blocks", op="lookup", approach="bws", kind="binary_search", key_bytes=8, n=1 << 22,
             m=1 << 24, keys="uniform", probes="uniform", miss=0.0),
        # a hash join: the table is built over the build side on every call
        dict(name="hash_join", op="lookup", approach="hj", kind="btree", key_bytes=8, n=1 << 22, m=1 << 24,
             keys="uniform", probes="uniform", miss=0.1),
        # the partitioner on its own, stable, at the driver's default fan-out
        dict(name="partition", op="partition", key_bytes=8, m=10_000_019, radix_bits=10, passes=1),
        # the fact-dimension aggregate: 30 of 2557 days qualify
        dict(name="join_aggregate", op="aggregate", strategy="lane_refill", kind="learned_plr", dim=2_000_000,
             rows=60_000_000),
        # the build side indexed for one query
        dict(name="build_learned", op="build", kind="learned_plr", key_bytes=8, n=12_345_677, m=1 << 20,
             keys="uniform", probes="uniform", miss=0.0),
        # one training step of the MLP root at its default width and minibatch
        dict(name="train_step", op="train", hidden=32, samples=65_536),
    ]


def log_size(rng, lo, hi):
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi))))


def draw(rng):
    op = rng.choice(["lookup", "lookup", "lookup", "bws", "partitioning", "hj", "build", "partition", "aggregate",
                     "train"])
    if op == "partition":
        return dict(op="partition", key_bytes=rng.choice([4, 8, 8]), m=log_size(rng, 1 << 14, 1 << 25),
                    radix_bits=rng.randint(4, 14), passes=rng.choice([1, 1, 2]))
    if op == "aggregate":
        return dict(op="aggregate",
                    strategy=rng.choice(["lane_refill", "lane_refill", "sorted", "partitioned", "plain",
                                         "lookup_first"]),
                    kind=rng.choice(["learned_plr", "learned_plr", "btree", "hash"]),
                    dim=log_size(rng, 1 << 12, 4_000_000), rows=log_size(rng, 1 << 16, 60_000_000))
    if op == "train":
        return dict(op="train", hidden=rng.choice([8, 16, 32, 32, 64]), samples=log_size(rng, 1 << 10, 1 << 22))
    key_bytes = rng.choice([4, 8, 8])
    case = dict(op="lookup", approach="plain", key_bytes=key_bytes,
                keys=rng.choice(["uniform", "uniform", "dense", "lognormal", "clustered"]),
                probes=rng.choice(["uniform", "uniform", "zipf", "sorted"]), miss=rng.choice([0.0, 0.0, 0.1, 0.5]))
    if op == "build":
        case.update(op="build", kind=rng.choice(["learned_plr", "learned_plr", "btree", "hash", "radix_spline"]),
                    n=log_size(rng, 1 << 12, 1 << 22), m=log_size(rng, 1 << 10, 1 << 20))
        del case["approach"]
    elif op == "hj":
        case.update(approach="hj", kind="btree", n=log_size(rng, 1 << 12, 1 << 24), m=log_size(rng, 1 << 14, 1 << 25))
    elif op == "partitioning":
        case.update(approach="partitioning", kind=rng.choice(["btree", "learned_plr", "binary_search"]),
                    n=log_size(rng, 1 << 16, 1 << 25), m=log_size(rng, 1 << 18, 1 << 25),
                    radix_bits=rng.randint(6, 12), passes=rng.choice([1, 1, 2]), window=1 << rng.randint(16, 24))
    elif op == "bws":
        case.update(approach="bws", kind=rng.choice(["binary_search", "btree", "harmonia", "learned_plr"]),
                    n=log_size(rng, 1 << 12, 1 << 24), m=log_size(rng, 1 << 12, 1 << 24))
    else:
        case.update(kind=rng.choice(["learned_plr", "learned_plr", "learned_mlp", "btree", "btree", "harmonia",
                                     "radix_spline", "hash", "binary_search"]),
                    n=log_size(rng, 1 << 12, 1 << 24), m=log_size(rng, 1 << 8, 1 << 25))
    if case["kind"] == "radix_spline":
        # the spline is fitted on the host: a build's pass stays shorter than the largest lookup
        case["n"] = min(case["n"], (1 << 17) + 37 if op == "build" else (1 << 22) + 37)
    if case["keys"] == "clustered":
        case["n"] = min(case["n"], (1 << 22) - 5)   # 64 clusters of spread 2^20 hold about this many distinct keys
    if case["kind"] == "binary_search":
        case["m"] = min(case["m"], 1 << 23)
    if case["kind"] == "harmonia":
        case["n"] -= case["n"] % 32                 # whole leaf nodes
    return case


def work(case):
    op = case["op"]
    if op == "partition":
        return {"bytes": case["m"] * (2 * case["key_bytes"] + 4), "flops": 0}
    if op == "aggregate":
        return {"bytes": case["rows"] * 4 + int(case["rows"] * 30 / 2557) * 14, "flops": 0}
    if op == "train":
        return {"bytes": case["samples"] * 8, "flops": case["samples"] * case["hidden"] * 12}
    kb, n, m = case["key_bytes"], case["n"], case["m"]
    if op == "build" or case["approach"] == "hj":
        return {"bytes": n * kb + m * (kb + 4), "flops": 0}
    return {"bytes": min(n, m) * kb + m * (kb + 4), "flops": 0}


# ---- inputs ------------------------------------------------------------------------------

def sample_keys(kind, n, key_bytes, gen):
    """n values of the key distribution, duplicates among them, as int64."""
    space = KEY_SPACE if key_bytes == 8 else 1 << 32
    if kind == "uniform":
        return torch.randint(0, space - 1, (n,), dtype=torch.int64, device="cuda", generator=gen)
    z = torch.randn(n, dtype=torch.float64, device="cuda", generator=gen)
    if kind == "lognormal":  # lognormal(0, 2), six sigma at the top of the range
        return (torch.exp(2.0 * z - 12.0) * space).clamp(max=float(space) * (1 - 2.0 ** -40)).to(torch.int64)
    centres = torch.randint(1 << 24, space - (1 << 24), (64,), dtype=torch.int64, device="cuda", generator=gen)
    which = torch.randint(0, 64, (n,), device="cuda", generator=gen)
    return centres[which] + (z * (1 << 20)).to(torch.int64).clamp(-(1 << 23), 1 << 23)


def sorted_keys(case, gen):
    """The column: n distinct ascending keys as int64."""
    n = case["n"]
    if case["keys"] == "dense":
        return torch.arange(n, dtype=torch.int64, device="cuda")
    have = torch.empty(0, dtype=torch.int64, device="cuda")
    want = n + n // 8 + 256 if case["keys"] != "uniform" or case["key_bytes"] == 4 else n + 16
    while have.numel() < n:
        more = sample_keys(case["keys"], want, case["key_bytes"], gen)
        have = torch.unique_consecutive(torch.sort(torch.cat([have, more])).values)
    if have.numel() == n:
        return have
    pick = torch.arange(n, dtype=torch.int64, device="cuda") * (have.numel() - 1) // max(n - 1, 1)
    return have[pick]


def probe_keys(case, keys, gen):
    n, m = case["n"], case["m"]
    if case["probes"] == "zipf":  # theta = 1 over the key rank
        u = torch.rand(m, dtype=torch.float64, device="cuda", generator=gen)
        rank = torch.exp(u * math.log(n)).to(torch.int64).clamp(max=n - 1)
    else:
        rank = torch.randint(0, n, (m,), device="cuda", generator=gen)
    probes = keys[rank]
    del rank
    if case["miss"] > 0:
        # absent keys are uniform over the key space, but for dense keys just past the last one
        top = 2 * n if case["keys"] == "dense" else (KEY_SPACE - 1 if case["key_bytes"] == 8 else (1 << 32) - 2)
        low = n if case["keys"] == "dense" else 0
        away = torch.rand(m, device="cuda", generator=gen) < case["miss"]
        other = torch.randint(low, top, (m,), dtype=torch.int64, device="cuda", generator=gen)
        probes = torch.where(away, other, probes)
    if case["probes"] == "sorted":
        probes = torch.sort(probes).values
    return probes


def key_view(values, key_bytes):
    if key_bytes == 8:
        return View(values, np.uint64)
    return View(values.to(torch.int32), np.uint32)  # the low 32 bits


def training_state(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    h, count = case["hidden"], case["samples"]
    # a monotone ramp network near the CDF it is fitted to, as in the middle of training
    edges = torch.linspace(0, 1, h + 1, dtype=torch.float32, device="cuda")
    w1 = h * (1 + 0.1 * torch.rand(h, device="cuda", generator=gen))
    b1 = -edges[:h] * w1
    w2 = (1 + 0.1 * torch.rand(h, device="cuda", generator=gen)) / h
    params = torch.cat([w1, b1, w2, torch.full((1,), 0.01, device="cuda")]).to(torch.float32)
    x = torch.rand(count, device="cuda", generator=gen)
    y = (x * x * (3 - 2 * x)).to(torch.float32)
    return params, x, y


def prepare(case, seed):
    op = case["op"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if op == "train":
        params, x, y = training_state(case, seed)
        grad = torch.zeros(3 * case["hidden"] + 1, dtype=torch.float32, device="cuda")
        loss = torch.zeros(1, dtype=torch.float32, device="cuda")
        return dict(op=op, hidden=case["hidden"], params=View(params, np.float32), x=View(x, np.float32),
                    y=View(y, np.float32), grad=View(grad, np.float32), loss=View(loss, np.float32))
    if op == "partition":
        kb, m, bits = case["key_bytes"], case["m"], case["radix_bits"]
        keys = key_view(sample_keys("uniform", m, kb, gen), kb)
        prm = gj.PartitionParams(bits, (63 if kb == 8 else 32) - bits, case["passes"])
        cap = int(gj._lib.call("gj_partition_capacity", m, kb, bits))
        scratch = int(gj._lib.call("gj_partition_scratch_bytes", m, kb, ctypes.byref(prm)))
        state = dict(op=op, keys=keys, m=m, key_bytes=kb, params=prm, scratch_bytes=scratch,
                     out_keys=torch.zeros(cap, dtype=torch.int64 if kb == 8 else torch.int32, device="cuda"),
                     payloads=torch.zeros(cap, dtype=torch.int32, device="cuda"),
                     offsets=torch.zeros(1 << bits, dtype=torch.int64, device="cuda"),
                     counts=torch.zeros(1 << bits, dtype=torch.int64, device="cuda"),
                     scratch=torch.zeros(max(scratch, 16), dtype=torch.uint8, device="cuda"))
        state["out"] = gj.Partitioned(state["out_keys"].data_ptr(), state["payloads"].data_ptr(),
                                      state["offsets"].data_ptr(), state["counts"].data_ptr(), cap, None)
        return state
    if op == "aggregate":
        dim, rows = case["dim"], case["rows"]
        column = View(torch.arange(1, dim + 1, dtype=torch.int32, device="cuda"), np.uint32)
        flag = (torch.rand(dim, device="cuda", generator=gen) < 1 / 3).to(torch.uint8)
        fkey = torch.randint(1, dim + 1, (rows,), dtype=torch.int32, device="cuda", generator=gen)
        date = torch.randint(0, 2557, (rows,), dtype=torch.int32, device="cuda", generator=gen)
        price = torch.randint(90_000, 10_500_001, (rows,), dtype=torch.int64, device="cuda", generator=gen)
        disc = torch.randint(0, 11, (rows,), dtype=torch.int8, device="cuda", generator=gen)
        result = torch.zeros(4, dtype=torch.int64, device="cuda")
        return dict(op=op, index=gj.Index(case["kind"], column), fkey=View(fkey, np.int32), date=View(date, np.int32),
                    price=View(price, np.int64), disc=View(disc, np.int8), flag=View(flag, np.uint8),
                    result=View(result, np.int64), strategy=case["strategy"])
    keys = sorted_keys(case, gen)
    probes = key_view(probe_keys(case, keys, gen), case["key_bytes"])
    column = key_view(keys, case["key_bytes"])
    del keys
    state = dict(op=op, kind=case["kind"], column=column, probes=probes,
                 out=View(torch.zeros(case["m"], dtype=torch.int32, device="cuda"), np.uint32))
    extra = {k: case[k] for k in ("radix_bits", "passes", "window") if k in case}
    state["params"] = gj.lookup_params(case.get("approach", "plain"), **extra)
    if op == "lookup":
        state["index"] = gj.Index(case["kind"], column)
    return state


# ---- one pass ----------------------------------------------------------------------------

def run(state):
    op = state["op"]
    if op == "lookup":
        state["index"].lookup(state["probes"], state["out"], params=state["params"])
        return state["out"].tensor
    if op == "build":
        index = gj.Index(state["kind"], state["column"])
        index.lookup(state["probes"], state["out"], params=state["params"])
        index.close()
        return state["out"].tensor
    if op == "partition":
        gj._lib.check(gj._lib.call("gj_partition", state["keys"].ptr, state["m"], state["key_bytes"],
                                   ctypes.byref(state["params"]), ctypes.byref(state["out"]),
                                   ctypes.c_void_p(state["scratch"].data_ptr()), state["scratch_bytes"], None))
        return {k: state[k] for k in ("out_keys", "payloads", "offsets", "counts")}
    if op == "aggregate":
        state["result"].tensor.zero_()  # the call adds to it
        gj.join_aggregate(state["index"], state["fkey"], state["date"], state["price"], state["disc"], state["flag"],
                          1200, 1230, state["result"], strategy=state["strategy"])
        return state["result"].tensor
    gj.mlp_loss_grad(state["params"], state["hidden"], state["x"], state["y"], state["grad"], state["loss"])
    return {"grad": state["grad"].tensor, "loss": state["loss"].tensor}


def exact(case, seed):
    """Row ids, partitions and sums are whole numbers; only a training step computes others."""
    if case["op"] != "train":
        return None
    params, x, y = (t.double() for t in training_state(case, seed))
    h = case["hidden"]
    w1, b1, w2, b2 = params[:h], params[h:2 * h], params[2 * h:3 * h], params[3 * h]
    grad, loss = torch.zeros_like(params), torch.zeros(1, dtype=torch.float64, device="cuda")
    for i in range(0, x.numel(), 1 << 18):
        xs, ys = x[i:i + (1 << 18), None], y[i:i + (1 << 18)]
        a = xs * w1 + b1
        ramp = a.clamp(0.0, 1.0)
        r = ramp @ w2 + b2 - ys
        g = 2.0 * r / x.numel()
        slope = ((a > 0) & (a < 1)).double() * (g[:, None] * w2)
        grad += torch.cat([(slope * xs).sum(0), slope.sum(0), (g[:, None] * ramp).sum(0), g.sum()[None]])
        loss += (r * r).sum() / x.numel()
    return {"grad": grad, "loss": loss}
