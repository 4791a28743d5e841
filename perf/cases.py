"""The joins this library is measured on, one pass each.

Every case is a call that a program makes with its relations resident on the
GPU (`where = EO_DEVICE`): it keeps a Context, its input arrays and an output
buffer with room for the rows, and each pass is the join itself, through the
C ABI.  The sizes are
those of the repository's own workloads (bench.py's C1 to C5 and the distance
join) and odd ones between them.

The fused joins return their rows in no particular order: two results are
equal when they are equal as multisets.  `Rows` holds a result as the library
left it and orders it when it is read, so that equal results read equal.
Rows of the deterministic order are read as they are.
"""
from __future__ import annotations

import ctypes
import functools
import math

import numpy as np
import torch

import eating_one_amd as eo
from eating_one_amd import _abi

INT31 = (1 << 31) - 1


def listed():
    return [
        # one lookup-sized join, where the call's latency is the cost
        dict(name="join_tiny", op="join", nR=1000, nS=4000, theta=0.0, sel=1.0, mode="pairs"),
        # C1, the shape of the CPU programs: a small dimension against a million rows
        dict(name="join_c1", op="join", nR=1 << 16, nS=1 << 20, theta=0.0, sel=1.0, mode="pairs"),
        # an ordinary query join: odd sizes, skewed foreign keys, half of them matching
        dict(name="join_mid", op="join", nR=3_000_017, nS=12_345_678, theta=0.5, sel=0.5, mode="pairs"),
        # C2, the headline: the largest join the benchmark runs
        dict(name="join_c2", op="join", nR=1 << 27, nS=1 << 28, theta=0.0, sel=1.0, mode="pairs"),
        # a left outer join with the reference's 16-byte RESULT rows, as written to its result files
        dict(name="join_outer16", op="join", nR=1_500_001, nS=5_000_003, theta=0.0, sel=0.5, mode="outer16"),
        # rows in the same order on every run (tests, checkpointed pipelines)
        dict(name="join_ordered", op="join", nR=1 << 22, nS=1 << 23, theta=0.0, sel=1.0, mode="ordered"),
        # C3 on the block nested-loop join: duplicates on both sides
        dict(name="nlj_c3", op="nlj", nR=1 << 18, nS=1 << 18, keys=1 << 16),
        # the FP64 distance join of bench.py
        dict(name="dist_2p17", op="dist", nR=1 << 17, nS=1 << 17, box=64.0),
        # C3 on the hash index: build on new data, then join
        dict(name="hash_index_c3", op="hashed", nR=1 << 18, nS=1 << 18, keys=1 << 16, resident=False),
        # a sorted index built on new data, then probed by binary search
        dict(name="sorted_index_build", op="sorted", nR=5_000_011, nS=8_000_009, learned=False, resident=False),
        # C4 at a quarter: a resident learned index of lognormal keys, 80 % of the probes present
        dict(name="learned_index_c4", op="sorted", nR=1 << 24, nS=1 << 25, learned=True, resident=True),
        # the benchmark's fixed batch: 1024 joins of 2^10 to 2^16, a quarter on resident tables
        dict(name="batch_1024", op="batch", n=1024, lo=10, hi=16, replay=False),
    ]


def _log2_size(rng, lo, hi):
    """A size spread over its logarithm, mostly no round number."""
    n = int(2.0 ** rng.uniform(lo, hi))
    return n | 1 if rng.random() < 0.5 else n


def draw(rng):
    op = rng.choice(["join"] * 6 + ["nlj", "dist", "hashed", "hashed", "sorted", "sorted", "batch"])
    if op == "join":
        mode = rng.choice(["pairs", "pairs", "pairs", "rows16", "outer", "outer16", "ordered"])
        big = 27.0 if mode == "pairs" else 24.0
        return dict(op=op, nR=_log2_size(rng, 8, big), nS=_log2_size(rng, 10, big + 1),
                    theta=rng.choice([0.0, 0.0, 0.5, 0.9]), sel=rng.choice([0.1, 0.5, 1.0]), mode=mode)
    if op == "nlj":
        nR, nS = _log2_size(rng, 8, 18), _log2_size(rng, 8, 18)
        return dict(op=op, nR=nR, nS=nS, keys=max(1 << rng.randint(12, 20), nR * nS >> 23))
    if op == "dist":
        return dict(op=op, nR=_log2_size(rng, 8, 17), nS=_log2_size(rng, 8, 17), box=rng.choice([32.0, 64.0, 100.0]))
    if op == "hashed":
        nR, nS = _log2_size(rng, 10, 22), _log2_size(rng, 10, 24)
        return dict(op=op, nR=nR, nS=nS, keys=max(nR // rng.choice([1, 2, 4]), 16), resident=rng.random() < 0.5)
    if op == "sorted":
        return dict(op=op, nR=_log2_size(rng, 10, 24), nS=_log2_size(rng, 10, 25), learned=rng.random() < 0.5,
                    resident=rng.random() < 0.5)
    lo = rng.randint(8, 11)
    return dict(op=op, n=rng.randint(16, 1024), lo=lo, hi=rng.randint(lo + 2, 18), replay=rng.random() < 0.3)


@functools.lru_cache(maxsize=None)
def _context():
    """The one context a program keeps."""
    return eo.Context(0)


# ---- inputs -----------------------------------------------------------------------


def _tuples(keys):
    """(key, payload = row) tuples of int32 keys."""
    t = torch.empty((keys.numel(), 2), dtype=torch.int32, device="cuda")
    t[:, 0] = keys
    t[:, 1] = torch.arange(keys.numel(), dtype=torch.int32, device="cuda")
    return t


def _randint(g, lo, hi, n):
    return torch.randint(lo, hi, (n,), generator=g, device="cuda", dtype=torch.int64)


def _ranks(g, n_items, theta, size):
    """Ranks in [0, n_items) of a Zipf(theta) draw (theta 0: uniform), by the
    inverse of the continuous bounded power law."""
    if theta == 0.0:
        return _randint(g, 0, n_items, size)
    u = torch.rand(size, generator=g, device="cuda", dtype=torch.float64)
    e = 1.0 - theta
    r = torch.pow(u * (float(n_items + 1) ** e - 1.0) + 1.0, 1.0 / e)
    return (r.to(torch.int64) - 1).clamp_(0, n_items - 1)


def _foreign_key(g, case):
    """R: a permutation of [0, nR); S: a share `sel` of keys of R, the rest absent from it."""
    nR, nS = case["nR"], case["nS"]
    rkeys = torch.randperm(nR, generator=g, device="cuda").to(torch.int32)
    skeys = rkeys[_ranks(g, nR, case["theta"], nS)]
    if case["sel"] < 1.0:
        miss = torch.rand(nS, generator=g, device="cuda") >= case["sel"]
        skeys = torch.where(miss, _randint(g, nR, INT31, nS).to(torch.int32), skeys)
    return _tuples(rkeys), _tuples(skeys)


def _uniform(g, case):
    """Keys uniform in [0, keys) on both sides (duplicates on both)."""
    return (_tuples(_randint(g, 0, case["keys"], case["nR"]).to(torch.int32)),
            _tuples(_randint(g, 0, case["keys"], case["nS"]).to(torch.int32)))


def _lognormal(g, case, sigma=2.0, hit=0.8):
    """C4: unique lognormal keys scaled into [0, 2^31), collisions moved to the
    next free integer, in random order; 80 % of the probes are keys of R."""
    nR, nS = case["nR"], case["nS"]
    z = torch.randn(nR, generator=g, device="cuda", dtype=torch.float64)
    d = (torch.exp(z * sigma) * (INT31 / math.exp(sigma * 4.753424))).clamp_(0, INT31 - nR).to(torch.int64)
    d = torch.sort(d).values
    row = torch.arange(nR, device="cuda")
    keys = (torch.cummax(d - row, 0).values + row).to(torch.int32)
    probes = keys[_randint(g, 0, nR, nS)]
    miss = torch.rand(nS, generator=g, device="cuda") >= hit
    probes = torch.where(miss, _randint(g, 0, INT31, nS).to(torch.int32), probes)
    return _tuples(keys[torch.randperm(nR, generator=g, device="cuda")]), _tuples(probes)


def _points(g, n, box):
    """The reference's 32-byte 3-D points {id, pad, x, y, z}."""
    p = torch.empty((n, 4), dtype=torch.float64, device="cuda")
    p[:, 1:] = torch.rand((n, 3), generator=g, device="cuda", dtype=torch.float64) * box
    head = p.view(torch.int32)
    head[:, 0] = torch.arange(n, dtype=torch.int32, device="cuda")
    head[:, 1] = 0
    return p


# ---- the calls --------------------------------------------------------------------


def _check(status, what):
    if status != _abi.EO_OK:
        raise RuntimeError(f"{what}: status {status}: {_abi.load().eo_last_error().decode()}")


def _ascending(rows):
    """Rows (int32, 2 or 4 columns) in ascending order of their 64-bit halves."""
    halves = rows.contiguous().view(torch.int64)
    for col in reversed(range(halves.shape[1])):
        halves = halves[torch.sort(halves[:, col], stable=True).indices]
    return halves.view(torch.int32)


def _padded(rows, cap):
    """The whole buffer as it is read: the rows, then -1 (what lies past them is not the join's)."""
    full = torch.full((cap, rows.shape[1]), -1, dtype=torch.int32, device="cuda")
    full[: len(rows)] = rows
    return full


class Rows(dict):
    """A join's count and its output buffer, the rows read in ascending order:
    the join's own order is unspecified (`ordered`: it is part of the result)."""

    def __init__(self, n, out, ordered=False):
        super().__init__(n=n, rows=out)
        self._ordered = ordered

    def __getitem__(self, key):
        value = super().__getitem__(key)
        if key != "rows":
            return value
        rows = value[: self["n"]]
        return _padded(rows if self._ordered else _ascending(rows), len(value))


class BatchRows(dict):
    """A batch's counts and rows, read request by request, each request's in ascending order."""

    def __init__(self, counts, offsets, out):
        super().__init__(counts=counts, rows=out)
        self._offsets = offsets

    def __getitem__(self, key):
        value = super().__getitem__(key)
        if key != "rows":
            return value
        counts, off = torch.from_numpy(self["counts"]).cuda(), torch.from_numpy(self._offsets).cuda()
        req = torch.repeat_interleave(torch.arange(len(counts), device="cuda"), counts)
        first = torch.cumsum(counts, 0) - counts
        row = torch.arange(req.numel(), device="cuda") - first[req] + off[req]
        packed = value[row].view(torch.int64).reshape(-1)
        order = torch.sort(packed, stable=True).indices
        order = order[torch.sort(req[order], stable=True).indices]
        return _padded(packed[order].reshape(-1, 1).view(torch.int32), len(value))


class _Join:
    """One join call: C entry point, arguments, output buffer for up to `cap` rows."""

    def __init__(self, entry, args, opts, cap, cols=2, ordered=False):
        self.entry, self.args, self.opts, self.ordered = entry, args, opts, ordered
        self.n = ctypes.c_uint64()
        self.out = torch.empty((cap, cols), dtype=torch.int32, device="cuda")

    def __call__(self):
        _check(self.entry(*self.args, self.out.data_ptr(), len(self.out), ctypes.byref(self.n),
                          ctypes.byref(self.opts)), "join")
        return Rows(self.n.value, self.out, self.ordered)


def _capacity(expected):
    """Rows to allow for when about `expected` come back."""
    return int(expected * 1.05 + 20 * math.sqrt(expected)) + 1024


def prepare(case, seed):
    ctx = _context()
    L, h = ctx.lib, ctx.handle
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    op = case["op"]
    if op == "batch":
        return _prepare_batch(ctx, case, seed)
    if op == "dist":
        R, S = _points(g, case["nR"], case["box"]), _points(g, case["nS"], case["box"])
    elif op in ("nlj", "hashed"):
        R, S = _uniform(g, case)
    elif op == "sorted":
        R, S = _lognormal(g, case)
    else:
        R, S = _foreign_key(g, case)
    torch.cuda.synchronize()  # the library runs on its context's own stream
    mode = case.get("mode", "pairs")
    opts = ctx.opts(where=_abi.EO_DEVICE, result16=mode.endswith("16"), left_outer=mode.startswith("outer"),
                    deterministic=mode == "ordered")
    both = (h, R.data_ptr(), len(R), S.data_ptr(), len(S))
    state = {"ctx": ctx, "R": R, "S": S, "case": case}
    if op == "join":  # a foreign key: at most one row per S tuple
        state["join"] = _Join(L.eo_hash_join, both, opts, len(S), 4 if mode.endswith("16") else 2, mode == "ordered")
    elif op == "nlj":
        state["join"] = _Join(L.eo_nlj_join, both, opts, _capacity(_rows(case)))
    elif op == "dist":
        state["join"] = _Join(L.eo_nlj_dist_join, (*both, 1.0), opts, _capacity(_rows(case)))
    else:
        index = None
        if case["resident"]:
            index = _build_index(state)
            state["index"] = eo.Index(ctx, index)  # freed with the state
        cap = len(S) if op == "sorted" else _capacity(_rows(case))
        state["join"] = _Join(L.eo_index_join, (h, index, S.data_ptr(), len(S)), opts, cap)
    return state


def _build_index(state):
    """The handle of a new index on R."""
    L, h, R, case = state["ctx"].lib, state["ctx"].handle, state["R"], state["case"]
    index, opts = ctypes.c_void_p(), state["ctx"].opts(where=_abi.EO_DEVICE)
    if case["op"] == "hashed":
        _check(L.eo_hidx_build(h, R.data_ptr(), len(R), ctypes.byref(opts), ctypes.byref(index)), "eo_hidx_build")
    else:
        _check(L.eo_sidx_build(h, R.data_ptr(), len(R), int(case["learned"]), ctypes.byref(opts),
                               ctypes.byref(index)), "eo_sidx_build")
    return index.value


def _prepare_batch(ctx, case, seed):
    """A request stream like C5's: |R| and |S| = 2^U, a quarter of the build
    sides resident tables, S keys present with a probability between 0.1 and 1.
    With replay the batch has been submitted once, as a replayed one has."""
    n, rng = case["n"], np.random.default_rng(5)
    size = lambda k: (2.0 ** rng.uniform(case["lo"], case["hi"], k)).astype(np.int64)  # noqa: E731
    table_size, nR, nS = size(16), size(n), size(n)
    use = np.where(rng.random(n) < 0.25, rng.integers(0, 16, n), -1)
    nR = np.where(use >= 0, table_size[use], nR)
    sel = rng.uniform(0.1, 1.0, n)
    pad = lambda x: (x + 1) // 2 * 2  # noqa: E731  16-byte aligned starts
    r_off = np.concatenate([[0], np.cumsum(np.where(use >= 0, 0, pad(nR)))])
    s_off = np.concatenate([[0], np.cumsum(pad(nS))])
    dR, dS = eo.DeviceArray(ctx, 8 * int(r_off[-1]) + 8), eo.DeviceArray(ctx, 8 * int(s_off[-1]))
    out = torch.empty((int(s_off[-1]), 2), dtype=torch.int32, device="cuda")
    tables = []
    for k, m in enumerate(table_size):
        d = eo.DeviceArray(ctx, 8 * int(m))
        ctx.gen_build(d, int(m), seed=seed * 4096 + k)
        tables.append(ctx.table_create(d, n=int(m)))
    reqs = (_abi.Request * n)()
    for i in range(n):
        R = None
        if use[i] < 0:
            R = dR.ptr + 8 * int(r_off[i])
            ctx.gen_build(dR, int(nR[i]), seed=seed * 4096 + 1024 + i, offset=8 * int(r_off[i]))
        ctx.gen_probe(dS, int(nS[i]), int(nR[i]), float(sel[i]), seed=seed * 4096 + 2048 + i,
                      offset=8 * int(s_off[i]))
        reqs[i] = eo.request(R=R, nR=nR[i], S=dS.ptr + 8 * int(s_off[i]), nS=nS[i], tag=i,
                             out=out.data_ptr() + 8 * int(s_off[i]), out_cap=nS[i],
                             table=tables[use[i]] if use[i] >= 0 else None)
    torch.cuda.synchronize()
    state = {"ctx": ctx, "case": case, "R": dR, "S": dS, "out": out, "tables": tables, "batch": ctx.batch(),
             "reqs": reqs, "results": (_abi.Result * n)(), "opts": ctx.opts(where=_abi.EO_DEVICE),
             "offsets": s_off[:-1].astype(np.int64)}
    if case["replay"]:
        _submit(state)
        _wait(state)
    return state


def _submit(state):
    _check(state["ctx"].lib.eo_batch_submit(state["batch"].handle, state["reqs"], len(state["reqs"]),
                                            ctypes.byref(state["opts"])), "eo_batch_submit")


def _wait(state):
    _check(state["ctx"].lib.eo_batch_wait(state["batch"].handle, state["results"], len(state["results"])),
           "eo_batch_wait")


_RESULT = np.dtype([("tag", np.uint64), ("n_out", np.uint64), ("status", np.int32), ("reserved", np.uint32)])


def run(state):
    case = state["case"]
    if case["op"] == "batch":
        if case["replay"]:
            _check(state["ctx"].lib.eo_batch_replay(state["batch"].handle), "eo_batch_replay")
        else:
            _submit(state)
        _wait(state)
        counts = np.frombuffer(state["results"], dtype=_RESULT)["n_out"].astype(np.int64)
        return BatchRows(counts, state["offsets"], state["out"])
    if case.get("resident", True):
        return state["join"]()
    index = _build_index(state)
    join = state["join"]
    join.args = (join.args[0], index, *join.args[2:])
    try:
        return join()
    finally:
        state["ctx"].lib.eo_index_free(index)


def _rows(case):
    """Expected rows of a join."""
    op, nR, nS = case["op"], case["nR"], case["nS"]
    if op == "dist":
        return nR * nS * (4.0 / 3.0 * math.pi) / case["box"] ** 3
    if op in ("nlj", "hashed"):
        return nR * nS / case["keys"]
    if op == "sorted":
        return 0.8 * nS
    return nS if case["mode"].startswith("outer") else nS * case["sel"]


def work(case):
    """Inputs read once, rows written once (expected counts); a distance join
    also evaluates every pair (3 differences, 3 squares, 2 sums)."""
    op = case["op"]
    if op == "batch":
        # the mean of 2^U, U uniform in [lo, hi]; a share of 0.55 of S matches
        size = (2.0 ** case["hi"] - 2.0 ** case["lo"]) / (math.log(2.0) * (case["hi"] - case["lo"]))
        return {"bytes": case["n"] * size * 8 * (2 + 0.55), "flops": 0}
    nR, nS = case["nR"], case["nS"]
    tuple_bytes, row_bytes = 32 if op == "dist" else 8, 16 if case.get("mode", "").endswith("16") else 8
    return {"bytes": tuple_bytes * (nR + nS) + row_bytes * _rows(case),
            "flops": 8.0 * nR * nS if op == "dist" else 0}


def exact(case, seed):
    """The outputs are row numbers and counts: there is nothing to round."""
    return None
