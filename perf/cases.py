"""What the engine is timed on: one case per way a program uses it, through its public entry points.

A case names a program or an operator sequence and its sizes.  ``prepare`` makes the input
relation a program has in hand (rows in device memory for the whole programs and operators, host
arrays for the batched and served forms, whose entry points take host rows), ``run`` is one call or one
sequence of calls.  Inputs differ from seed to seed; sizes are those of the repository's benchmark,
tests and generators, and the ranges around them.

Whole relations come back as host rows (``rows``: true), as the executables write them.  Where the
relation is far larger than a program would bring to the host (800 MB to 166 GB), the call is the one
that the benchmark and the single join's executable make: the relation is formed in device memory, and its counts and
the digest over every row come back.  So it is for the components, whose number depends on the ids
(the rounds stop by the reference's rule).

A case that returns whole relations keeps one graph and renames its ids by the seed: other inputs and
other outputs, of the same size.  The others make another graph for another seed.

Every output is a whole number (tuples, counts, digests), so there is no rounding to compare
against a wider type and ``exact`` has no value to give.
"""
import ctypes
import math
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

import mnmgdatalog_amd as dlg
from mnmgdatalog_amd import workloads

_keep = {}


def _ctx():
    """The context (stream, device memory pool) that a program opens once and keeps."""
    if "ctx" not in _keep:
        _keep["ctx"] = dlg.Ctx(0)
    return _keep["ctx"]


def _server():
    """The request loop that a serving program starts once and keeps."""
    if "server" not in _keep:
        _keep["server"] = dlg.Server(0, workers=16, max_batch=16)
    return _keep["server"]


def listed():
    return [
        # a few hundred edges, many calls: what a rule engine's small strata look like; launches and latency
        {"name": "tc_small", "kind": "tc_er", "edges": 700, "degree": 1.6, "rows": True},
        # a skewed graph of ordinary size, few rounds, dense closure (the benchmark's power-law TC)
        {"name": "tc_powerlaw", "kind": "tc_powerlaw", "vertices": 3000, "edges": 7000, "rows": True},
        # more ids than the bitmap layout takes: sort, hash set, join and merge on tuples
        {"name": "tc_wide_ids", "kind": "tc_wide", "vertices": 400_000, "degree": 0.9, "stride": 1, "rows": True},
        # road-network-shaped, ~500 rounds, the benchmark's default workload: 2e10 tuples, 166 GB on the device
        {"name": "tc_grid_400", "kind": "tc_grid", "side": 400, "rows": False},
        # finite-element mesh, three-way join (the benchmark's SG workload): 2e9 tuples
        {"name": "sg_mesh_35", "kind": "sg_mesh", "cells": 35, "rows": False},
        # components of a high-diameter graph, ~500 short rounds
        {"name": "wcc_grid_400", "kind": "wcc_grid", "side": 400, "rows": False},
        # components of a social-network-shaped graph at the served form's resident size: 2.6e8 rows
        {"name": "wcc_rmat_23", "kind": "wcc_rmat", "scale": 23, "factor": 16, "rows": False},
        # one self-join of random rows, 1e8 tuples (the reference's published size)
        {"name": "single_join_10m", "kind": "single_join", "edges": 10_000_000, "range": 1_000_000, "rows": False},
        # many independent closures in one call (the benchmark's batched workload)
        {"name": "batch_tc_512", "kind": "batch", "program": "tc", "count": 512, "max_edges": 23_911, "rows": False},
        # a burst of small requests through the request loop, each answered with its rows
        {"name": "served_32", "kind": "served", "requests": 32, "median": 2000},
        # one semi-naive round put together from the operators, as a program with its own rules does: small deltas
        {"name": "round_small", "kind": "round", "edges": 7001, "ids": 3000, "delta": 2053, "full": 60_013},
        # the same with relations that fill the device
        {"name": "round_large", "kind": "round", "edges": 4_000_037, "ids": 1_000_000, "delta": 4_100_011, "full": 33_000_001},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["tc_er", "tc_powerlaw", "tc_wide", "tc_grid", "sg_mesh", "wcc_grid", "wcc_rmat", "single_join", "batch",
                       "served", "round"])
    if kind == "tc_er":
        m = _log(rng, 60, 15_000)
        return {"kind": kind, "edges": m, "degree": round(rng.uniform(0.8, 4.0), 2), "rows": m <= 6000}
    if kind == "tc_powerlaw":
        n = _log(rng, 300, 6000)
        return {"kind": kind, "vertices": n, "edges": int(n * rng.uniform(1.5, 3.0)), "rows": n <= 4000}
    if kind == "tc_wide":
        return {"kind": kind, "vertices": _log(rng, 270_000, 1_000_000), "degree": round(rng.uniform(0.4, 0.93), 2),
                "stride": rng.choice([1, 3, 1000]), "rows": True}
    if kind == "tc_grid":
        side = _log(rng, 16, 300)
        return {"kind": kind, "side": side, "rows": side <= 70}
    if kind == "sg_mesh":
        cells = rng.randint(3, 33)
        return {"kind": kind, "cells": cells, "rows": cells <= 13}
    if kind == "wcc_grid":
        return {"kind": kind, "side": _log(rng, 20, 500), "rows": False}
    if kind == "wcc_rmat":
        return {"kind": kind, "scale": rng.randint(8, 22), "factor": rng.randint(4, 16), "rows": False}
    if kind == "single_join":
        m = _log(rng, 5000, 10_000_000)
        r = max(50, int(m / rng.uniform(6.0, 100.0)))
        return {"kind": kind, "edges": m, "range": r, "rows": m <= 200_000}
    if kind == "batch":
        return {"kind": kind, "program": rng.choice(["tc", "tc", "wcc"]), "count": _log(rng, 8, 400),
                "max_edges": _log(rng, 1500, 20_000), "rows": False}
    if kind == "served":
        return {"kind": kind, "requests": rng.randint(8, 48), "median": _log(rng, 300, 3000)}
    m = _log(rng, 1000, 6_000_000)
    ids = max(100, int(m / rng.uniform(1.0, 6.0)))
    d = int(m * rng.uniform(0.2, 1.3))
    return {"kind": "round", "edges": m, "ids": ids, "delta": d, "full": d + int(m * rng.uniform(0.5, 8.0))}


def _rng(seed, salt):
    return np.random.default_rng([int(seed) & 0x7FFFFFFF, salt])


def _gen_seed(seed):
    return workloads.SEED + 7919 * int(seed)


def _rmat(scale, factor, seed):
    """An undirected R-MAT graph (.57, .19, .19, .05), both directions of every edge, sorted by
    (source, end) as the generator and a sorted edge file have it, made on the device."""
    g = torch.Generator(device="cuda").manual_seed(_gen_seed(seed))
    m = factor << scale
    src = torch.zeros(m, dtype=torch.int64, device="cuda")
    dst = torch.zeros(m, dtype=torch.int64, device="cuda")
    for _ in range(scale):
        u = torch.rand(m, device="cuda", generator=g)
        s = u >= 0.76
        src.mul_(2).add_(s)
        dst.mul_(2).add_(((u >= 0.57) & ~s) | (u >= 0.95))
        del u, s
    lo, hi = torch.minimum(src, dst), torch.maximum(src, dst)
    del src, dst
    key = ((lo << scale) | hi)[lo != hi]
    del lo, hi
    key = torch.unique(key)
    a, b = key >> scale, key & ((1 << scale) - 1)
    both = torch.sort(torch.cat([key, (b << scale) | a])).values
    del key, a, b
    return torch.stack([both >> scale, both & ((1 << scale) - 1)], dim=1).to(torch.int32).contiguous()


def _device(rows):
    return torch.from_numpy(np.ascontiguousarray(rows, dtype=np.int32)).cuda()


def _in_order(rows):
    """The rows sorted by (source, end), as the generators and a sorted edge file have them."""
    return rows[np.lexsort((rows[:, 1], rows[:, 0]))]


def _renamed(rows, seed):
    """The relation with its ids permuted among themselves."""
    n = int(rows.max()) + 1
    return _in_order(_rng(seed, 4).permutation(n).astype(np.int32)[rows])


def _turned(rows, side, dims, seed):
    """A grid or mesh of side**dims points seen from another corner, its axes in another order, its
    ids from another origin."""
    r = _rng(seed, 5)
    at = [rows // side**k % side for k in range(dims)]
    at = [side - 1 - x if r.integers(2) else x for x in at]
    order = r.permutation(dims)
    return _in_order(sum(at[int(order[k])] * side**k for k in range(dims)) + int(r.integers(1_000_000)))


def _relation(case, seed):
    """The input rows of a whole program, in device memory."""
    kind = case["kind"]
    s = workloads.SEED if case["rows"] else _gen_seed(seed)
    if kind in ("tc_er", "tc_powerlaw", "tc_wide"):
        if kind == "tc_er":
            n = max(8, int(round(case["edges"] / case["degree"])))
            rows = dlg.gen_erdos_renyi(n, min(case["edges"], n * (n - 1) // 2), s)
        elif kind == "tc_powerlaw":
            rows = dlg.gen_powerlaw(case["vertices"], case["edges"], 2.1, s)
        else:
            rows = dlg.gen_erdos_renyi(case["vertices"], int(case["vertices"] * case["degree"]), s)
        return _device(_renamed(rows, seed) * np.int32(case.get("stride", 1)))
    if kind in ("tc_grid", "wcc_grid"):
        return _device(_turned(dlg.gen_grid(case["side"], 0.55, 0.01, 20, s), case["side"], 2, seed))
    if kind == "sg_mesh":   # the mesh with 1 % of its edges missing
        rows = dlg.gen_tetmesh(case["cells"])
        rows = rows[_rng(s, 1).random(len(rows)) >= 0.01]
        return _device(_turned(rows, case["cells"] + 1, 3, seed))
    if kind == "wcc_rmat":
        return _rmat(case["scale"], case["factor"], seed)
    g = torch.Generator(device="cuda").manual_seed(s)
    rows = torch.randint(0, case["range"], (case["edges"], 2), dtype=torch.int32, device="cuda", generator=g)
    name = torch.from_numpy(_rng(seed, 4).permutation(case["range"]).astype(np.int32)).cuda() + 1
    return name[rows.long()].contiguous()


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        rng = _rng(seed, 2)
        u, d = rng.random(case["count"]), rng.uniform(2.0, 4.0, case["count"])
        m = workloads.c4_edges(u, case["max_edges"])
        with ThreadPoolExecutor(8) as ex:
            inst = list(ex.map(lambda i: workloads.er_or_rmat(i, int(m[i]), float(d[i]), _gen_seed(seed) + i), range(case["count"])))
        return {"case": case, "ctx": _ctx(), "instances": inst}
    if kind == "served":
        reqs = workloads.served_requests(case["requests"], case["median"], 1.0, 8000, workloads.SEED)
        reqs = [(p, _renamed(r, seed + i) if p == "tc" else r + np.int32(_rng(seed, 6 + i).integers(1_000_000)))
                for i, (p, r) in enumerate(reqs)]   # a components request keeps its ids' order, which its answer's size hangs on
        return {"case": case, "server": _server(), "requests": reqs}
    if kind == "round":
        g = torch.Generator(device="cuda").manual_seed(workloads.SEED)
        ids = case["ids"]

        def pairs(n):
            return torch.randint(0, ids, (n, 2), dtype=torch.int64, device="cuda", generator=g)

        edges, full = pairs(case["edges"]), pairs(case["full"])
        full = torch.unique(full[:, 0] * ids + full[:, 1])
        pick = torch.randperm(full.numel(), device="cuda", generator=g)[: case["delta"]]
        # the full relation (a sorted set), of which the last round's new tuples (the delta) are a part
        name = torch.from_numpy(_rng(seed, 4).permutation(ids)).cuda()
        full = name[full // ids] * ids + name[full % ids]
        delta, full = full[pick].sort().values, full.sort().values

        def tuples(key):
            return (((key // ids) ^ 0x80000000) << 32) | ((key % ids) ^ 0x80000000)

        return {"case": case, "ctx": _ctx(), "edges": name[edges].to(torch.int32).contiguous(), "full": tuples(full),
                "delta": tuples(delta), "rel": torch.empty(case["edges"], dtype=torch.int64, device="cuda")}
    return {"case": case, "ctx": _ctx(), "rows": _relation(case, seed)}


def _answer(r, rows):
    out = {k: int(r[k]) for k in ("iterations", "output_size", "secondary", "nodes")}
    if "raw_join_rows" in r:
        out["raw_join_rows"] = int(r["raw_join_rows"])
    if rows:
        out["rows"] = r["rows"]
    else:
        out["digest"] = np.array([r["output_sum"]], dtype=np.uint64).view(np.int64)
        out["order_breaks"] = int(r["output_order_breaks"])
    return out


def _room(state, name, n):
    """A buffer that the program keeps for its next rounds, grown when a round needs more."""
    t = state.get(name)
    if t is None or t.numel() < n:
        t = torch.empty(max(n, 1), dtype=torch.int64, device="cuda")
        torch.cuda.current_stream().synchronize()   # the block may come from work on torch's stream
        state[name] = t
    return t


def _round(s):
    """N = unique(delta join E) minus F, F' = F + N, with the operators alone."""
    c, lib = s["ctx"], s["ctx"].L
    h, out, n = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_int64()
    rel, full, delta = s["rel"], s["full"], s["delta"]
    c.check(lib.dlg_pack_rows(c.h, s["edges"].data_ptr(), rel.numel(), dlg.ORIENT_KV, rel.data_ptr()), "pack_rows")
    c.check(lib.dlg_hash_build(c.h, rel.data_ptr(), rel.numel(), 0.0, ctypes.byref(h)), "hash_build")
    c.check(lib.dlg_join(c.h, h, delta.data_ptr(), delta.numel(), dlg.PROJ_HV_PV, ctypes.byref(out), ctypes.byref(n)), "join")
    raw = n.value
    c.check(lib.dlg_sort_unique(c.h, out, raw, ctypes.byref(n)), "sort_unique")
    uniq = n.value
    new = _room(s, "new", uniq)
    c.check(lib.dlg_set_difference(c.h, out, uniq, full.data_ptr(), full.numel(), new.data_ptr(), ctypes.byref(n)), "set_difference")
    grown = _room(s, "grown", full.numel() + n.value)
    c.check(lib.dlg_merge(c.h, full.data_ptr(), full.numel(), new.data_ptr(), n.value, grown.data_ptr()), "merge")
    c.check(lib.dlg_dev_free(c.h, out), "dev_free")
    lib.dlg_hash_free(c.h, h)
    return {"raw": raw, "new": new[: n.value], "full": grown[: full.numel() + n.value]}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "round":
        return _round(state)
    if kind == "served":
        srv = state["server"]
        tickets = [srv.submit(p, r) for p, r in state["requests"]]
        got = [srv.wait(t) for t in tickets]
        return {"rows": [g["rows"] for g in got],
                "counts": np.array([[g["status"], g["iterations"], g["output_size"], g["secondary"], g["nodes"]] for g in got])}
    if kind == "batch":
        res, _ = state["ctx"].batch_run(case["program"], state["instances"], keep_output=False, check_output=1)
        return {"counts": np.array([[r["iterations"], r["output_size"], r["secondary"], r["nodes"], r["output_order_breaks"]] for r in res]),
                "digests": np.array([r["output_sum"] for r in res], dtype=np.uint64).view(np.int64)}
    prog = kind if kind == "single_join" else kind.split("_")[0]
    rows = state["rows"]
    r = state["ctx"].run(prog, None, keep_output=case["rows"], check_output=0 if case["rows"] else 1,
                         device_rows=rows.data_ptr(), n=rows.shape[0])
    return _answer(r, case["rows"])


def _closure(n, degree):
    """Tuples of the closure of a random directed graph, about."""
    if degree < 0.95:
        return n * degree / (1.0 - degree)
    s = 0.5
    for _ in range(60):
        s = 1.0 - math.exp(-degree * s)
    return max(s * s * n * n, 8.0 * n)


def work(case):
    """The input rows read once and the output tuples written once, 8 bytes each."""
    kind = case["kind"]
    if kind == "tc_er":
        rows, out = case["edges"], _closure(case["edges"] / case["degree"], case["degree"])
    elif kind == "tc_powerlaw":
        rows, out = case["edges"], 0.7 * case["vertices"] ** 2
    elif kind == "tc_wide":
        rows, out = case["vertices"] * case["degree"], _closure(case["vertices"], case["degree"])
    elif kind == "tc_grid":
        rows, out = 2.22 * case["side"] ** 2, 0.81 * case["side"] ** 4
    elif kind == "sg_mesh":
        v = (case["cells"] + 1) ** 3
        rows, out = 6.0 * case["cells"] ** 3, 0.95 * v * v
    elif kind == "wcc_grid":
        rows, out = 2.22 * case["side"] ** 2, 0.1 * case["side"] ** 2
    elif kind == "wcc_rmat":
        rows, out = 2.0 * (case["factor"] << case["scale"]), 1000.0
    elif kind == "single_join":
        raw, cells = case["edges"] ** 2 / case["range"], float(case["range"]) ** 2
        rows, out = case["edges"], cells * -math.expm1(-raw / cells)
    elif kind == "batch":
        lo, hi = math.log(workloads.C4_MIN_EDGES), math.log(max(case["max_edges"], workloads.C4_MIN_EDGES + 1))
        mean = (math.exp(hi) - math.exp(lo)) / (hi - lo)
        square = (math.exp(2 * hi) - math.exp(2 * lo)) / (2 * (hi - lo))
        rows = case["count"] * mean
        out = case["count"] * (square * 0.55 / 9.0 if case["program"] == "tc" else 10.0)
    elif kind == "served":
        mean = case["median"] * math.exp(0.5)
        rows, out = case["requests"] * mean, 0.5 * case["requests"] * 0.55 / 9.0 * (case["median"] * math.exp(1.0)) ** 2
    else:
        raw = case["delta"] * case["edges"] / case["ids"]
        return {"bytes": 8.0 * (case["edges"] + case["delta"] + 2 * case["full"] + 2 * raw), "flops": 0.0}
    return {"bytes": 8.0 * (rows + out), "flops": 0.0}


def exact(case, seed):
    return None   # every output is a whole number
