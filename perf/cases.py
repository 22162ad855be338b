"""The calls whose time counts: the device path of this library as a program with resident data uses it.

A case is a dict of plain values; its "op" names the entry point:

* fw        closure of one dense distance matrix (Context.fw), in place on a
            copy, as a program that keeps its input does
* minplus   one min-plus product (Context.minplus)
* batch     many independent graphs to all-pairs distances: dense matrices
            from resident CSRs, then the planned batched closure
* parts     the per-part solve of a partitioned graph, all parts or a run of
            them, in groups of 32 as fapGraph solves them
* sssp      distance rows from a set of sources (stage 1 of a plain part
            solve, a query wave of the server)
* pred      predecessor rows of one solved part (is_path_needed)
* serve     a burst of mixed requests through the server until every answer
            is in the caller's hands

Device buffers are torch tensors handed over by pointer; the work runs on the
context's own stream.
"""

import math
import weakref

import numpy as np
import torch

import fastapsp_amd as fa
from fastapsp_amd import synth

INF = fa.INF

_ctx = None


def _context():
    """One context per process, as one per host thread is the library's rule."""
    global _ctx
    if _ctx is None:
        _ctx = fa.Context(0)
    return _ctx


class State(dict):
    """What a case's program holds between calls."""


def listed():
    return [
        # a part of a small partition: latency and launches count; odd size
        # and odd row stride, so no 16-byte row accesses
        {"name": "fw_n97", "op": "fw", "n": 97, "ld": 97, "p": 0.1, "whi": 100},
        # the part matrix of a 512 x 512 grid cut in 256
        {"name": "fw_n1024", "op": "fw", "n": 1024, "ld": 1024, "p": 0.05, "whi": 100},
        # a mid-size dense graph, ragged against every tile
        {"name": "fw_n2999", "op": "fw", "n": 2999, "ld": 3000, "p": 0.01, "whi": 255},
        # the dense headline size
        {"name": "fw_n8192", "op": "fw", "n": 8192, "ld": 8192, "p": 0.01, "whi": 1000},
        # stage 3 of one 512 x 512 grid part: inner rows x boundary by boundary x V
        {"name": "minplus_part", "op": "minplus", "M": 909, "N": 262144, "K": 115, "pad": 1,
         "accumulate": False, "finite": 1.0, "whi": 60000},
        # the square headline product
        {"name": "minplus_n8192", "op": "minplus", "M": 8192, "N": 8192, "K": 8192, "pad": 0,
         "accumulate": False, "finite": 0.01, "whi": 1000},
        # many uneven graphs at once
        {"name": "batch_512", "op": "batch", "count": 512, "nlo": 64, "nhi": 2048, "degree": 6,
         "whi": 255},
        # a small graph solved whole: 64 x 64 unit grid, 8 parts
        {"name": "parts_grid64", "op": "parts", "graph": "grid", "side": 64, "K": 8, "count": 8,
         "drop": 0.05, "diag": 0.0, "whi": 1},
        # a road-like network's group of parts, the library's default group
        {"name": "parts_grid512", "op": "parts", "graph": "grid", "side": 512, "K": 256,
         "count": 32, "drop": 0.10, "diag": 0.02, "whi": 100},
        # one part's boundary rows by SSSP over the whole network
        {"name": "sssp_grid512", "op": "sssp", "graph": "grid", "side": 512, "sources": 74,
         "drop": 0.10, "diag": 0.02, "whi": 100},
        # path rows of one part of a 256 x 256 network
        {"name": "pred_grid256", "op": "pred", "graph": "grid", "side": 256, "K": 64,
         "drop": 0.10, "diag": 0.02, "whi": 100},
        # a served burst: whole-graph requests and query batches, half each
        {"name": "serve_burst", "op": "serve", "graphs": 12, "queries": 12, "nlo": 256,
         "nhi": 4096, "degree": 6, "side": 256, "drop": 0.10, "diag": 0.02, "whi": 255},
    ]


def _log(rng, lo, hi):
    """An integer of [lo, hi], uniform in its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["fw", "fw", "fw", "minplus", "minplus", "minplus", "batch", "parts", "parts",
                     "sssp", "pred", "serve"])
    if op == "fw":
        n = _log(rng, 64, 8192)
        return {"op": op, "n": n, "ld": n + rng.choice([0, -n % 4, -n % 32]),
                "p": rng.choice([0.01, 0.05, 0.5, 1.0]), "whi": rng.choice([100, 255, 1000])}
    if op == "minplus":
        while True:
            M, N, K = _log(rng, 8, 8192), _log(rng, 64, 262144), _log(rng, 16, 8192)
            if M * N * K <= 8192 ** 3 and M * K + K * N + M * N <= 300_000_000:
                break
        return {"op": op, "M": M, "N": N, "K": K, "pad": rng.choice([0, 0, 1, 3]),
                "accumulate": rng.random() < 0.5, "finite": rng.choice([0.01, 0.3, 1.0]),
                "whi": rng.choice([100, 1000, 60000, 1000000])}
    if op == "batch":
        nlo = _log(rng, 48, 512)
        return {"op": op, "count": _log(rng, 16, 512), "nlo": nlo,
                "nhi": min(2048, nlo * rng.choice([2, 8, 32])), "degree": rng.choice([6, 12]),
                "whi": 255}
    graph = rng.choice(["grid", "grid", "rgg"])
    if op == "parts":
        side = _log(rng, 32, 400)
        K = max(2, side * side // rng.randint(300, 1100))
        return {"op": op, "graph": graph, "side": side, "K": K,
                "count": K if side <= 200 else min(K, rng.randint(1, 32)),
                "drop": 0.10, "diag": 0.02, "whi": rng.choice([1, 100, 255])}
    if op == "sssp":
        return {"op": op, "graph": graph, "side": _log(rng, 48, 512), "sources": _log(rng, 1, 300),
                "drop": 0.10, "diag": 0.02, "whi": rng.choice([1, 100, 255])}
    if op == "pred":
        side = _log(rng, 64, 300)
        return {"op": op, "graph": graph, "side": side, "K": max(2, side * side // 1000),
                "drop": 0.10, "diag": 0.02, "whi": rng.choice([100, 255])}
    return {"op": op, "graphs": rng.randint(1, 12), "queries": rng.randint(1, 12), "nlo": 256,
            "nhi": rng.choice([1024, 4096]), "degree": 6, "side": _log(rng, 64, 256),
            "drop": 0.10, "diag": 0.02, "whi": 255}


# ---- inputs -----------------------------------------------------------------
def _distances(rows, cols, ld, finite, whi, gen):
    """rows x cols distances (row stride ld): finite with that probability, in 1 .. whi."""
    m = torch.randint(1, whi + 1, (rows, ld), dtype=torch.int32, device="cuda", generator=gen)
    if finite < 1.0:
        m.masked_fill_(torch.rand((rows, ld), device="cuda", generator=gen) >= finite, INF)
    return m


def _sizes(case, count):
    """The graphs' sizes, log-uniform; the case's own, whatever the seed of their contents."""
    return synth.loguniform_sizes(count, case["nlo"], case["nhi"], 4)


def _csr(case, seed):
    """The case's network: a road-like grid, or a directed random geometric graph of as many vertices."""
    V = case["side"] ** 2
    if case.get("graph", "grid") == "rgg":
        u, v, w = synth.rgg_graph(V, 6, 1, case["whi"], seed)
        return synth.to_csr(V, u, v, w, True)
    u, v, w = synth.grid_graph(case["side"], case["side"], case["drop"], case["diag"], 1,
                               case["whi"], seed)
    return synth.to_csr(V, u, v, w, False)


def _partitioned(case, seed, state):
    """The network on the device with its partition: graph and part table (offset, size, boundary)."""
    ro, col, w = _csr(case, seed)
    with fa.Graph.from_csr(ro, col, w.astype(np.float32), case["K"]) as g:
        g.preCondition()
        n, off, b, _ = g.part_info()
        st2ed, gid = g.getMapping(), g.getGraphId()
    ed2st = np.empty_like(st2ed)
    ed2st[st2ed] = np.arange(st2ed.size, dtype=np.int32)
    dg = _upload(ro, col, w, state)
    dg.set_partition(gid, st2ed, ed2st)
    state["st2ed"], state["csr"] = st2ed, (ro, col, w)
    return dg, off[1:], n[1:], b[1:]


def _upload(ro, col, w, state):
    dg = _context().upload_graph(ro, col, w)
    weakref.finalize(state, dg.close)
    return dg


def prepare(case, seed):
    ctx, s = _context(), State(case)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed) & 0x7FFFFFFFFFFFFFFF)
    host = np.random.default_rng(int(seed) & 0x7FFFFFFFFFFFFFFF)
    op = case["op"]
    if op == "fw":
        m = _distances(case["n"], case["n"], case["ld"], case["p"], case["whi"], gen)
        m[:, :case["n"]].fill_diagonal_(0)
        s["source"], s["matrix"] = m, torch.empty_like(m)
    elif op == "minplus":
        M, N, K, pad = case["M"], case["N"], case["K"], case["pad"]
        s["A"] = _distances(M, K, K + pad, case["finite"], case["whi"], gen)
        s["B"] = _distances(K, N, N, case["finite"], case["whi"], gen)
        s["C"] = _distances(M, N, N, case["finite"], case["whi"], gen)
        if case["accumulate"]:  # the base; C itself is lowered in place
            s["base"] = s["C"].clone()
    elif op == "batch":
        ns = _sizes(case, case["count"])
        s["graphs"], s["mats"], s["lds"] = [], [], []
        for i, n in enumerate(int(x) for x in ns):
            u, v, w = synth.rgg_graph(n, case["degree"], 1, case["whi"], seed * 1009 + i)
            s["graphs"].append(_upload(*synth.to_csr(n, u, v, w, True), s))
            s["lds"].append((n + 31) // 32 * 32)
        # one buffer, a matrix per graph at a 128-byte boundary
        words = [n * ld for n, ld in zip(ns, s["lds"])]
        at = np.concatenate([[0], np.cumsum(words)])
        s["buffer"] = torch.full((int(at[-1]),), INF, dtype=torch.int32, device="cuda")
        s["mats"] = [s["buffer"].data_ptr() + 4 * int(a) for a in at[:-1]]
        plan = ctx.fw_plan(s["mats"], ns, s["lds"])
        weakref.finalize(s, plan.close)
        s["plan"] = plan
    elif op in ("parts", "pred"):
        dg, off, n, b = _partitioned(case, seed, s)
        V = dg.V
        count = case["count"] if op == "parts" else 1
        s["graph"] = dg
        s["starts"], s["sizes"], s["boundary"] = off[:count], n[:count], b[:count]
        rows = int(s["sizes"].sum())
        s["rows"] = torch.empty((rows, V), dtype=torch.int32, device="cuda")
        at = np.concatenate([[0], np.cumsum(s["sizes"])])[:-1]
        s["blocks"] = [s["rows"].data_ptr() + 4 * V * int(a) for a in at]
        dg.build_index()
        if op == "pred":
            s["path"] = torch.empty_like(s["rows"])
            dg.subgraph_solve_batch(s["starts"], s["sizes"], s["boundary"], s["blocks"], V)
    elif op == "sssp":
        dg = _upload(*_csr(case, seed), s)
        s["graph"] = dg
        s["sources_at"] = torch.from_numpy(
            host.choice(dg.V, size=case["sources"], replace=False).astype(np.int32)).cuda()
        s["rows"] = torch.empty((case["sources"], dg.V), dtype=torch.int32, device="cuda")
    else:
        s["server"] = fa.Server(hbm_budget=4 << 30)
        ro, col, w = _csr(case, seed)
        s["server"].attach_graph(ro, col, w)
        V = case["side"] ** 2
        ns = _sizes(case, case["graphs"])
        s["requests"] = []
        for i, n in enumerate(int(x) for x in ns):
            u, v, w = synth.rgg_graph(n, case["degree"], 1, case["whi"], seed * 1009 + i)
            s["requests"].append(synth.to_csr(n, u, v, w, True))
        s["results"] = [torch.empty(int(n) * (int(n) + 64), dtype=torch.int32, device="cuda")
                        for n in ns]
        s["pairs"] = [(host.integers(0, V, k).astype(np.int32), host.integers(0, V, k).astype(np.int32))
                      for k in synth.loguniform_sizes(case["queries"], 1, 64, 5)]
    return s


# ---- one pass ---------------------------------------------------------------
def _copy(dst, src, words):
    ctx = _context()
    fa.check(fa.load().fap_copy_i32(ctx.handle, dst, src, words, None), "copy")


def run(s):
    ctx, op = _context(), s["op"]
    if op == "fw":
        n, ld = s["n"], s["ld"]
        _copy(s["matrix"].data_ptr(), s["source"].data_ptr(), n * ld)
        ctx.fw(s["matrix"].data_ptr(), n, ld)
        return s["matrix"][:, :n]
    if op == "minplus":
        M, N, K = s["M"], s["N"], s["K"]
        if s["accumulate"]:
            _copy(s["C"].data_ptr(), s["base"].data_ptr(), M * N)
        ctx.minplus(s["A"].data_ptr(), K + s["pad"], s["B"].data_ptr(), N, s["C"].data_ptr(), N,
                    M, N, K, s["accumulate"])
        return s["C"]
    if op == "batch":
        ctx.dense_from_graphs(s["graphs"], s["mats"], s["lds"])
        s["plan"].run()
        return s["buffer"]
    if op == "parts":
        s["graph"].subgraph_solve_groups(s["starts"], s["sizes"], s["boundary"], s["blocks"],
                                         s["graph"].V, 32)
        return s["rows"]
    if op == "sssp":
        s["graph"].sssp(s["sources_at"].data_ptr(), s["sources"], s["rows"].data_ptr(),
                        s["graph"].V)
        return s["rows"]
    if op == "pred":
        V = s["graph"].V
        s["graph"].subgraph_pred(int(s["starts"][0]), int(s["sizes"][0]), s["rows"].data_ptr(), V,
                                 s["path"].data_ptr(), V)
        return s["path"]
    srv = s["server"]
    graphs = [srv.submit_graph(*r) for r in s["requests"]]
    queries = [srv.submit_queries(a, b) for a, b in s["pairs"]]
    out = []
    for rid, to in zip(graphs, s["results"]):
        srv.wait(rid)
        ptr, ld, n = srv.block(rid)
        words = (n - 1) * ld + n
        _copy(to.data_ptr(), ptr, words)
        out.append(to.as_strided((n, n), (ld, 1)))
    for rid in queries:
        srv.wait(rid)
        out.append(srv.answers(rid))
    ctx.sync()  # the copies are done: the server may reuse the blocks
    for rid in graphs + queries:
        srv.release(rid)
    return out


# ---- what a pass cannot do without -------------------------------------------
def work(case):
    """int32 values read and written once, and two operations (add, min) per
    relaxation of the dense stages, as the library counts them."""
    op = case["op"]
    if op == "fw":
        return {"bytes": 8.0 * case["n"] ** 2, "flops": 2.0 * case["n"] ** 3}
    if op == "minplus":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": 4.0 * (M * K + K * N + M * N * (2 if case["accumulate"] else 1)),
                "flops": 2.0 * M * N * K}
    if op == "batch" or op == "serve":
        count = case["count"] if op == "batch" else case["graphs"]
        lo, hi = math.log(case["nlo"]), math.log(case["nhi"])
        mean = [1.0 if hi <= lo else (math.exp(k * hi) - math.exp(k * lo)) / (k * (hi - lo))
                for k in (2, 3)]  # of n^2 and n^3, n log-uniform
        if hi <= lo:
            mean = [case["nlo"] ** 2.0, case["nlo"] ** 3.0]
        return {"bytes": 4.0 * count * mean[0], "flops": 2.0 * count * mean[1]}
    V = case["side"] ** 2
    E = 6 * V if case["graph"] == "rgg" else 4 * V * (1 - case["drop"]) + 2 * V * case["diag"]
    if op == "sssp":
        return {"bytes": 8.0 * E + 4.0 * V + 4.0 * V * case["sources"]}
    n = V / case["K"]
    if op == "pred":
        return {"bytes": 8.0 * n * V + 8.0 * E}
    b = min(n, 3.6 * math.sqrt(n))  # the boundary of a part of a planar network
    return {"bytes": case["count"] * 4.0 * n * V + 8.0 * E,
            "flops": case["count"] * (2.0 * (n - b) * b * V + 2.0 * n ** 3)}


def _closure(m):
    for k in range(m.shape[0]):
        torch.minimum(m, m[:, k:k + 1] + m[k:k + 1, :], out=m)
    return m


def exact(case, seed):
    """The distances in 64-bit integers; None where plain torch takes too long."""
    op = case["op"]
    if op == "fw" and case["n"] <= 4096:
        s = prepare(case, seed)
        return _closure(s["source"][:, :case["n"]].to(torch.int64))
    if op == "minplus" and case["M"] * case["N"] * case["K"] <= 60_000_000_000:
        s = prepare(case, seed)
        A, B = s["A"].to(torch.int64), s["B"].to(torch.int64)
        out = s["C"].to(torch.int64) if case["accumulate"] else torch.full(
            (case["M"], case["N"]), INF, dtype=torch.int64, device="cuda")
        for k in range(case["K"]):
            torch.minimum(out, A[:, k:k + 1] + B[k:k + 1, :], out=out)
        return out
    if op == "parts" and case["side"] <= 64 and case["count"] == case["K"]:
        s = prepare(case, seed)
        ro, col, w = s["csr"]
        V = ro.size - 1
        m = torch.full((V, V), INF, dtype=torch.int64, device="cuda")
        src = torch.from_numpy(np.repeat(np.arange(V), np.diff(ro))).cuda()
        m[src, torch.from_numpy(col.astype(np.int64)).cuda()] = torch.from_numpy(
            w.astype(np.int64)).cuda()
        m.fill_diagonal_(0)
        return _closure(m)[torch.from_numpy(s["st2ed"].astype(np.int64)).cuda()]
    return None
