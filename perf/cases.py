"""The work a user of this framework has it do, as cases that can be timed.

Every case goes through the package's public entry points, on inputs made
from a seed: graphs of the generators' two families (R-MAT and lattice),
graphs of small SCCs as dependency analyses meet them, batches, a server,
a fresh graph bound and summarised, a host call, and the edge-list builder.

A case is a dict of plain values:

* solve     one SCC solve of a graph that is bound already (the program holds
            the context); labels go into a caller's device tensor, or to host
            memory with to = "host"
* analyse   a graph that is new to the context: bind it (checked), solve, and
            take the SCC-size histogram and summary
* batch     every graph of a bound batch in one pass
* serve     requests for every resident graph of a server, answers in host
            memory
* host      the one-call form on host arrays (scc_detection)
* build     a device edge list into the CSR pair

Every output is a whole number, so there is no separate 64-bit value to hold
them against: they are either the same or wrong.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

import ispan_amd as I


def listed():
    return [
        # the smallest graphs a program solves in a loop: latency, host labels
        {"name": "solve_rmat_1000", "kind": "solve", "graph": "rmat", "V": 1000, "ef": 16.0, "to": "host"},
        # an ordinary graph with a size that fits nothing
        {"name": "solve_rmat_700k", "kind": "solve", "graph": "rmat", "V": 700001, "ef": 12.0, "to": "device"},
        # the benchmark's default graph: R-MAT scale 24, edge factor 16
        {"name": "solve_rmat_s24", "kind": "solve", "graph": "rmat", "V": 1 << 24, "ef": 16.0, "to": "device"},
        # a large graph of low degree and high diameter (road-like)
        {"name": "solve_grid_4096", "kind": "solve", "graph": "grid", "n": 4096, "p": 0.6, "to": "device"},
        # a sparse web-like graph: edge factor 3, most vertices outside the giant
        {"name": "solve_sparse_3m", "kind": "solve", "graph": "rmat", "V": 3000017, "ef": 3.0, "to": "device"},
        # dependency graphs of many modules, no giant: islands of a few groups
        {"name": "solve_islands", "kind": "solve", "graph": "modules", "groups": 100000, "island": 8, "wcc": 0,
         "to": "device"},
        # the same as one long chain of groups (a layered program)
        {"name": "solve_chain", "kind": "solve", "graph": "modules", "groups": 20000, "island": 20000, "wcc": 0,
         "to": "device"},
        # a graph new to the context: bind with its check, solve, summarise
        {"name": "analyse_rmat_2m", "kind": "analyse", "graph": "rmat", "V": 2000003, "ef": 16.0},
        # many graphs of 1e3 to 1e5 vertices in one pass, as the batched benchmark
        {"name": "batch_400", "kind": "batch", "n": 400, "lo": 1000, "hi": 100000},
        # a burst of requests that names every resident graph once
        {"name": "serve_32", "kind": "serve", "n": 32, "lo": 1000, "hi": 131072},
        # a program with host arrays and no context of its own
        {"name": "host_rmat_200k", "kind": "host", "graph": "rmat", "V": 200003, "ef": 8.0},
        # edge list on the device -> checked, deduplicated CSR pair
        {"name": "build_16m", "kind": "build", "V": 1 << 20, "m": 16000001},
    ]


def _log(rng: random.Random, lo: float, hi: float) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_graph(rng: random.Random, hi: int) -> dict:
    """A graph of any family with at most about hi vertices."""
    kind = rng.choice(("rmat", "rmat", "rmat", "grid"))
    if kind == "grid":
        return {"graph": "grid", "n": _log(rng, 32, math.isqrt(hi)), "p": round(rng.uniform(0.3, 0.8), 3)}
    return {"graph": "rmat", "V": _log(rng, 1000, hi), "ef": round(rng.uniform(2.5, 16.0), 2)}


def draw(rng: random.Random):
    kind = rng.choice(("solve", "solve", "solve", "modules", "modules", "analyse", "batch", "serve", "host", "build"))
    if kind == "solve":
        c = {"kind": "solve", **_draw_graph(rng, 1 << 24)}
        size = c["V"] if "V" in c else c["n"] * c["n"]
        return {**c, "to": "host" if size < 20000 and rng.random() < 0.5 else "device"}
    if kind == "modules":
        if rng.random() < 0.5:
            return {"kind": "solve", "graph": "modules", "groups": _log(rng, 1000, 100000),
                    "island": _log(rng, 2, 32), "wcc": rng.choice((0, 0, 1, 2)), "to": "device"}
        g = _log(rng, 1000, 20000)
        return {"kind": "solve", "graph": "modules", "groups": g, "island": g, "wcc": rng.choice((0, 0, 2)),
                "to": "device"}
    if kind == "analyse":
        return {"kind": "analyse", **_draw_graph(rng, 2000003)}
    if kind == "batch":
        return {"kind": "batch", "n": _log(rng, 8, 400), "lo": 1000, "hi": _log(rng, 5000, 100000)}
    if kind == "serve":
        return {"kind": "serve", "n": rng.randint(1, 32), "lo": 1000, "hi": _log(rng, 2000, 131072)}
    if kind == "host":
        return {"kind": "host", **_draw_graph(rng, 200003)}
    V = _log(rng, 1000, 1 << 20)
    return {"kind": "build", "V": V, "m": max(1, int(V * rng.uniform(2.0, 15.0)))}


class _Held:
    """What a program holds between calls; releases it when it goes."""

    def __init__(self, case: dict):
        self.case = case
        self.closers = []

    def __del__(self):
        for close in reversed(self.closers):
            try:
                close()
            except Exception:
                pass


class _Ints:
    """int32 device memory of the library, as torch.as_tensor takes it; owner
    is kept for as long as the tensor lives."""

    def __init__(self, ptr: int, n: int, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<i4", "data": (ptr, False), "strides": None,
                                         "version": 2}


def _tensor(ptr: int, n: int, owner) -> torch.Tensor:
    return torch.as_tensor(_Ints(ptr, n, owner), device="cuda") if n else torch.empty(0, dtype=torch.int32,
                                                                                      device="cuda")


def _modules(solver, groups: int, island: int, seed: int):
    """Groups of 1 to 6 vertices, each on a cycle of its own; group g has
    edges forward to groups g+1, g+2 and g+3 of its island (`island`
    consecutive groups).  Every group is an SCC, every island a weakly
    connected piece."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    # the same number of groups of each size whatever the seed
    size = (torch.arange(groups, device="cuda") % 6 + 1)[torch.randperm(groups, generator=gen, device="cuda")]
    first = torch.cumsum(size, 0) - size
    V = int(size.sum())
    v = torch.arange(V, device="cuda")
    g = torch.repeat_interleave(torch.arange(groups, device="cuda"), size)
    src, dst = [v], [first[g] + (v - first[g] + 1) % size[g]]
    i = torch.arange(groups, device="cuda")
    for t in (1, 2, 3):
        a = i[: max(groups - t, 0)]
        a = a[a // island == (a + t) // island]
        at = torch.rand(a.numel(), generator=gen, device="cuda")
        src.append(first[a] + (at * size[a]).long())
        dst.append(first[a + t])
    s, d = torch.cat(src).int().contiguous(), torch.cat(dst).int().contiguous()
    torch.cuda.synchronize()
    return solver.build_csr(V, s.numel(), s.data_ptr(), d.data_ptr())


def _graph(solver, case: dict, seed: int):
    if case["graph"] == "rmat":
        return solver.gen_rmat(case["V"], case["ef"], seed)
    if case["graph"] == "grid":
        return solver.gen_grid(case["n"], case["p"], seed)
    return _modules(solver, case["groups"], case["island"], seed)


def _many(solver, case: dict, seed: int):
    """Graphs of log-uniform size and edge factor 4 to 16.  The sizes belong
    to the case, so that every seed asks for the same amount of work."""
    rng = np.random.default_rng(case["n"] * 1000003 + case["hi"])
    sizes = np.exp(rng.uniform(np.log(case["lo"]), np.log(case["hi"]), case["n"])).astype(int)
    efs = rng.uniform(4.0, 16.0, case["n"])
    return [solver.gen_rmat(int(V), float(ef), seed * 4099 + i) for i, (V, ef) in enumerate(zip(sizes, efs))]


def _to_host(d_graph) -> I.HostGraph:
    parts = [(d_graph.fw_beg, d_graph.V + 1), (d_graph.fw_adj, d_graph.E), (d_graph.bw_beg, d_graph.V + 1),
             (d_graph.bw_adj, d_graph.E)]
    return I.HostGraph(*[_tensor(p, n, d_graph).cpu().numpy() for p, n in parts])


def prepare(case, seed):
    s = _Held(case)
    kind = case["kind"]
    if kind == "serve":
        s.server = I.Server()
        s.closers.append(s.server.close)
        with I.Solver() as solver:
            graphs = _many(solver, case, seed)
            s.ids = [s.server.add_graph(g) for g in graphs]
            for g in graphs:
                g.free()
        return s
    if kind == "host":
        with I.Solver() as solver:
            g = _graph(solver, case, seed)
            s.graph = _to_host(g)
            g.free()
        return s
    s.solver = I.Solver()
    s.closers.append(s.solver.close)
    if kind == "batch":
        graphs = _many(s.solver, case, seed)
        b = I.DeviceBatch.from_device(graphs)
        for g in graphs:
            g.free()
        s.solver.batch_bind(b)
        s.n = int(b.v_off[-1])
        b.free()
        return s
    if kind == "build":
        # endpoints with the skew of real edge lists, duplicates and
        # self-loops among them
        gen = torch.Generator(device="cuda").manual_seed(seed)
        u = torch.rand((2, case["m"]), generator=gen, device="cuda", dtype=torch.float64)
        e = (u * u * case["V"]).int().clamp_(0, case["V"] - 1)
        s.src, s.dst = e[0].contiguous(), e[1].contiguous()
        # the program's own arrays, as long as the edge list: the builder
        # says how many edges are left
        s.out = [torch.zeros(n, dtype=torch.int32, device="cuda")
                 for n in (case["V"] + 1, case["m"], case["V"] + 1, case["m"])]
        return s
    s.graph = _graph(s.solver, case, seed)
    s.closers.append(s.graph.free)
    s.params = I.default_params(wcc_mode=case.get("wcc", 0))
    s.labels = torch.empty(s.graph.V, dtype=torch.int32, device="cuda")
    if kind == "solve":
        s.solver.bind(s.graph)
    return s


def run(state):
    s, kind = state, state.case["kind"]
    if kind == "solve":
        if s.case["to"] == "host":
            s.solver.solve(s.params)
            return s.solver.labels()
        s.solver.solve(s.params, s.labels.data_ptr())
        return s.labels
    if kind == "analyse":
        s.solver.bind(s.graph)
        s.solver.solve(s.params, s.labels.data_ptr())
        bins, summary = s.solver.scc_histogram()
        return {"labels": s.labels, "bins": bins, "summary": summary}
    if kind == "batch":
        s.solver.batch_solve()
        return _tensor(I.lib().ispan_batch_labels_device(s.solver.handle), s.n, s)
    if kind == "serve":
        return [s.server.wait(rid)[0] for rid in s.server.submit_many(s.ids)]
    if kind == "host":
        return I.scc_detection(s.graph)
    g = s.solver.build_csr(s.case["V"], s.case["m"], s.src.data_ptr(), s.dst.data_ptr())
    for out, p, n in zip(s.out, (g.fw_beg, g.fw_adj, g.bw_beg, g.bw_adj), (g.V + 1, g.E, g.V + 1, g.E)):
        out[:n].copy_(_tensor(p, n, g))
    g.free()  # the runtime waits for the copies
    return {"E": g.E, "csr": s.out}


def _size(case) -> tuple[float, float]:
    """Vertices and edges, near enough."""
    if case["kind"] in ("batch", "serve"):
        mean = (case["hi"] - case["lo"]) / math.log(max(case["hi"], case["lo"] + 1) / case["lo"])
        return case["n"] * mean, case["n"] * mean * 10.0
    if case["graph"] == "rmat":
        return case["V"], case["V"] * case["ef"]
    if case["graph"] == "grid":
        n = case["n"]
        return n * n, 2.0 * n * (n - 1) * (1.0 + case["p"])
    return 3.5 * case["groups"], 6.5 * case["groups"]


def work(case):
    if case["kind"] == "build":
        # the edge list once, the CSR pair once
        return {"bytes": 8.0 * case["m"] + 8.0 * (case["V"] + 1) + 8.0 * case["m"], "flops": 0}
    V, E = _size(case)
    # a solve cannot do without both offset arrays, one adjacency entry of
    # every vertex in each direction (what puts it into an SCC or keeps it
    # out), and its label; it need not read every list to the end
    solve = 8.0 * (V + 1) + 8.0 * V + 4.0 * V
    if case["kind"] == "analyse":
        # the check of a new graph reads all of it, the summary every label
        return {"bytes": solve + 8.0 * (V + 1) + 8.0 * E + 4.0 * V, "flops": 0}
    if case["kind"] == "host":
        # the whole graph crosses to the device and is checked there
        return {"bytes": solve + 8.0 * (V + 1) + 8.0 * E, "flops": 0}
    return {"bytes": solve, "flops": 0}
