"""Timed cases of the bound propagation engine: the calls its users make, over
the sizes they make them at.

A case names an entry point, a family of constraint systems with its sizes,
and how the rounds are driven.

Entry points (`entry`)
  device  Problem.propagate_device: the matrix and the bounds live on the
          device, e.g. the root node or one node of a tree search.
  host    Problem.propagate: the matrix lives on the device, the bounds are
          the caller's numpy arrays (a solver that keeps its nodes on the host).
  dropin  gpu_propagate: host arrays in, host arrays out, nothing kept; the
          shape of the reference's stateless calls.
  batch   Batch.propagate_device: many independent systems in shared launches.
  nodes   Problem.propagate_nodes_device: many bound vectors of one system,
          each a propagated root with a few columns changed (children of a
          branch-and-bound node), in shared launches.
  server  Server: the same nodes as requests that name only the changed
          columns, stepped until all have completed.

Families (`family`)
  mixed     integer coefficients in [-10, 10], 60% integer columns in [0, 10],
            40% continuous ones in [-100, 100], 10% of the bounds infinite,
            row lengths uniform; many rounds.
  powerlaw  Zipf row lengths up to tens of thousands, 50% binary, 20% integer
            and 30% continuous columns, coefficients over six decades.
  cover     half covering rows, half knapsack rows over binary columns, 2% of
            them fixed to zero; few rounds.

Sync types (`sync`): loop (a host loop of launches, the default), graph
(captured chunks of launches) and persistent (one launch).
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "gpu-domain-propagator_amd"))

import gdp_amd.interface as gdp  # noqa: E402
from gdp_amd.instances import Instance  # noqa: E402

INF = 1e20
EPS = 1e-9
CONT = 3
MAX_ROUNDS = 100
CHANGES = 768  # room for changed columns per request of a server, on average
SYNC = {"loop": gdp.CPU_LOOP, "graph": gdp.GPU_LOOP, "persistent": gdp.MEGAKERNEL}


def listed():
    return [
        # a node of a small MIP solved on the host: 22,000 nonzeros, about 30
        # rounds, where launches and waits are all that counts
        dict(name="host node, 2000 rows", entry="host", family="mixed", sync="persistent", m=2000, n=1000, hi=20),
        # the same kind of system through the default round loop, odd sizes
        dict(name="device loop, 7001 rows", entry="device", family="mixed", sync="loop", m=7001, n=3001, hi=20),
        # captured launches on an ordinary instance
        dict(name="device graph, 20000 rows", entry="device", family="mixed", sync="graph", m=20000, n=10000, hi=20),
        # an ordinary instance, one launch
        dict(name="device, 200000 rows", entry="device", family="mixed", sync="persistent", m=200_000, n=100_000,
             hi=20),
        # many rounds over a matrix that does not fit the L2 caches, wider than tall
        dict(name="device chains, 100003 rows", entry="device", family="mixed", sync="persistent", m=100_003,
             n=500_009, hi=60),
        # the largest: the root node of a 1M-row system with very long rows
        dict(name="device root, 1M rows", entry="device", family="powerlaw", sync="persistent", m=1_000_000,
             n=500_000, hi=50_000, zipf=1.95),
        # a structured binary system: two rounds over long lists of short rows
        dict(name="device cover, 200000 rows", entry="device", family="cover", sync="loop", m=200_000, n=1_000_000),
        # stateless calls, small and ordinary: upload, layout, rounds, download
        dict(name="drop-in, 2000 rows", entry="dropin", family="mixed", sync="loop", m=2000, n=1000, hi=20),
        dict(name="drop-in, 200000 rows", entry="dropin", family="powerlaw", sync="loop", m=200_000, n=100_000,
             hi=5000, zipf=2.08),
        # presolving many uneven MIPs at once
        dict(name="batch, 64 systems", entry="batch", family="mixed", sync="persistent", count=64, m=1000,
             m_hi=50_000, hi=30),
        # one level of a search tree: children of the propagated root
        dict(name="nodes, 256 children", entry="nodes", family="powerlaw", sync="persistent", count=256, m=200_000,
             n=100_000, hi=5000, zipf=2.08, changed=50),
        # the same children as small requests to a server
        dict(name="server, 256 requests", entry="server", family="powerlaw", sync="persistent", count=256,
             m=200_000, n=100_000, hi=5000, zipf=2.08, changed=50),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    entry = rng.choice(["device", "device", "device", "device", "host", "dropin", "batch", "nodes", "server"])
    if entry == "batch":
        return dict(entry=entry, family="mixed", sync=rng.choice(["persistent", "graph", "loop"]),
                    count=rng.randint(8, 64), m=_log_int(rng, 500, 2000), m_hi=_log_int(rng, 5000, 50_000),
                    hi=rng.randint(4, 40))
    if entry in ("nodes", "server"):
        m = _log_int(rng, 5000, 200_000)
        return dict(entry=entry, family="powerlaw", sync="persistent", count=_log_int(rng, 8, 256), m=m,
                    n=max(1000, int(m * rng.uniform(0.3, 1.0))), hi=_log_int(rng, 500, 5000),
                    zipf=round(rng.uniform(1.95, 2.2), 3), changed=rng.randint(1, 50))
    family = rng.choice(["mixed", "mixed", "powerlaw", "cover"]) if entry != "dropin" else \
        rng.choice(["mixed", "powerlaw"])
    case = dict(entry=entry, family=family, sync=rng.choice(["loop", "graph", "persistent", "persistent"]))
    if family == "mixed":
        m = _log_int(rng, 500, 300_000)
        case.update(m=m, n=max(200, int(m * math.exp(rng.uniform(math.log(0.3), math.log(4.0))))),
                    hi=rng.randint(5, 50))
    elif family == "powerlaw":
        m = _log_int(rng, 5000, 1_000_000 if entry == "device" else 300_000)
        case.update(m=m, n=max(1000, int(m * rng.uniform(0.3, 0.9))), hi=_log_int(rng, 300, 50_000),
                    zipf=round(rng.uniform(1.95, 2.3), 3))
    else:
        m = _log_int(rng, 2000, 200_000)
        case.update(m=m, n=int(m * rng.uniform(1.0, 5.0)))
    return case


# ---------------------------------------------------------------------------
# constraint systems, drawn on the GPU from the seed
# ---------------------------------------------------------------------------

def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _gen(seed):
    g = torch.Generator(device=_dev())
    g.manual_seed(seed)
    return g


class System:
    """A constraint system as numpy arrays in CSR form, and its row ids."""

    def __init__(self, m, n, col, row_ptr, rows, val, lhs, rhs, lb, ub, vartype):
        self.m, self.n, self.col, self.row_ptr, self.rows, self.val = m, n, col, row_ptr, rows, val
        self.lhs, self.rhs, self.lb, self.ub, self.vartype = lhs, rhs, lb, ub, vartype

    def instance(self):
        return Instance(self.m, self.n, self.col, self.row_ptr, self.val, self.lhs, self.rhs, self.lb, self.ub,
                        self.vartype)


def _structure(g, m, n, lengths):
    """Rows of the given lengths with distinct random columns (duplicates drop
    out, so rows may end a little shorter)."""
    d = _dev()
    rows = torch.repeat_interleave(torch.arange(m, device=d), lengths)
    cols = torch.randint(0, n, (rows.numel(),), device=d, generator=g)
    key = torch.unique(rows * n + cols)
    rows = torch.div(key, n, rounding_mode="floor")
    ptr = torch.zeros(m + 1, dtype=torch.int64, device=d)
    ptr[1:] = torch.cumsum(torch.bincount(rows, minlength=m), 0)
    return rows, (key - rows * n).to(torch.int32), ptr.to(torch.int32)


def _uniform(g, k):
    return torch.rand(k, device=_dev(), generator=g, dtype=torch.float64)


def _point(g, lb, ub, vartype, width):
    """A point inside the bounds, integral for integer columns."""
    lo = torch.where(lb <= -INF, torch.where(ub >= INF, torch.full_like(lb, -width), ub - width), lb)
    hi = torch.where(ub >= INF, torch.where(lb <= -INF, torch.full_like(lb, width), lb + width), ub)
    x = lo + (hi - lo) * _uniform(g, lb.numel())
    r = torch.minimum(torch.maximum(torch.round(x), torch.ceil(lo)), torch.floor(hi))
    return torch.where(vartype != CONT, r, x)


def _system(family, m, n, seed, hi=20, zipf=1.95):
    g, d = _gen(seed), _dev()
    if family == "mixed":
        lengths = torch.randint(2, min(hi, n) + 1, (m,), device=d, generator=g)
    elif family == "powerlaw":
        k = np.arange(2, min(hi, n) + 1, dtype=np.float64) ** -zipf
        cdf = torch.from_numpy(np.cumsum(k) / k.sum()).to(d)
        lengths = (2 + torch.searchsorted(cdf, _uniform(g, m), right=True)).clamp(2, min(hi, n))
    else:
        mc = m // 2
        lengths = torch.cat([torch.randint(3, 41, (mc,), device=d, generator=g),
                             torch.randint(10, 201, (m - mc,), device=d, generator=g)])
    rows, col, ptr = _structure(g, m, n, lengths)
    nnz = rows.numel()
    u = _uniform(g, n)
    if family == "cover":
        val = torch.where(rows < m // 2, torch.ones(nnz, dtype=torch.float64, device=d),
                          torch.randint(1, 1001, (nnz,), device=d, generator=g).double())
        vartype = torch.zeros(n, dtype=torch.int32, device=d)
        lb = torch.zeros(n, dtype=torch.float64, device=d)
        ub = torch.where(u < 0.02, 0.0, 1.0).double()
    elif family == "mixed":
        mag = torch.randint(1, 11, (nnz,), device=d, generator=g).double()
        val = torch.where(_uniform(g, nnz) < 0.5, -mag, mag)
        ints = u < 0.6
        vartype = torch.where(ints, 1, CONT).to(torch.int32)
        lb = torch.where(ints, 0.0, -100.0).double()
        ub = torch.where(ints, 10.0, 100.0).double()
        lb[_uniform(g, n) < 0.1] = -INF
        ub[_uniform(g, n) < 0.1] = INF
    else:
        mag = torch.where(_uniform(g, nnz) < 0.3, 10.0 ** (6.0 * _uniform(g, nnz) - 3.0),
                          torch.randint(1, 21, (nnz,), device=d, generator=g).double())
        val = torch.where(_uniform(g, nnz) < 0.5, -mag, mag)
        vartype = torch.where(u < 0.5, 0, torch.where(u < 0.7, 1, CONT)).to(torch.int32)
        cont = vartype == CONT
        lb = torch.where(cont, -1e4, 0.0).double()
        ub = torch.where(cont, 1e4, torch.where(vartype == 0, 1.0, 100.0).double())
        lb[cont & (_uniform(g, n) < 0.05)] = -INF
        ub[cont & (_uniform(g, n) < 0.05)] = INF
    width = 1e4 if family == "powerlaw" else 10.0
    x0 = _point(g, lb, ub, vartype, width)
    slack = _uniform(g, 2 * m).cpu().numpy()
    side = _uniform(g, 2 * m).cpu().numpy()
    # sums in row order on the host: the same bits from the same seed
    h = {k: v.cpu().numpy() for k, v in dict(rows=rows, col=col, ptr=ptr, val=val, lb=lb, ub=ub, x0=x0,
                                             vartype=vartype).items()}
    r, c, v = h["rows"], h["col"], h["val"]
    if family == "cover":
        first = np.arange(m) < m // 2
        lhs = np.where(first, 1.0, -INF)
        rhs = np.where(first, INF, 0.3 * np.bincount(r, weights=v, minlength=m))
    else:
        act = np.bincount(r, weights=v * h["x0"][c], minlength=m)
        if family == "mixed":
            lhs, rhs = act - 5.0 * slack[:m], act + 5.0 * slack[m:]
            one, drop = side[:m] < 0.3, side[m:] < 0.5
            lhs[one & drop] = -INF
            rhs[one & ~drop] = INF
        else:
            lo = np.where(h["lb"] <= -INF, h["x0"] - width, h["lb"])
            up = np.where(h["ub"] >= INF, h["x0"] + width, h["ub"])
            rng = np.bincount(r, weights=np.abs(v) * (up - lo)[c], minlength=m)
            lhs, rhs = act - 0.1 * rng * slack[:m], act + 0.1 * rng * slack[m:]
    return System(m, n, c, h["ptr"], r, v, lhs, rhs, h["lb"], h["ub"], h["vartype"])


def _systems(case, seed):
    """The system of a case, or the list of a batch's."""
    if case["entry"] != "batch":
        return _system(case["family"], case["m"], case["n"], seed, case.get("hi", 20), case.get("zipf", 1.95))
    rng = np.random.default_rng([case["count"], case["m"], case["m_hi"], case["hi"]])  # sizes: the case's, not the seed's
    out = []
    for k in range(case["count"]):
        m = int(np.exp(rng.uniform(np.log(case["m"]), np.log(max(case["m"] + 1, case["m_hi"])))))
        hi = int(rng.integers(4, case["hi"] + 1))
        out.append(_system(case["family"], m, max(2, m // 2), seed * 1009 + k, hi))
    return out


def _children(case, seed, system, lb, ub):
    """Children of the node (lb, ub): 1..changed integer columns each, cut to a
    random half of their domain: (columns, lower, upper) per child."""
    rng = np.random.default_rng(seed + 77)
    free = np.flatnonzero((system.vartype != CONT) & (ub - lb >= 1) & (ub < INF) & (lb > -INF))
    out = []
    for _ in range(case["count"]):
        k = min(int(rng.integers(1, case["changed"] + 1)), free.size)
        j = np.sort(rng.choice(free, size=k, replace=False)).astype(np.int32)
        mid = np.floor((lb[j] + ub[j]) / 2)
        down = rng.random(k) < 0.5
        out.append((j, np.where(down, lb[j], np.minimum(mid + 1, ub[j])), np.where(down, mid, ub[j])))
    return out


# ---------------------------------------------------------------------------
# what a program holds before the call, and the call
# ---------------------------------------------------------------------------

def prepare(case, seed):
    entry = case["entry"]
    system = _systems(case, seed)
    s = {"entry": entry, "sync": SYNC[case["sync"]]}
    if entry == "dropin":
        s["instance"] = system.instance()
        return s
    if entry == "batch":
        s["batch"] = gdp.Batch([x.instance() for x in system])
        s["lb0"] = torch.from_numpy(np.concatenate([x.lb for x in system])).to(_dev())
        s["ub0"] = torch.from_numpy(np.concatenate([x.ub for x in system])).to(_dev())
        s["lb"], s["ub"] = torch.empty_like(s["lb0"]), torch.empty_like(s["ub0"])
        return s
    s["problem"] = gdp.Problem(system.instance())
    if entry == "host":
        s["lb"], s["ub"] = system.lb, system.ub
        return s
    if entry == "device":
        s["lb0"], s["ub0"] = torch.from_numpy(system.lb).to(_dev()), torch.from_numpy(system.ub).to(_dev())
        s["lb"], s["ub"] = torch.empty_like(s["lb0"]), torch.empty_like(s["ub0"])
        return s
    root = s["problem"].propagate(system.lb, system.ub, gdp.MEGAKERNEL)
    s["children"] = _children(case, seed, system, root.lbs, root.ubs)
    if entry == "server":
        s["server"] = gdp.Server(s["problem"], 8 << 30, case["count"])
        s["server"].set_base(root.lbs, root.ubs)
        size = case["count"] * CHANGES
        s["changes"] = {"cols": np.zeros(size, np.int32), "lb": np.zeros(size), "ub": np.zeros(size)}
        return s
    s["problem"].reserve(case["count"])
    lb, ub = np.tile(root.lbs, (case["count"], 1)), np.tile(root.ubs, (case["count"], 1))
    for k, (j, l, u) in enumerate(s["children"]):
        lb[k, j], ub[k, j] = l, u
    s["hints"] = [j for j, _, _ in s["children"]]
    s["lb0"], s["ub0"] = torch.from_numpy(lb).to(_dev()), torch.from_numpy(ub).to(_dev())
    s["lb"], s["ub"] = torch.empty_like(s["lb0"]), torch.empty_like(s["ub0"])
    return s


def _fresh_bounds(s):
    """The bounds to propagate, in the buffers that the call works in; the
    library works on a stream of its own, so they are there before the call."""
    s["lb"].copy_(s["lb0"])
    s["ub"].copy_(s["ub0"])
    torch.cuda.current_stream().synchronize()


def _infos(infos):
    return {"rounds": np.array([i.rounds for i in infos], np.int64),
            "infeasible": np.array([i.infeasible for i in infos], np.int64)}


def run(s):
    entry, sync = s["entry"], s["sync"]
    if entry == "dropin":
        o = gdp.gpu_propagate(s["instance"], sync)
        return {"lb": o.lbs, "ub": o.ubs, "rounds": o.rounds, "infeasible": int(o.infeasible)}
    if entry == "host":
        o = s["problem"].propagate(s["lb"], s["ub"], sync)
        return {"lb": o.lbs, "ub": o.ubs, "rounds": o.rounds, "infeasible": int(o.infeasible)}
    if entry == "server":
        server = s["server"]
        tickets = [server.submit_delta(j, l, u) for j, l, u in s["children"]]
        while server.pending() > 0:
            server.step()
        # the requests' changed columns, one after the other in the program's
        # own buffers (the library returns a request's columns in no fixed order)
        out, at, infos, counts = s["changes"], 0, [], []
        for t in tickets:
            cols, lbs, ubs, info = server.result_changes(t)
            order = np.argsort(cols)
            for key, v in (("cols", cols), ("lb", lbs), ("ub", ubs)):
                out[key][at:at + cols.size] = v[order]
            at += cols.size
            infos.append(info)
            counts.append(cols.size)
        for v in out.values():
            v[at:] = 0
        return {**out, "counts": np.array(counts, np.int64), **_infos(infos)}
    _fresh_bounds(s)
    if entry == "device":
        i = s["problem"].propagate_device(s["lb"].data_ptr(), s["ub"].data_ptr(), sync)
        return {"lb": s["lb"], "ub": s["ub"], "rounds": i.rounds, "infeasible": i.infeasible}
    if entry == "batch":
        infos = s["batch"].propagate_device(s["lb"].data_ptr(), s["ub"].data_ptr(), sync)
    else:
        row = s["lb"].shape[1] * 8
        infos = s["problem"].propagate_nodes_device([s["lb"].data_ptr() + k * row for k in range(len(s["hints"]))],
                                                    [s["ub"].data_ptr() + k * row for k in range(len(s["hints"]))],
                                                    s["hints"], sync)
    return {"lb": s["lb"], "ub": s["ub"], **_infos(infos)}


# ---------------------------------------------------------------------------
# what a pass cannot do without, and its values
# ---------------------------------------------------------------------------

def _expected_nnz(family, m, hi, zipf):
    if family == "mixed":
        return m * (2 + hi) / 2
    if family == "cover":
        return m * (21.5 + 105) / 2
    k = np.arange(2, hi + 1, dtype=np.float64)
    return m * float((k ** (1 - zipf)).sum() / (k ** -zipf).sum())


def work(case):
    """The matrix, the sides, the types and the bounds read once, the bounds
    written once; per nonzero the two products and sums of the activities, the
    width test and a candidate."""
    if case["entry"] == "batch":
        ratio = case["m_hi"] / case["m"]
        m = case["count"] * (case["m_hi"] - case["m"]) / math.log(ratio)
        n, nnz, vectors = m / 2, m * (2 + (4 + case["hi"]) / 2) / 2, 1
    else:
        m, n, vectors = case["m"], case["n"], 1
        nnz = _expected_nnz(case["family"], m, min(case.get("hi", 20), n), case.get("zipf", 1.95))
        if case["entry"] in ("nodes", "server"):
            vectors = case["count"]
    return {"bytes": 12.0 * nnz + 20.0 * m + 4.0 * n + 32.0 * n * vectors, "flops": 10.0 * nnz * vectors}


class _Exact:
    """Round-synchronous propagation in plain float64."""

    def __init__(self, systems):
        d = _dev()
        row0 = np.concatenate([[0], np.cumsum([x.m for x in systems])])
        col0 = np.concatenate([[0], np.cumsum([x.n for x in systems])])
        cat = lambda f: torch.from_numpy(np.concatenate([f(k, x) for k, x in enumerate(systems)])).to(d)  # noqa: E731
        self.m, self.n = int(row0[-1]), int(col0[-1])
        self.row = cat(lambda k, x: x.rows + row0[k])
        self.col = cat(lambda k, x: x.col.astype(np.int64) + col0[k])
        self.val, self.lhs, self.rhs = cat(lambda k, x: x.val), cat(lambda k, x: x.lhs), cat(lambda k, x: x.rhs)
        self.lengths = cat(lambda k, x: np.diff(x.row_ptr).astype(np.int64))
        vartype = cat(lambda k, x: x.vartype)
        self.cont = (vartype == CONT)[self.col]

    def _by_row(self, v, reduce):
        """Sum or maximum (at least 0) of each row's entries, at the entries."""
        return torch.segment_reduce(v, reduce, lengths=self.lengths, unsafe=True, initial=0.0)[self.row]

    def _round(self, lb, ub):
        a, l, u = self.val, lb[self.col], ub[self.col]
        pos, lo_inf, up_inf = a > 0, l <= -INF, u >= INF
        min_inf, max_inf = torch.where(pos, lo_inf, up_inf), torch.where(pos, up_inf, lo_inf)
        zero = torch.zeros_like(a)
        minact = self._by_row(torch.where(min_inf, zero, torch.where(pos, a * l, a * u)), "sum")
        maxact = self._by_row(torch.where(max_inf, zero, torch.where(pos, a * u, a * l)), "sum")
        n_min, n_max = self._by_row(min_inf.double(), "sum"), self._by_row(max_inf.double(), "sum")
        lhs, rhs = self.lhs[self.row], self.rhs[self.row]
        slack, surplus, width = rhs - minact, lhs - maxact, a.abs() * (u - l)
        # the row can move a bound at all
        widest = self._by_row(width, "max")
        gate = ~((n_min > 1) & (n_max > 1)) & ((widest - INF >= -EPS) | (widest - torch.minimum(slack, -surplus) > EPS))
        # from the right side, through the minimum activity
        right = gate & (width - slack > EPS) & (rhs < INF)
        own_r = (n_min == 1) & min_inf
        cr = slack / a
        new_r = torch.where(n_min == 0, cr + torch.where(pos, l, u), cr)
        right &= (n_min == 0) | own_r
        # from the left side, through the maximum activity
        left = gate & (width + surplus > EPS) & (lhs > -INF)
        own_l = (n_max == 1) & max_inf
        cl = surplus / a
        new_l = torch.where(n_max == 0, cl + torch.where(pos, u, l), cl)
        left &= (n_max == 0) | own_l
        nl, nu = lb.clone(), ub.clone()
        moved = False
        for ok, new in ((right, new_r), (left, new_l)):
            up = ok & (pos if new is new_r else ~pos)
            cand = torch.where(self.cont, new, torch.floor(new + EPS))
            up = up & (cand - u < -EPS)
            nu.scatter_reduce_(0, self.col[up], cand[up], "amin")
            low = ok & (~pos if new is new_r else pos)
            cand = torch.where(self.cont, new, torch.ceil(new - EPS))
            low = low & (cand - l > EPS)
            nl.scatter_reduce_(0, self.col[low], cand[low], "amax")
            moved |= bool(up.any()) or bool(low.any())
        return nl, nu, moved

    def propagate(self, lb, ub):
        lb, ub = torch.from_numpy(lb).to(_dev()), torch.from_numpy(ub).to(_dev())
        if bool((lb - ub > EPS).any()):
            return lb, ub, 0, 1
        for r in range(1, MAX_ROUNDS + 1):
            lb, ub, moved = self._round(lb, ub)
            if not moved:
                return lb, ub, r, 0
            if bool((lb - ub > EPS).any()):
                return lb, ub, r, 1
        return lb, ub, MAX_ROUNDS, 0


def exact(case, seed):
    # a server's answer lists the columns that differ from the base in any bit:
    # one column more or less moves all that follow, so it has no value here
    # (the nodes cases hold the same numbers as whole vectors)
    if case["entry"] == "server":
        return None
    system = _systems(case, seed)
    systems = system if isinstance(system, list) else [system]
    e = _Exact(systems)
    lb0, ub0 = (np.concatenate([getattr(x, k) for x in systems]) for k in ("lb", "ub"))
    lb, ub, rounds, infeasible = e.propagate(lb0, ub0)
    if case["entry"] == "batch":
        return {"lb": lb, "ub": ub, "rounds": None, "infeasible": None}
    if case["entry"] != "nodes":
        return {"lb": lb, "ub": ub, "rounds": rounds, "infeasible": infeasible}
    base_l, base_u = lb.cpu().numpy(), ub.cpu().numpy()
    lbs, ubs = [], []
    for j, l, u in _children(case, seed, system, base_l, base_u):
        cl, cu = base_l.copy(), base_u.copy()
        cl[j], cu[j] = l, u
        cl, cu, _, _ = e.propagate(cl, cu)
        lbs.append(cl)
        ubs.append(cu)
    return {"lb": torch.stack(lbs), "ub": torch.stack(ubs), "rounds": None, "infeasible": None}
