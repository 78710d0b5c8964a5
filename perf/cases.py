"""The calls whose speed is measured, over the range that this library is used in.

A case is one call of a public entry point on a seeded synthetic graph: the
mean aggregation C = mean over the nonzeros of a row of val * H[col] through a
context (default schedule, or the schedule that tuning keeps for the graph
family), through the allocation-free entry and through the host-array entry,
and the two preprocessing calls on the GPU, the degree reordering and the
cost-weighted partition.  Graph families, sizes and widths are those of
cwlb_amd.workloads, bench.py and the tests; the drawn ones spread over the
same ranges, odd widths among them.

Graphs are made with torch on the GPU, so that making the inputs is quick;
exact() rebuilds them the same way and aggregates in float64.
"""
import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "cwlb-spmm_amd"))

from cwlb_amd import capi  # noqa: E402

COSTS = capi.read_costs(os.path.join(ROOT, "cwlb-spmm_amd", "resources", "spmm_costs_gfx950.txt"))
COMPUTE_UNITS = 256
DEV = "cuda"
FLAGS = {"none": 0, "zero": capi.ZERO_OUTPUT, "keep": capi.KEEP_EMPTY_ROWS}
# The share of the drawn edges that is left once duplicates are removed.
KEPT = {"er": 1.0, "chunglu": 0.91, "sbm": 0.999, "rmat": 0.972, "mesh": 1.0}


def _case(name, op, graph, n, deg, K, weights="unit", flags="none", schedule="default"):
    c = {"op": op, "graph": graph, "n": n, "deg": deg, "K": K, "weights": weights,
         "flags": flags, "schedule": schedule}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # The smallest call: a mini-batch sized graph, where launches and
        # host latency are most of the time.
        _case("er4096_k32", "spmm", "er", 4096, 8.0, 32),
        # A serving loop that may not allocate, on a small power-law graph
        # with weighted edges and a width that is no multiple of 4.
        _case("noalloc_chunglu20k_k50", "noalloc", "chunglu", 20_000, 10.0, 50,
              weights="uniform"),
        # An odd width (scalar rows), weighted edges, a mid-size skewed graph.
        _case("rmat18_k75", "spmm", "rmat", 1 << 18, 16.0, 75, weights="uniform"),
        # An ordinary power-law graph at the default schedule.
        _case("chunglu1m_k64", "spmm", "chunglu", 1_000_000, 10.0, 64),
        # A skewed graph at a width between powers of two; the call clears C,
        # as the reference's driver does before its kernel.
        _case("rmat21_k96_zero", "spmm", "rmat", 1 << 21, 16.0, 96, flags="zero"),
        # The headline: the large skewed graph, the schedule tuning keeps
        # there, C cleared once before repeated calls.
        _case("rmat22_k128_tuned", "spmm", "rmat", 1 << 22, 16.0, 128, flags="keep",
              schedule="hints"),
        # Very sparse, near-uniform rows, 2 GB of features: bound by latency.
        _case("mesh16m_k32", "spmm", "mesh", 16_000_000, 2.5, 32),
        # Dense communities, wide features, in the column phases tuning keeps:
        # the largest aggregation.
        _case("sbm240k_k600_phased", "spmm", "sbm", 240_000, 480.0, 600, schedule="phases"),
        # The large-K entry (K above the reference's work-group limit).
        _case("chunglu1m_k1028", "spmm", "chunglu", 1_000_000, 10.0, 1028),
        # Preprocessing on the GPU: once per graph, and once per graph and S.
        _case("reorder_rmat22", "reorder", "rmat", 1 << 22, 16.0, 0),
        _case("partition_rmat22", "partition", "rmat", 1 << 22, 16.0, 0),
        # The drop-in call on host arrays: copies in, aggregates, copies out.
        _case("host_chunglu300k_k128", "host", "chunglu", 300_000, 10.0, 128),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["spmm"] * 7 + ["noalloc", "noalloc", "host", "reorder", "partition"])
    graph = rng.choice(["er", "chunglu", "chunglu", "sbm", "rmat", "rmat", "mesh"])
    weights = rng.choice(["unit", "uniform"])
    flags = rng.choice(["none", "none", "zero", "keep"])
    schedule = "default"
    if graph == "sbm":
        n, deg = 50 * _log_int(rng, 20, 4800), rng.uniform(20.0, 480.0)
    elif graph == "rmat":
        n, deg = 1 << rng.randint(13, 22), rng.choice([8.0, 16.0, rng.uniform(4.0, 32.0)])
    elif graph == "mesh":
        n, deg = _log_int(rng, 64, 4000) ** 2, 2.5
    elif graph == "er":
        n, deg = _log_int(rng, 2000, 1_000_000), rng.uniform(2.0, 24.0)
    else:
        n, deg = _log_int(rng, 10_000, 2_000_000), rng.uniform(5.0, 20.0)
    if op in ("reorder", "partition"):
        return _case(None, op, graph, n, deg, 0, weights=weights)
    K = rng.choice([16, 32, 64, 96, 100, 128, 256, 600, rng.randint(3, 300),
                    _log_int(rng, 8, 1024), _log_int(rng, 1025, 4096)])
    # At most 8e9 multiply-adds and 2 GB of features (host arrays: 200 MB).
    room = min(8e9 / (n * deg), (5e7 if op == "host" else 5e8) / n)
    K = max(2, min(K, int(room)))
    if op == "host":
        flags = "none"
    elif op == "spmm" and rng.random() < 0.3:
        schedule = {"mesh": "ordered", "sbm": "phases"}.get(graph, "hints")
        flags = rng.choice([flags, "keep"])
    return _case(None, op, graph, n, deg, K, weights=weights, flags=flags, schedule=schedule)


# ------------------------------------------------------------------- inputs
def _edges(case, gen):
    """(rows, columns) of the drawn edges, int64, duplicates among them."""
    n, m = case["n"], int(case["n"] * case["deg"])

    def uniform(count, high):
        return torch.randint(0, high, (count,), generator=gen, device=DEV)

    def u01(count):
        return torch.rand(count, generator=gen, device=DEV)

    kind = case["graph"]
    if kind == "er":
        return uniform(m, n), uniform(m, n)
    if kind == "chunglu":
        # Both ends in proportion to i^(-1/1.1) (degree exponent 2.1), degrees
        # capped at 5% of the nodes.
        w = torch.arange(1, n + 1, device=DEV, dtype=torch.float64).pow_(-1.0 / 1.1)
        for _ in range(8):
            w = (w * (m / w.sum())).clamp_(max=0.05 * n)
        cdf = w.cumsum(0)
        cdf /= cdf[-1].clone()
        ends = [torch.searchsorted(cdf, torch.rand(m, generator=gen, device=DEV,
                                                   dtype=torch.float64)).clamp_(max=n - 1)
                for _ in range(2)]
        return ends[0], ends[1]
    if kind == "sbm":
        # 50 blocks, p_in : p_out = 20 : 1.
        size = n // 50
        r = uniform(m, n)
        inside = u01(m) < 20.0 / (20.0 + 49.0)
        c = torch.where(inside, r // size * size + uniform(m, size),
                        (r // size * size + size + uniform(m, n - size)) % n)
        return r, c
    if kind == "rmat":
        # a = .57, b = c = .19, d = .05, ids relabelled at random.
        r = torch.zeros(m, dtype=torch.int64, device=DEV)
        c = torch.zeros(m, dtype=torch.int64, device=DEV)
        for _ in range(n.bit_length() - 1):
            x = u01(m)
            r = r * 2 + (x >= 0.76)
            c = c * 2 + (((x >= 0.57) & (x < 0.76)) | (x >= 0.95))
        p = torch.randperm(n, generator=gen, device=DEV)
        return p[r], p[c]
    # mesh: a square lattice with 95% of deg from lattice edges, 5% shortcuts
    side = math.isqrt(n)
    keep = 0.95 * case["deg"] * n / (4.0 * n - 4.0 * side)
    ids = torch.arange(n, device=DEV)
    x, y = ids % side, ids // side
    rows, cols = [], []
    for ok, step in ((x > 0, -1), (x < side - 1, 1), (y > 0, -side), (y < side - 1, side)):
        at = ids[ok & (u01(n) < keep)]
        rows.append(at)
        cols.append(at + step)
    s = int(0.05 * m)
    rows.append(uniform(s, n))
    cols.append(uniform(s, n))
    return torch.cat(rows), torch.cat(cols)


def _csr(case, seed):
    """(row_ptr, col_idx, val, gen): the CSR, columns sorted and unique in
    each row, and the generator to draw the features from."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    n = case["n"]
    r, c = _edges(case, gen)
    key = torch.unique(r * n + c)
    del r, c
    row = torch.div(key, n, rounding_mode="floor")
    ci = (key - row * n).to(torch.int32)
    rp = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    rp[1:] = torch.bincount(row, minlength=n).cumsum(0)
    del key, row
    if case["weights"] == "unit":
        val = torch.ones(ci.numel(), device=DEV)
    else:
        val = 1.0 - torch.rand(ci.numel(), generator=gen, device=DEV)
    return rp.to(torch.int32), ci, val, gen


def _features(case, gen):
    return torch.rand((case["n"], case["K"]), generator=gen, device=DEV).mul_(2.0).sub_(1.0)


def _segment_size(nnz, n):
    """The middle one of the three wave-based candidates."""
    return capi.wave_based_s(nnz, n + 1, COMPUTE_UNITS, capi.recommended_candidate_w(nnz)[1])


def prepare(case, seed):
    rp, ci, val, gen = _csr(case, seed)
    n, nnz = case["n"], ci.numel()
    ctx = capi.Context(0, torch.cuda.current_stream().cuda_stream)
    origin = torch.empty(n, dtype=torch.int32, device=DEV)
    s = {"op": case["op"], "ctx": ctx, "n": n, "nnz": nnz, "K": case["K"],
         "flags": FLAGS[case["flags"]]}
    out = (origin, torch.empty_like(rp), torch.empty_like(ci), torch.empty_like(val))
    if case["op"] == "reorder":
        # Buffers for as many entries as the graph was drawn with.
        room = int(n * case["deg"])
        out = (origin, out[1], torch.zeros(room, dtype=torch.int32, device=DEV),
               torch.zeros(room, device=DEV))
        s.update(csr=(rp, ci, val), out=out)
        return s
    ctx.reorder_device(n, nnz, rp, ci, val, *out)
    _, rp, ci, val = out
    cap = capi.capacity_from_s(_segment_size(nnz, n), COSTS)
    if case["op"] == "partition":
        # A buffer for twice the tasks that the load alone would fill.
        tasks = torch.zeros((2 * _tasks(case) + 4096, 4), dtype=torch.int32, device=DEV)
        s.update(rp=rp, cap=cap, tasks=tasks)
        return s
    count = ctx.partition_device_count(rp, n, COSTS, cap)
    tasks = torch.zeros((count, 4), dtype=torch.int32, device=DEV)
    ctx.partition_device(rp, n, COSTS, cap, tasks, count)
    H = _features(case, gen)
    if case["op"] == "host":
        s["arrays"] = tuple(x.cpu().numpy() for x in (rp, ci, val, origin, H, tasks))
        return s
    C = torch.zeros((n, case["K"]), device=DEV)
    # What tuning keeps for the graph family at full size (bench.py).
    if case["schedule"] == "hints":
        ctx.set_schedule(64, 2)
        ctx.set_cache_hints(48 << 20)
    elif case["schedule"] == "ordered":
        ctx.set_schedule(4, 1)
        ctx.set_locality(2, 2)
        ctx.set_occupancy(6)
    elif case["schedule"] == "phases":
        ctx.set_schedule(16, 4)
        ctx.set_locality(2, 2)
        ctx.set_column_phases(16)
        ctx.set_lane_tiling(2)
    s.update(C=C, call=(rp, ci, val, origin, n, nnz, H, n, case["K"], tasks, count, C),
             large_k=case["K"] > 1024, stream=torch.cuda.current_stream().cuda_stream)
    return s


def run(s):
    op = s["op"]
    if op == "reorder":
        s["ctx"].reorder_device(s["n"], s["nnz"], *s["csr"], *s["out"])
        return s["out"]
    if op == "partition":
        count = s["ctx"].partition_device(s["rp"], s["n"], COSTS, s["cap"], s["tasks"],
                                          len(s["tasks"]))
        return s["tasks"], count
    if op == "host":
        return s["ctx"].spmm_host(*s["arrays"])[0]
    if op == "noalloc":
        capi.spmm_noalloc(s["stream"], *s["call"], flags=s["flags"], synchronize=False)
    else:
        s["ctx"].spmm(*s["call"], flags=s["flags"], timed=False, large_k=s["large_k"])
    return s["C"]


# ------------------------------------------------------------- what it takes
def _nnz(case):
    return int(case["n"] * case["deg"] * KEPT[case["graph"]])


def _tasks(case):
    """About as many tasks as the partition makes: the rows' cost over the
    capacity of one task."""
    nnz = _nnz(case)
    cap = capi.capacity_from_s(_segment_size(nnz, case["n"]), COSTS)
    return int((nnz * (COSTS[0] + COSTS[1]) + case["n"] * COSTS[2]) / cap) + 1


def work(case):
    n, K, nnz, tasks = case["n"], case["K"], _nnz(case), _tasks(case)
    if case["op"] == "reorder":
        return {"bytes": 16 * nnz + 12 * n, "flops": 0}
    if case["op"] == "partition":
        return {"bytes": 4 * n + 16 * tasks, "flops": 2 * n}
    return {"bytes": 8 * nnz + 8 * n + 16 * tasks + 8 * n * K, "flops": 2 * nnz * K}


def tolerance(case):
    if case["op"] in ("reorder", "partition"):
        return "exact"
    # 32-bit sums of up to 10^5 terms in another order: 2e-8 to 3.4e-7 from
    # float64 as measured (most where long rows are summed in sequence).
    return {"rel": 1.5e-6}


def exact(case, seed):
    """Plain torch on the same inputs: the stable (degree, id) order, or the
    weighted mean of every row in float64."""
    if case["op"] == "partition":
        return None
    rp, ci, val, gen = _csr(case, seed)
    n, K = case["n"], case["K"]
    deg = (rp[1:] - rp[:-1]).to(torch.int64)
    if case["op"] == "reorder":
        order = torch.argsort(deg, stable=True)
        length = deg[order]
        rp_out = torch.zeros_like(rp)
        rp_out[1:] = length.cumsum(0)
        first = rp[:-1].to(torch.int64)[order] - rp_out[:-1]
        at = torch.repeat_interleave(first, length) + torch.arange(ci.numel(), device=DEV)
        pad = int(n * case["deg"]) - ci.numel()
        return (order.to(torch.int32), rp_out, torch.nn.functional.pad(ci[at], (0, pad)),
                torch.nn.functional.pad(val[at], (0, pad)))
    H = _features(case, gen).double()
    C = torch.zeros((n, K), dtype=torch.float64, device=DEV)
    # Whole rows at a time, about 2 GB of gathered features in each step.
    step = max(1, (1 << 28) // K)
    starts = rp.cpu().to(torch.int64)
    a = 0
    while a < n:
        b = int(torch.searchsorted(starts, starts[a] + step, right=True)) - 1
        b = min(n, max(b, a + 1))
        p, q = int(starts[a]), int(starts[b])
        if q > p:
            rows = H[ci[p:q].long()] * val[p:q, None].double()
            C[a:b] = torch.segment_reduce(rows, "sum", lengths=deg[a:b], axis=0, unsafe=True,
                                          initial=0.0)
        a = b
    return C / deg.clamp(min=1)[:, None]
