"""What the library is timed on: calls that a program makes of it, through its Python entry points.

Sizes follow the library's own configurations: exclusive scans of 2^24 and up to 2^28 elements, gathers and scatters of
2^28 elements through a full random or a block-local permutation, stable splits of 2^25 to 2^28 pairs into 2 to 4096
buckets with uniform and Zipf keys, a 32-bit radix sort of 2^28 pairs, a 2^24 x 2^24 join count and a batch of 10,000
uneven jobs; beside them the small calls and the odd lengths that a program makes of the same entry points.
"""
import importlib
import math
import random

import torch

edpp = importlib.import_module("efficient-dpp_amd")

MAX_N = 1 << 28       # elements of the largest call
BLOCK = 4096          # block length of a block-local permutation
BATCH_BUCKETS = 256   # buckets of a batch's split jobs


def listed():
    return [
        # A short prefix sum in front of a compaction or an allocation: the latency of one call.
        {"name": "scan_small", "kind": "scan", "n": 10_007, "wide": False, "small_values": False},
        # The prefix sum of small counts (2^24 values of 0..15): one chip-wide call, no steady state.
        {"name": "scan_2p24", "kind": "scan", "n": 1 << 24, "wide": False, "small_values": True},
        # Offsets that need 64 bits, an odd number of them: a long stream through HBM.
        {"name": "scan_wide_odd", "kind": "scan", "n": 100_000_007, "wide": True, "small_values": False},
        # Reordering a column by a random row order and back: the largest random access.
        {"name": "permute_random_2p28", "kind": "permute", "n": 1 << 28, "wide": False, "local": False},
        # Reordering within pages: rows shuffled in 4096-element blocks, 8-byte values.
        {"name": "permute_local_wide", "kind": "permute", "n": 16_000 * BLOCK, "wide": True, "local": True},
        # Partitioning a small batch of records by one byte: launches count.
        {"name": "split_small_b256", "kind": "split", "n": 100_000, "buckets": 256, "wide": False, "zipf": False,
         "values": True},
        # A wide-machine partition by a few bits at full size.
        {"name": "split_b16_2p28", "kind": "split", "n": 1 << 28, "buckets": 16, "wide": False, "zipf": False,
         "values": True},
        # A skewed partition of about 2^25 records with 8-byte keys.
        {"name": "split_b256_zipf_wide", "kind": "split", "n": 33_554_467, "buckets": 256, "wide": True, "zipf": True,
         "values": True},
        # Ordering a short column of signed keys.
        {"name": "sort_keys_small", "kind": "sort", "n": 131_072, "signed": True, "values": False},
        # Ordering a full column with its row numbers.
        {"name": "sort_pairs_2p28", "kind": "sort", "n": 1 << 28, "signed": False, "values": True},
        # Size of an equi-join of two equally long columns.
        {"name": "join_2p24", "kind": "join", "r_n": 1 << 24, "s_n": 1 << 24},
        # Ten thousand uneven scans, splits and gathers as one planned launch.
        {"name": "batch_10k", "kind": "batch", "jobs": 10_000, "total": 1 << 28, "plan_seed": 2026},
    ]


def _log_size(rng, lo, hi):
    n = int(math.exp(rng.uniform(math.log(lo), math.log(hi))))
    return min(hi, n | 1 if rng.random() < 0.5 else n)


def draw(rng):
    kind = rng.choice(["scan", "permute", "split", "split", "sort", "join", "batch"])
    if kind == "scan":
        wide = rng.random() < 0.5
        return {"kind": kind, "n": _log_size(rng, 1_000, MAX_N), "wide": wide, "small_values": rng.random() < 0.5}
    if kind == "permute":
        local = rng.random() < 0.5
        wide = rng.random() < 0.5
        n = _log_size(rng, 10_000, MAX_N // 2 if wide else MAX_N)
        return {"kind": kind, "n": n, "wide": wide, "local": local}
    if kind == "split":
        wide = rng.random() < 0.5
        n = _log_size(rng, 10_000, MAX_N // 2 if wide else MAX_N)
        return {"kind": kind, "n": n, "buckets": 1 << rng.randint(1, 12), "wide": wide, "zipf": rng.random() < 0.5,
                "values": rng.random() < 0.7}
    if kind == "sort":
        return {"kind": kind, "n": _log_size(rng, 1_000, MAX_N), "signed": rng.random() < 0.5,
                "values": rng.random() < 0.5}
    if kind == "join":
        # columns of comparable length, the longer one up to 8 times the shorter
        r_n = _log_size(rng, 10_000, 1 << 26)
        return {"kind": kind, "r_n": r_n, "s_n": _log_size(rng, max(10_000, r_n // 8 + 1), min(1 << 26, 8 * r_n - 1))}
    jobs = _log_size(rng, 100, 10_000)
    return {"kind": kind, "jobs": jobs, "total": jobs * rng.randint(2_000, 26_000), "plan_seed": rng.randint(0, 10**6)}


# ------------------------------------------------------------------ inputs
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _ints(g, n, wide, below=None):
    """n random integers of the full range of their type, or of [0, below)."""
    dt = torch.int64 if wide else torch.int32
    lo, hi = (0, below) if below else ((-(1 << 62), 1 << 62) if wide else (-(1 << 31), 1 << 31))
    return torch.randint(lo, hi, (n,), generator=g, device="cuda", dtype=dt)


def _local_permutation(g, n):
    """A permutation that shuffles blocks of BLOCK elements and the elements of each; the ragged rest within itself."""
    nb = n // BLOCK
    idx = torch.empty(n, dtype=torch.int32, device="cuda")
    step = 4096  # blocks at a time
    to = torch.randperm(nb, generator=g, device="cuda", dtype=torch.int32) * BLOCK
    for b in range(0, nb, step):
        e = min(nb, b + step)
        inside = torch.rand(e - b, BLOCK, generator=g, device="cuda").argsort(dim=1).to(torch.int32)
        idx[b * BLOCK:e * BLOCK] = (inside + to[b:e, None]).reshape(-1)
    rest = n - nb * BLOCK
    if rest:
        idx[nb * BLOCK:] = torch.randperm(rest, generator=g, device="cuda", dtype=torch.int32) + nb * BLOCK
    return idx


def _split_keys(g, n, buckets, wide, zipf):
    """Keys whose low bits are the bucket (uniform, or Zipf over the ranks 1..buckets) below random high bits."""
    keys = _ints(g, n, wide)
    if zipf:
        w = 1.0 / torch.arange(1, buckets + 1, device="cuda", dtype=torch.float64)
        cdf = torch.cumsum(w, 0) / w.sum()
        for a in range(0, n, 1 << 24):
            u = torch.rand(min(1 << 24, n - a), generator=g, device="cuda", dtype=torch.float64)
            b = torch.searchsorted(cdf, u).clamp_(max=buckets - 1).to(keys.dtype)
            keys[a:a + u.numel()] &= ~(buckets - 1)
            keys[a:a + u.numel()] |= b
    return keys


def _batch_plan(case):
    """[(kind, width, n)] of a batch: lengths log-uniform over [2^4, 2^18] about the mean that `total` asks for, kinds and
    widths uniform, as a query engine's small operators come."""
    rng = random.Random(case["plan_seed"])
    raw = [math.exp(rng.uniform(math.log(16), math.log(1 << 18))) for _ in range(case["jobs"])]
    scale = case["total"] / sum(raw)
    return [(rng.choice(("scan", "split", "gather")), rng.choice((4, 8)), max(16, min(1 << 20, round(scale * x))))
            for x in raw]


def _batch_layout(case):
    """Per (kind, width): the jobs' lengths and their starts in one arena (64-element aligned), and its length."""
    out = {}
    for kind, width, n in _batch_plan(case):
        a = out.setdefault((kind, width), {"n": [], "at": [], "len": 0})
        a["n"].append(n)
        a["at"].append(a["len"])
        a["len"] += -(-n // 64) * 64
    return dict(sorted(out.items()))


def _batch_inputs(case, seed):
    """One arena of inputs per (kind, width)."""
    g = _generator(seed)
    layout = _batch_layout(case)
    for (kind, width), a in layout.items():
        wide = width == 8
        if kind == "scan":
            a["in"] = _ints(g, a["len"], wide, 16)
        else:
            a["in"] = _ints(g, a["len"], wide)
        if kind == "split":
            a["vals"] = torch.arange(a["len"], dtype=torch.int32, device="cuda")
        if kind == "gather":
            # a random permutation of every job's range: positions ordered by (job, random number)
            starts = torch.tensor(a["at"] + [a["len"]], device="cuda")
            job = torch.repeat_interleave(torch.arange(len(a["n"]), device="cuda"), starts[1:] - starts[:-1])
            inside = torch.arange(a["len"], device="cuda") - starts[job]
            pad = inside >= torch.tensor(a["n"], device="cuda")[job]
            r = torch.randint(0, 1 << 30, (a["len"],), generator=g, device="cuda") | (pad.to(torch.int64) << 31)
            a["idx"] = (torch.argsort((job << 32) | r) - starts[job]).to(torch.int32)
    return layout


def _inputs(case, seed):
    g = _generator(seed)
    kind = case["kind"]
    if kind == "scan":
        return {"in": _ints(g, case["n"], case["wide"], 16 if case["small_values"] else None)}
    if kind == "permute":
        n = case["n"]
        idx = (_local_permutation(g, n) if case["local"]
               else torch.randperm(n, generator=g, device="cuda", dtype=torch.int32))
        return {"in": _ints(g, n, case["wide"]), "idx": idx}
    if kind == "split":
        d = {"keys": _split_keys(g, case["n"], case["buckets"], case["wide"], case["zipf"])}
        if case["values"]:
            d["vals"] = torch.arange(case["n"], dtype=torch.int32, device="cuda")
        return d
    if kind == "sort":
        d = {"keys": _ints(g, case["n"], False)}
        if case["values"]:
            d["vals"] = torch.arange(case["n"], dtype=torch.int32, device="cuda")
        return d
    if kind == "join":
        # S refers to rows of R, as a foreign key does
        r = _ints(g, case["r_n"], False)
        at = torch.randint(0, case["r_n"], (case["s_n"],), generator=g, device="cuda")
        return {"r": r, "s": r[at]}
    return _batch_inputs(case, seed)


# ------------------------------------------------------------------ calls
def prepare(case, seed):
    st = {"case": case, "ctx": edpp.Context(0, stream=torch.cuda.current_stream().cuda_stream)}
    d = st["in"] = _inputs(case, seed)
    kind = case["kind"]
    if kind == "scan":
        st["out"] = torch.zeros_like(d["in"])
        st["total"] = torch.zeros(1, dtype=d["in"].dtype, device="cuda")
    elif kind == "permute":
        st["gathered"] = torch.zeros_like(d["in"])
        st["scattered"] = torch.zeros_like(d["in"])
    elif kind == "split":
        st["keys"] = torch.zeros_like(d["keys"])
        st["vals"] = torch.zeros_like(d["vals"]) if case["values"] else None
        st["start"] = torch.zeros(case["buckets"], dtype=torch.int32, device="cuda")
    elif kind == "sort":
        st["keys"] = torch.zeros_like(d["keys"])
        st["vals"] = torch.zeros_like(d["vals"]) if case["values"] else None
    elif kind == "join":
        st["count"] = torch.zeros(1, dtype=torch.int64, device="cuda")
    else:
        jobs = []
        for (op, width), a in d.items():
            a["out"] = torch.zeros_like(a["in"])
            if op == "scan":
                a["total"] = torch.zeros(len(a["n"]), dtype=a["in"].dtype, device="cuda")
            elif op == "split":
                a["vout"] = torch.zeros_like(a["vals"])
                a["start"] = torch.zeros(len(a["n"]), BATCH_BUCKETS, dtype=torch.int32, device="cuda")
            for j, (at, n) in enumerate(zip(a["at"], a["n"])):
                src, dst = a["in"][at:at + n], a["out"][at:at + n]
                if op == "scan":
                    jobs.append(edpp.make_job(edpp.JOB_SCAN, n, src, dst, width, aux=a["total"][j:j + 1]))
                elif op == "split":
                    jobs.append(edpp.make_job(edpp.JOB_SPLIT, n, src, dst, width, buckets=BATCH_BUCKETS,
                                              vals_in=a["vals"][at:at + n], vals_out=a["vout"][at:at + n],
                                              aux=a["start"][j]))
                else:
                    jobs.append(edpp.make_job(edpp.JOB_GATHER, n, src, dst, width, idx=a["idx"][at:at + n]))
        random.Random(case["plan_seed"]).shuffle(jobs)
        st["batch"] = edpp.Batch(st["ctx"], jobs)
    return st


def run(state):
    case, ctx, d = state["case"], state["ctx"], state["in"]
    kind = case["kind"]
    if kind == "scan":
        ctx.scan(d["in"], state["out"], total=state["total"], wide=case["wide"])
        return {"out": state["out"], "total": state["total"]}
    if kind == "permute":
        ctx.gather(d["in"], state["gathered"], d["idx"], wide=case["wide"])
        ctx.scatter(d["in"], state["scattered"], d["idx"], wide=case["wide"])
        return {"gathered": state["gathered"], "scattered": state["scattered"]}
    if kind == "split":
        ctx.split(d["keys"], state["keys"], case["buckets"], d.get("vals"), state["vals"], state["start"],
                  wide=case["wide"])
        return {"keys": state["keys"], "vals": state["vals"], "start": state["start"]}
    if kind == "sort":
        ctx.sort(d["keys"], state["keys"], d.get("vals"), state["vals"], signed=case["signed"])
        return {"keys": state["keys"], "vals": state["vals"]}
    if kind == "join":
        ctx.join_count(d["r"], d["s"], state["count"])
        return {"count": state["count"]}
    state["batch"].run()
    return {"%s%d" % k: {name: a[name] for name in ("out", "vout", "start", "total") if name in a}
            for k, a in d.items()}


def work(case):
    kind = case["kind"]
    if kind == "scan":
        return {"bytes": 2 * (8 if case["wide"] else 4) * case["n"], "flops": case["n"]}
    if kind == "permute":  # a gather and a scatter: index, source and destination once each
        return {"bytes": 2 * (2 * (8 if case["wide"] else 4) + 4) * case["n"], "flops": 0}
    if kind == "split":
        per = 2 * ((8 if case["wide"] else 4) + (4 if case["values"] else 0))
        return {"bytes": per * case["n"] + 4 * case["buckets"], "flops": 0}
    if kind == "sort":
        return {"bytes": (16 if case["values"] else 8) * case["n"], "flops": 0}
    if kind == "join":
        return {"bytes": 4 * (case["r_n"] + case["s_n"]) + 8, "flops": 0}
    total = 0
    for op, width, n in _batch_plan(case):
        total += {"scan": 2 * width * n + width, "split": (2 * width + 8) * n + 4 * BATCH_BUCKETS,
                  "gather": (2 * width + 4) * n}[op]
    return {"bytes": total, "flops": 0}


# ------------------------------------------------------------------ what the calls define
def _exact_scan(x):
    """Exclusive sums and the total, wrapping as the type does."""
    s = torch.cumsum(x, 0, dtype=torch.int64)
    return (s - x).to(x.dtype), s[-1:].to(x.dtype)


def _exact_split(keys, vals, buckets):
    b = (keys & (buckets - 1)).to(torch.int16 if buckets <= 1 << 14 else torch.int32)
    order = torch.sort(b, stable=True).indices
    count = torch.bincount(b.to(torch.int32), minlength=buckets)
    return keys[order], vals[order] if vals is not None else None, (torch.cumsum(count, 0) - count).to(torch.int32)


def exact(case, seed):
    kind = case["kind"]
    d = _inputs(case, seed)
    if kind == "scan":
        out, total = _exact_scan(d["in"])
        return {"out": out, "total": total}
    if kind == "permute":
        back = torch.empty_like(d["in"])
        at = d["idx"].long()
        back[at] = d["in"]
        return {"gathered": d["in"][at], "scattered": back}
    if kind == "split":
        k, v, start = _exact_split(d["keys"], d.get("vals"), case["buckets"])
        return {"keys": k, "vals": v, "start": start}
    if kind == "sort":
        k = d["keys"]
        if not case["signed"]:  # unsigned order: the sign bit turned
            k = k ^ -(1 << 31)
        order = torch.sort(k, stable=True).indices
        return {"keys": d["keys"][order], "vals": d["vals"][order] if case["values"] else None}
    if kind == "join":
        keys, count = torch.unique(d["r"], return_counts=True)
        at = torch.searchsorted(keys, d["s"]).clamp_(max=keys.numel() - 1)
        return {"count": torch.where(keys[at] == d["s"], count[at], 0).sum().reshape(1)}
    out = {}
    for (op, width), a in d.items():
        r = {"out": torch.zeros_like(a["in"])}
        if op == "scan":
            r["total"] = torch.zeros(len(a["n"]), dtype=a["in"].dtype, device="cuda")
        elif op == "split":
            r["vout"] = torch.zeros_like(a["vals"])
            r["start"] = torch.zeros(len(a["n"]), BATCH_BUCKETS, dtype=torch.int32, device="cuda")
        for j, (at, n) in enumerate(zip(a["at"], a["n"])):
            s = slice(at, at + n)
            if op == "scan":
                r["out"][s], r["total"][j:j + 1] = _exact_scan(a["in"][s])
            elif op == "split":
                r["out"][s], r["vout"][s], r["start"][j] = _exact_split(a["in"][s], a["vals"][s], BATCH_BUCKETS)
            else:
                r["out"][s] = a["in"][s][a["idx"][s].long()]
        out["%s%d" % (op, width)] = r
    return out
