"""The workloads this runtime is timed on, each through its public entry points.

A case names one program of the C ABI and its sizes. `prepare` makes what a
user's program has in hand before the call (device inputs and outputs, a graph
batch, a running server), `run` makes one pass and returns every output,
`work` says what a pass cannot do without, and `exact` walks the photon
workload in plain 64-bit torch, the only one whose outputs are not whole
numbers. Device memory is torch's; the entry points take its addresses.
"""

import ctypes
import math

import numpy as np
import torch

import harmonize_amd as hz

# Promises are 16 bytes in every integer workload and 40 in the photon walk.
# Mean Collatz steps of a start near n: 10.41 ln n (3n + 1 and n / 2 counted
# apart); mean events per source photon of the default walk: 21.6.
STEPS_PER_LN = 10.41
EVENTS_PER_PHOTON = 21.6

# The configuration the autotuner chose for batches of this class on this
# device (split threshold in spec_param); {} is the library's own default.
BFS_TUNED = {"groups": 2048, "queues": 16, "block_groups": 4, "stash": 8, "spec_param": 128}


def listed():
    return [
        # A request of a few starts: what a call costs before it has any size.
        {"name": "collatz-1k", "kind": "collatz", "program": "async", "count": 1024, "bits": 32},
        # An ordinary job, no multiple of the 64-lane wavefront.
        {"name": "collatz-300k", "kind": "collatz", "program": "async", "count": 300007, "bits": 32},
        # Collatz at scale: the benchmark's headline workload.
        {"name": "collatz-64m", "kind": "collatz", "program": "async", "count": 1 << 26, "bits": 40},
        # The level-synchronous program on the configuration of 2^20 starts.
        {"name": "collatz-event-1m", "kind": "collatz", "program": "event", "count": 1 << 20, "bits": 32},
        # A small Monte Carlo batch with a coarse tally of odd length.
        {"name": "photon-5k", "kind": "photon", "program": "async", "count": 5003, "bins": 257},
        # The branching photon walk at its default size.
        {"name": "photon-10m", "kind": "photon", "program": "async", "count": 10000000, "bins": 1000},
        # The same walk, a generation a launch.
        {"name": "photon-event-1m", "kind": "photon", "program": "event", "count": 1000003, "bins": 1000},
        # Many graphs searched by one program: the benchmark's batch.
        {"name": "bfs-async-64", "kind": "bfs", "program": "async", "graphs": 64, "low": 14.0, "high": 22.0,
         "tuned": True},
        {"name": "bfs-event-64", "kind": "bfs", "program": "event", "graphs": 64, "low": 14.0, "high": 22.0,
         "tuned": False},
        # Value-returning operations: a tree of futures whose total is read by many.
        {"name": "futures-1m", "kind": "futures", "leaves": 1 << 20, "readers": 1 << 14},
        # Promises held on few, long barriers beside as many free ones.
        {"name": "barrier-4m", "kind": "barrier", "dep": 1 << 21, "free": 1 << 21, "barriers": 64},
        # A burst of jobs served by a resident kernel, outputs read back.
        {"name": "serve-48", "kind": "serve", "jobs": 48, "low": 10.0, "high": 20.0},
    ]


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["collatz", "collatz", "collatz-event", "photon", "photon", "photon-event", "bfs", "bfs",
                       "futures", "barrier", "serve"])
    if kind == "collatz":
        return {"kind": "collatz", "program": "async", "count": _log_uniform(rng, 1 << 10, 1 << 26),
                "bits": rng.choice([32, 40])}
    if kind == "collatz-event":
        return {"kind": "collatz", "program": "event", "count": _log_uniform(rng, 1 << 12, 1 << 20),
                "bits": rng.choice([32, 40])}
    if kind == "photon":
        return {"kind": "photon", "program": "async", "count": _log_uniform(rng, 1 << 10, 10000000),
                "bins": _log_uniform(rng, 64, 1000)}
    if kind == "photon-event":
        return {"kind": "photon", "program": "event", "count": _log_uniform(rng, 1 << 12, 1000003),
                "bins": _log_uniform(rng, 64, 1000)}
    if kind == "bfs":
        program = rng.choice(["async", "event"])
        return {"kind": "bfs", "program": program, "graphs": rng.randint(1, 48), "low": 10.0,
                "high": round(rng.uniform(14.0, 21.0), 2), "tuned": program == "async" and rng.random() < 0.5}
    if kind == "futures":
        return {"kind": "futures", "leaves": 1 << rng.randint(8, 20), "readers": _log_uniform(rng, 1, 1 << 14) - 1}
    if kind == "barrier":
        return {"kind": "barrier", "dep": _log_uniform(rng, 1 << 12, 1 << 21), "free": _log_uniform(rng, 1 << 12, 1 << 21),
                "barriers": _log_uniform(rng, 16, 1024)}
    return {"kind": "serve", "jobs": rng.randint(4, 48), "low": 10.0, "high": round(rng.uniform(14.0, 20.0), 2)}


def _call(name, *args):
    hz.check(getattr(hz.lib(), name)(*args), name)


def _sizes(case, count):
    """Log-uniform sizes in [2^low, 2^high], the same ones for every seed of a case."""
    rng = np.random.default_rng(count)
    return np.rint(2.0 ** rng.uniform(case["low"], case["high"], size=count)).astype(np.int64)


def _starts(seed, count, bits):
    """Starts uniform in [1, 2^bits)."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randint(1, 1 << bits, (count,), dtype=torch.int64, device="cuda", generator=g)


def _photon_params(case, seed):
    return hz.photon_params(photons=case["count"], bins=case["bins"], seed=seed * 0x9E3779B1 + 0x5EED)


def prepare(case, seed):
    kind = case["kind"]
    state = {"case": case, "config": hz.make_config(max_launches=1 << 20), "stats": hz.RunStats()}
    if kind == "collatz":
        state["starts"] = _starts(seed, case["count"], case["bits"])
        state["steps"] = torch.empty(case["count"], dtype=torch.int32, device="cuda")
        if case["program"] == "async" and case["count"] >= 1 << 22:
            # What the benchmark runs the workload at scale with.
            state["config"] = hz.make_config(arena=1 << 18, queues=16)
    elif kind == "photon":
        params = state["params"] = _photon_params(case, seed)
        state["tally"] = torch.empty((params.replicas, params.bins + hz.PHOTON_EXTRA_SLOTS), dtype=torch.float64,
                                     device="cuda")
        state["events"] = torch.empty(case["count"], dtype=torch.int32, device="cuda")
    elif kind == "bfs":
        state["batch"] = hz.BfsBatch.rmat(seed, _sizes(case, case["graphs"]).astype(np.uint32))
        state["config"] = hz.make_config(max_launches=1 << 16)
        if case["program"] == "async":
            state["config"] = hz.make_config(flags=hz.RUN_GRAPH, **(BFS_TUNED if case["tuned"] else {}))
        state["levels"] = torch.as_tensor(_DeviceLevels(state["batch"]), device="cuda")
    elif kind == "futures":
        state["starts"] = _starts(seed, case["leaves"], 20)
        state["echo"] = torch.empty(max(1, case["readers"]), dtype=torch.int64, device="cuda")
        state["forwarded"] = torch.empty_like(state["echo"])
        state["total"] = ctypes.c_uint64()
    elif kind == "barrier":
        # Steps are numbered, not drawn: the seed moves the free ones' count.
        state["free"] = case["free"] - seed % 61
        state["config"] = hz.make_config(arena=1 << 17, max_launches=1000)
        state["hits"] = torch.empty(case["dep"], dtype=torch.int32, device="cuda")
        state["counter"] = torch.empty(1, dtype=torch.int32, device="cuda")
        state["violations"] = torch.empty(1, dtype=torch.int32, device="cuda")
    else:
        rng = np.random.default_rng(seed + 1)
        sizes = _sizes(case, case["jobs"])
        state["trace"] = list(zip(sizes.tolist(), rng.integers(1, 1 << 40, size=len(sizes)).tolist()))
        state["arrivals"] = np.zeros(len(sizes))
        state["server"] = hz.Resident(pool_bytes=2 << 30, keep_outputs=True)
    return state


class _DeviceLevels:
    """The batch's level array where the search leaves it, for torch to view."""

    def __init__(self, batch):
        info = hz.BfsInfo()
        _call("hz_bfs_batch_info", batch.handle, ctypes.byref(info))
        self.batch = batch  # the view keeps the batch alive
        self.__cuda_array_interface__ = {"shape": (info.total_vertices,), "typestr": "<i4", "version": 2,
                                         "data": (info.d_level, False)}


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    config, stats = ctypes.byref(state["config"]), ctypes.byref(state["stats"])
    if kind == "collatz":
        _call("hz_collatz_run", hz.KINDS[case["program"]], state["starts"].data_ptr(), case["count"],
              state["steps"].data_ptr(), config, stats)
        return {"steps": state["steps"], "promises": state["stats"].promises}
    if kind == "photon":
        _call("hz_photon_run", hz.KINDS[case["program"]], ctypes.byref(state["params"]), state["tally"].data_ptr(),
              state["events"].data_ptr(), config, stats)
        return {"events": state["events"], "promises": state["stats"].promises, "tally": state["tally"].sum(dim=0)}
    if kind == "bfs":
        _call("hz_bfs_batch_run", state["batch"].handle, hz.KINDS[case["program"]], config, stats)
        return {"levels": state["levels"]}
    if kind == "futures":
        _call("hz_futures_run", hz.ASYNC, state["starts"].data_ptr(), case["leaves"], case["readers"],
              state["echo"].data_ptr(), state["forwarded"].data_ptr(), ctypes.byref(state["total"]), config, stats)
        return {"total": state["total"].value, "promises": state["stats"].promises,
                "echo": state["echo"][:case["readers"]], "forwarded": state["forwarded"][:case["readers"]]}
    if kind == "barrier":
        _call("hz_barrier_run", case["dep"], state["free"], case["barriers"], state["counter"].data_ptr(),
              state["hits"].data_ptr(), state["violations"].data_ptr(), config, stats)
        return {"counter": state["counter"], "hits": state["hits"], "violations": state["violations"]}
    server = state["server"]
    jobs = server.run_trace(state["trace"], state["arrivals"])
    steps = np.concatenate([server.output(j["id"]) for j in jobs])
    for j in jobs:
        server.release(j["id"])
    return {"steps": steps.view(np.int32)}


def work(case):
    """Bytes of inputs read and outputs written once, and the operations the
    promises take whatever runs them: 4 for a Collatz step (parity, shift or
    multiply-add, count), about 400 for a photon event (two Philox draws, a
    logarithm, a square root), 2 for an edge, 6 for a future's or a barrier's
    promise."""
    kind = case["kind"]
    if kind == "collatz":
        steps = STEPS_PER_LN * (math.log(2.0) * case["bits"] - 1.0)
        return {"bytes": 12.0 * case["count"], "flops": 4.0 * steps * case["count"]}
    if kind == "photon":
        return {"bytes": 4.0 * case["count"] + 8.0 * (case["bins"] + hz.PHOTON_EXTRA_SLOTS),
                "flops": 400.0 * EVENTS_PER_PHOTON * case["count"]}
    if kind == "bfs":
        a, b = case["low"] * math.log(2.0), case["high"] * math.log(2.0)
        vertices = case["graphs"] * (math.exp(b) - math.exp(a)) / max(b - a, 1e-9)
        # Row offsets read, levels written, 16 edges a vertex read.
        return {"bytes": (8.0 + 4.0 * 16.0) * vertices, "flops": 2.0 * 16.0 * vertices}
    if kind == "futures":
        steps = STEPS_PER_LN * (math.log(2.0) * 20 - 1.0)
        return {"bytes": 8.0 * case["leaves"] + 16.0 * case["readers"], "flops": 6.0 * (steps + 2.0) * case["leaves"]}
    if kind == "barrier":
        return {"bytes": 4.0 * case["dep"], "flops": 6.0 * (2.0 * case["dep"] + case["free"])}
    a, b = case["low"] * math.log(2.0), case["high"] * math.log(2.0)
    starts = case["jobs"] * (math.exp(b) - math.exp(a)) / (b - a)
    return {"bytes": 12.0 * starts, "flops": 4.0 * STEPS_PER_LN * (math.log(2.0) * 32 - 1.0) * starts}


# ------------------------------------------------------- the walk in 64 bits

_MASK = 0xFFFFFFFF


def _philox(c0, c1, c2, c3, k0, k1):
    """Philox4x32-10 (Salmon et al., SC'11) on int64 tensors of 32-bit words."""
    for _ in range(10):
        p0, p1 = c0 * 0xD2511F53, c2 * 0xCD9E8D57
        c0, c1, c2, c3 = (((p1 >> 32) & _MASK) ^ c1 ^ k0, p1 & _MASK, ((p0 >> 32) & _MASK) ^ c3 ^ k1, p0 & _MASK)
        k0, k1 = (k0 + 0x9E3779B9) & _MASK, (k1 + 0xBB67AE85) & _MASK
    return c0, c1, c2, c3


def _direction(a, b):
    """Marsaglia's disc method for one draw: a unit vector, and where it took."""
    v1, v2 = (a >> 8).double() / 8388608.0 - 1.0, (b >> 8).double() / 8388608.0 - 1.0
    s = v1 * v1 + v2 * v2
    t = 2.0 * torch.sqrt(torch.clamp(1.0 - s, min=0.0))
    return torch.stack([v1 * t, v2 * t, 1.0 - 2.0 * s]), (s > 0.0) & (s < 1.0)


def _lowbias32(h):
    h = h ^ (h >> 16)
    h = (h * 0x7FEB352D) & _MASK
    h = h ^ (h >> 15)
    h = (h * 0x846CA68B) & _MASK
    return h ^ (h >> 16)


def exact(case, seed):
    """The photon walk's tally with every quantity in binary64."""
    if case["kind"] != "photon":
        return None
    p = _photon_params(case, seed)
    f32 = lambda x: float(np.float32(x))  # the parameters as the call takes them
    thickness, albedo, k0, k1 = f32(p.thickness), f32(p.albedo), p.seed & _MASK, (p.seed >> 32) & _MASK
    dev, bins = "cuda", p.bins
    tally = torch.zeros(bins + 5, dtype=torch.float64, device=dev)
    book = lambda slots, values: tally.index_add_(0, slots, values)
    n = case["count"]
    pid = torch.arange(n, dtype=torch.int64, device=dev)
    lin = torch.zeros_like(pid)
    pos, way = torch.zeros((3, n), dtype=torch.float64, device=dev), torch.zeros((3, n), dtype=torch.float64, device=dev)
    way[2] = 1.0
    w = torch.ones(n, dtype=torch.float64, device=dev)
    event = 0
    while pid.numel() and event < p.max_events:
        ev = torch.full_like(pid, event)
        r0, r1, r2, r3 = _philox(pid, ev, lin, torch.zeros_like(pid), k0, k1)
        dist = -torch.log(((r0 >> 8) + 1).double() / 16777216.0) / f32(p.sigma_t)
        pos = pos + dist * way
        z = pos[2]
        out = (z < 0.0) | (z > thickness)
        book(torch.where(z[out] < 0.0, bins, bins + 1), w[out])
        keep = ~out
        pid, lin, pos, w, r1, r2, r3 = pid[keep], lin[keep], pos[:, keep], w[keep], r1[keep], r2[keep], r3[keep]
        z = pos[2]
        book((z * (bins / thickness)).long().clamp(max=bins - 1), w - w * albedo)
        w = w * albedo
        region = (z / f32(p.region_width)).long().clamp(max=p.regions - 1)
        target = torch.exp2(-region.double())
        ratio = w / target
        low = ratio < f32(p.roulette_below)
        dies = low & ((r1 >> 8).double() / 16777216.0 >= ratio)
        lives = low & ~dies
        book(torch.full_like(pid[dies], bins + 2), w[dies])
        book(torch.full_like(pid[lives], bins + 3), (target - w)[lives])
        copies = torch.ones_like(pid)
        for k in range(1, int(p.max_split).bit_length()):
            copies = torch.where(~low & (ratio > f32(p.split_above)) & (ratio >= float(1 << k)), 1 << k, copies)
        w = torch.where(lives, target, w / copies.double())
        if event + 1 >= p.max_events:
            book(torch.full_like(pid[~dies], bins + 4), (w * copies.double())[~dies])
            break
        copies = torch.where(dies, 0, copies)
        at = torch.repeat_interleave(torch.arange(pid.numel(), device=dev), copies)
        copy = torch.arange(at.numel(), device=dev) - (torch.cumsum(copies, 0) - copies)[at]
        parent = lin[at]
        pid, pos, w = pid[at], pos[:, at], w[at]
        way, good = _direction(r2[at], r3[at])
        good &= copy == 0
        for attempt in range(32):
            miss = torch.nonzero(~good).flatten()
            if not miss.numel():
                break
            q = _philox(pid[miss], torch.full_like(miss, event), parent[miss], 1 + (copy[miss] << 8) + attempt, k0, k1)
            for a, b in ((q[0], q[1]), (q[2], q[3])):
                d, ok = _direction(a, b)
                ok &= ~good[miss]
                way[:, miss[ok]] = d[:, ok]
                good[miss[ok]] = True
        child = parent ^ ((event * 0x9E3779B9) & _MASK) ^ (((copy + 1) * 0x85EBCA6B) & _MASK)
        lin = torch.where(copy == 0, parent, _lowbias32(child))
        event += 1
    return {"events": None, "promises": None, "tally": tally}
