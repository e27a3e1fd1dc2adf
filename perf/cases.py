"""The work a user has this library do, as measurable cases.

Every case is one call (or one short sequence of calls) of a public entry point of
`gpurecsplit_amd`: building an MPHF from keys in device or host memory or from
strings, building many at once, building through a plan, and querying one in bulk.
Keys are uniform 128-bit hashes (what a string or integer key becomes before it
reaches the construction), so the generator's stream stands for any key set.

  listed()            the cases
  draw(rng)           one more case of the same ranges
  prepare(case, seed) inputs, contexts, plans and structures, on the GPU
  run(state)          one pass; returns the bytes or indexes the user gets
  work(case)          bytes and operations a pass cannot do without
  exact(case, seed)   None: outputs are bytes and indexes, not rounded numbers
"""
import math

import numpy as np
import torch

import gpurecsplit_amd as gra
from gpurecsplit_amd.keys import splitmix64_keys_device

# Operations of one key-seed evaluation: 64-bit add (2), fold (1), MurmurHash3 fmix32
# to 16 bits (9), remap (2), update of the node's predicate (2).
OPS_PER_EVAL = 16


def _case(name, kind, n, leaf, bucket, rotate=True, remap64=False, sets=1, structure=0):
    return {"name": name, "kind": kind, "n": n, "leaf": leaf, "bucket": bucket, "rotate": rotate,
            "remap64": remap64, "sets": sets, "structure": structure}


def listed():
    return [
        # A small function built on the fly (one partition, one block of a file):
        # latency of the launches and host round trips.
        _case("build_1k_l8", "device", 1_000, 8, 100),
        # An index of one medium table or one served job.
        _case("build_100k_l12", "device", 100_000, 12, 100),
        # The quick-construction setting on a million keys that start in host
        # memory, as the drop-in constructor takes them.
        _case("build_1m_l8_host", "host", 1_000_000, 8, 100),
        # The compact setting at full size, the headline configuration.
        _case("build_5m_l16", "device", 5_000_000, 16, 2000),
        # Small buckets of large leaves: almost all time goes to the leaves.
        _case("build_5m_l18", "device", 5_000_000, 18, 50),
        # The most compact setting, a few buckets (a key costs about 400 times the
        # headline's), not a multiple of the bucket size.
        _case("build_7k_l24", "device", 7_001, 24, 2000),
        # Without rotation fitting, keys in host memory, an odd count.
        _case("build_500k_l13_brute_host", "host", 500_003, 13, 200, rotate=False),
        # The 64-bit-remap variant.
        _case("build_200k_l14_remap64", "device", 200_009, 14, 500, remap64=True),
        # Many functions of very different sizes at once (one per shard, key sets of
        # 1e3 to 1e6 keys).
        _case("batch_512_l12", "batch", 1_000_000, 12, 100, sets=512),
        # A compact function of a fixed size built again and again through a plan.
        _case("plan_100k_l16", "plan", 100_000, 16, 2000),
        # String keys, hashed on the GPU.
        _case("strings_100k_l8", "strings", 100_000, 8, 100),
        # Bulk lookups, in random order, in a function over as many keys.
        _case("query_3m_l12", "query", 3_000_000, 12, 100, structure=3_000_000),
    ]


# Largest key count drawn per kind, and the expected evaluations a drawn pass may
# cost (the headline build's are 2.4e12; the 64-bit remap costs several times more
# per evaluation).
_MAX_N = {"device": 5_000_000, "host": 5_000_000, "batch": 1_000_000, "plan": 1_000_000, "strings": 200_000,
          "query": 3_000_000}
_MAX_EVALS = 8.0e11


def draw(rng):
    kind = rng.choice(["device", "device", "device", "host", "batch", "plan", "strings", "query"])
    leaf = rng.choice([4, 6, 8, 8, 10, 11, 12, 12, 13, 14, 15, 16, 16, 17, 18, 18, 20, 22, 24])
    bucket = rng.choice([20, 50, 100, 100, 200, 500, 1000, 2000])
    if kind in ("batch", "strings", "query"):
        leaf, bucket = min(leaf, 14), min(bucket, 500)
    rotate, remap64 = rng.random() < 0.85, rng.random() < 0.12
    n = int(round(math.exp(rng.uniform(math.log(1_000), math.log(_MAX_N[kind])))))
    sets = int(round(math.exp(rng.uniform(math.log(8), math.log(512))))) if kind == "batch" else 1
    structure = int(round(math.exp(rng.uniform(math.log(1_000), math.log(2_000_000))))) if kind == "query" else 0
    c = _case("", kind, n, leaf, bucket, rotate, remap64, sets, structure)
    limit = _MAX_EVALS / 4 if remap64 else _MAX_EVALS
    while _evals(c)[0] > limit and c["n"] > 1_000:
        c["n"] = max(1_000, c["n"] // 2 - 1)
    while _evals(c)[0] > limit:  # large leaves without rotations, or with the slower remap
        c["leaf"] -= 2
    del c["name"]
    return c


# ---------------------------------------------------------------- inputs and passes

def _batch_sizes(case):
    """Key counts of a batch's sets, part of the case: log-uniform in [1e3, n]."""
    rng = np.random.default_rng(case["sets"])
    lo, hi = math.log(min(1_000, case["n"])), math.log(case["n"])
    return np.exp(rng.uniform(lo, hi, size=case["sets"])).astype(np.int64).clip(1)


def _strings(n, seed):
    """Distinct keys of 12 to about 90 bytes, like paths of one site."""
    rng = np.random.default_rng(seed)
    parts = rng.integers(0, 1 << 62, size=(n, 2))
    depth = rng.integers(0, 5, size=n)
    return [f"/{i:x}/{a:x}" + f"/{b:016x}" * d for i, ((a, b), d) in enumerate(zip(parts.tolist(), depth.tolist()))]


def prepare(case, seed):
    kind, n = case["kind"], case["n"]
    ctx = gra.Context.default(0)
    opt = {"leaf_size": case["leaf"], "rotate": case["rotate"], "remap64": case["remap64"], "ctx": ctx}
    state = {"kind": kind, "bucket": case["bucket"], "opt": opt}
    if kind == "strings":
        state["keys"] = _strings(n, seed)
    elif kind == "batch":
        state["offsets"] = np.concatenate([[0], np.cumsum(_batch_sizes(case))]).astype(np.uint64)
        state["keys"] = splitmix64_keys_device(seed, int(state["offsets"][-1]))
    elif kind == "query":
        built = splitmix64_keys_device(seed, case["structure"])
        state["rs"] = gra.GPURecSplit(built, case["bucket"], **opt)
        g = torch.Generator(device="cuda:0")
        g.manual_seed(seed)
        state["keys"] = built[torch.randint(case["structure"], (n,), device="cuda:0", generator=g)]
    elif kind == "host":
        state["keys"] = splitmix64_keys_device(seed, n).cpu().numpy().view(np.uint64)
    else:
        state["keys"] = splitmix64_keys_device(seed, n)
        if kind == "plan":
            state["plan"] = gra.Plan(n, case["bucket"], **opt)
    if kind != "query":
        # room for any structure of these keys (about 0.2 to 0.5 bytes per key)
        total = int(state["offsets"][-1]) if kind == "batch" else n
        state["out"] = np.zeros(total + 4096 * case["sets"], dtype=np.uint8)
    return state


def _store(state, blobs):
    """Writes serialized structures back to back into the caller's buffer, as a
    program that ships or stores them does; returns the buffer and their lengths."""
    out, at = state["out"], 0
    for data in blobs:
        out[at:at + len(data)] = np.frombuffer(data, dtype=np.uint8)
        at += len(data)
    return out, np.array([len(data) for data in blobs], dtype=np.int64)


def run(state):
    kind, keys, bucket, opt = state["kind"], state["keys"], state["bucket"], state["opt"]
    if kind == "query":
        return state["rs"].query_device(keys)
    if kind == "plan":
        return _store(state, [state["plan"].build(keys)])
    if kind == "batch":
        built, _ = gra.build_batch(keys, state["offsets"], bucket, **opt)
    elif kind == "strings":
        built = [gra.GPURecSplit.from_strings(keys, bucket, **opt)]
    else:
        built = [gra.GPURecSplit(keys, bucket, **opt)]
    out = _store(state, [rs.serialize() for rs in built])
    for rs in built:
        rs.close()
    return out


def exact(case, seed):
    """Outputs are bytes of a fixed format and indexes, the same for every correct
    construction; no computed number is rounded."""
    return None


# ---------------------------------------------------------------- work

def _alive(m, unit, fan):
    """Expected keys read per candidate of a node of m keys in `fan` parts of `unit`
    (the last part may be smaller) when a candidate stops at the first part that
    overflows: the sum over k of P(no part above `unit` after k keys)."""
    lam = m / fan
    j = np.arange(m + 1)
    logf = np.concatenate([[0.0], np.cumsum(np.log(np.arange(1, m + 1)))])
    part = np.where(j <= unit, np.exp(j * math.log(lam) - lam - logf), 0.0)
    total = np.ones(1)
    for _ in range(fan):
        total = np.convolve(total, part)[: m + 1]
    every = np.exp(j * math.log(m) - m - logf)
    return float(np.minimum(total[:m] / np.maximum(every[:m], 1e-300), 1.0).sum())


def _node_evals(m, unit, fan, leaf, rotate):
    """Expected evaluations of one node's search: candidates tried times keys read."""
    if unit == 1:
        alive = _alive(m, 1, m)
        log_p = math.lgamma(m + 1) - m * math.log(m)
        if not (rotate and m == leaf):
            return math.exp(-log_p) * alive
        # an even and an odd half of about m / 2 keys each, all m rotations at once
        half = m // 2
        f = math.exp(math.lgamma(m + 1) - math.lgamma(m - half + 1) - half * math.log(m))
        first = sum(math.exp(math.lgamma(m + 1) - math.lgamma(m - k + 1) - k * math.log(m)) for k in range(half))
        return math.exp(-log_p) / m * first * (1.0 + f)
    sizes = [unit] * (fan - 1) + [m - (fan - 1) * unit]
    log_p = math.lgamma(m + 1) + sum(s * math.log(s / m) - math.lgamma(s + 1) for s in sizes)
    return math.exp(-log_p) * (m if fan == 2 else _alive(m, unit, fan))


def _tree_evals(m, leaf, rotate, memo):
    """Expected evaluations of the split tree of a bucket of m keys."""
    if m < 2:
        return 0.0
    if m in memo:
        return memo[m]
    lower = leaf * (max(2, math.ceil(0.35 * leaf + 0.5)))
    upper = lower * (2 if leaf < 7 else math.ceil(0.21 * leaf + 0.9))
    if m <= leaf:
        e = _node_evals(m, 1, m, leaf, rotate)
    else:
        if m > upper:
            unit, fan = -(-(m // 2) // upper) * upper, 2
        else:
            unit = lower if m > lower else leaf
            fan = -(-m // unit)
        last = m - (fan - 1) * unit
        e = _node_evals(m, unit, fan, leaf, rotate)
        e += (fan - 1) * _tree_evals(unit, leaf, rotate, memo) + _tree_evals(last, leaf, rotate, memo)
    memo[m] = e
    return e


def _evals(case):
    """(expected evaluations, keys) of a build of the case, at the mean bucket size."""
    if case["kind"] == "batch":
        lo = min(1_000, case["n"])
        n = case["sets"] * ((case["n"] - lo) / math.log(case["n"] / lo) if case["n"] > lo else lo)
    else:
        n = case["structure"] or case["n"]
    b = min(case["bucket"], max(2, int(n)))
    return n / b * _tree_evals(b, case["leaf"], case["rotate"], {}), n


def work(case):
    evals, n = _evals(case)
    if case["kind"] == "query":
        # the key, one descriptor walk (about one evaluation per tree level) and the index
        return {"bytes": case["n"] * 24 + int(case["structure"] * 0.25), "flops": case["n"] * 4 * OPS_PER_EVAL}
    # keys in, about 2 bits per key out
    return {"bytes": int(n * (50 if case["kind"] == "strings" else 16) + n * 0.25), "flops": evals * OPS_PER_EVAL}
