"""The work a program has this framework do, as cases that can be timed.

A case is a dict of plain values; ``prepare`` makes, on the GPU, what a program
has in hand before the call, ``run`` makes the calls through the public API
(``Hashmap``, ``BatchedMaps``, ``hashinator_amd.tools``) and returns what they
give.  Every case ends in a state that is a function of its inputs (tables in
Robin Hood order, values and hit flags of lookups), so a pass can be repeated
on one state and compared slot for slot.

Kinds of case (``op``):

step     a fresh map of 2^sp slots, filled to ``lf``, then a retrieve of the
         keys and as many absent ones (the benchmark's step); ``form`` is how
         the keys are handed over: separate arrays, pairs, or keys whose
         values are their positions
retrieve a resident map answers ``n`` queries, ``hits`` of them present; the
         table in Robin Hood order or in arrival order
update   a resident map takes new values for ``n`` of its keys and is asked
         for them: the small calls of a program that iterates
churn    a resident map loses ``frac`` of its keys, is cleaned, answers
         queries for them and others, and takes them back
grow     a small map takes ``batches`` equal inserts at the default target
         load factor and grows on the way
extract  pairs under a rule and all keys of a resident map's bucket array
copy_if  stable compaction of pairs, by a built-in rule or by flags
scan     exclusive prefix sum
batch    many independent small maps: insert, retrieve, erase, clean
"""
from __future__ import annotations

import math

import numpy as np
import torch

from hashinator_amd import Hashmap
from hashinator_amd._lib import HN_PRED_LT, HN_PRED_MASKEQ
from hashinator_amd.batch import BatchedMaps
from hashinator_amd.tools import copy_if_flags, copy_if_pairs, copy_keys_if_pairs, pred, split_prefix_scan

DEV = "cuda"
_IDT = {32: torch.int32, 64: torch.int64}


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the smallest call: a map of a thousand slots made, filled and asked
        # (the unit-test sizes); latency and launches
        {"name": "step_u64_2p10", "op": "step", "bits": 64, "sp": 10, "lf": 0.5, "keys": "uniform", "form": "soa"},
        # a thousand keys at a time into a resident map, as an iterating program does
        {"name": "update_u32_2p20", "op": "update", "bits": 32, "sp": 20, "lf": 0.6, "keys": "uniform", "n": 1000},
        # the small map of the benchmark: 524,288 keys in 2^20 slots, cache-resident
        {"name": "step_u32_2p20", "op": "step", "bits": 32, "sp": 20, "lf": 0.5, "keys": "uniform", "form": "soa"},
        # the benchmark's headline map: 241.6 M keys, half uniform, half runs of ids, at load factor 0.9
        {"name": "step_u64_2p28", "op": "step", "bits": 64, "sp": 28, "lf": 0.9, "keys": "runs", "form": "soa"},
        # lookups with a ragged count in a table beyond the L2s
        {"name": "retrieve_u64_2p24", "op": "retrieve", "bits": 64, "sp": 24, "lf": 0.75, "keys": "runs",
         "n": 12_345_679, "hits": 0.5, "order": "home"},
        # the reference's own layout (clusters in arrival order), 32-bit keys, mostly present
        {"name": "retrieve_u32_2p22_arrival", "op": "retrieve", "bits": 32, "sp": 22, "lf": 0.8, "keys": "uniform",
         "n": 4_000_003, "hits": 0.9, "order": "arrival"},
        # erase a quarter, clean, look up, insert again: the benchmark's erase/clean stage at 2^26 slots
        {"name": "churn_u64_2p26", "op": "churn", "bits": 64, "sp": 26, "lf": 0.9, "keys": "runs", "frac": 0.25},
        # a map that starts small and grows at the default target load factor
        {"name": "grow_u64_12M", "op": "grow", "bits": 64, "sp": 16, "keys": "runs", "n": 12_000_001, "batches": 4},
        # extraction of a half-tombstoned table's pairs and keys
        {"name": "extract_u64_2p26", "op": "extract", "bits": 64, "sp": 26, "lf": 0.7, "keys": "uniform",
         "frac": 0.2},
        # stable compaction of pairs at a ragged size
        {"name": "copy_if_u64_2p27", "op": "copy_if", "bits": 64, "n": (1 << 27) + 4321, "keep": 0.3, "rule": "lt"},
        # the prefix scan at the benchmark's size
        {"name": "scan_u32_2p28", "op": "scan", "bits": 32, "n": 1 << 28},
        # many uneven maps of velocity-grid cells (2^8..2^16 slots, load factor 0.6) in one call
        {"name": "batch_u32_1024", "op": "batch", "bits": 32, "maps": 1024, "sp_lo": 8, "sp_hi": 16, "lf": 0.6,
         "frac": 0.2},
    ]


def _logint(rng, lo, hi):
    """An integer between lo and hi, spread over its logarithm, odd as often as even."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["step", "step", "retrieve", "retrieve", "update", "churn", "grow", "extract", "copy_if", "scan",
                     "batch"])
    bits = rng.choice([32, 64])
    keys = rng.choice(["uniform", "runs"])
    c = {"op": op, "bits": bits}
    if op == "step":
        c.update(sp=rng.randint(10, 26), lf=round(rng.uniform(0.3, 0.92), 3), keys=keys,
                 form=rng.choice(["soa", "soa", "pairs", "index"]))
    elif op == "retrieve":
        order = rng.choice(["home", "home", "arrival"])
        c.update(sp=rng.randint(12, 27), lf=round(rng.uniform(0.3, 0.9 if order == "home" else 0.8), 3), keys=keys,
                 n=_logint(rng, 1_000, 60_000_000), hits=round(rng.uniform(0.0, 1.0), 3), order=order)
    elif op == "update":
        sp = rng.randint(10, 24)
        c.update(sp=sp, lf=round(rng.uniform(0.3, 0.8), 3), keys=keys, n=_logint(rng, 8, 1 << (sp - 3)))
    elif op == "churn":
        c.update(sp=rng.randint(12, 26), lf=round(rng.uniform(0.4, 0.9), 3), keys=keys,
                 frac=round(rng.uniform(0.25, 0.5), 3))
    elif op == "grow":
        c.update(sp=rng.randint(5, 16), keys=keys, n=_logint(rng, 4_000, 24_000_000), batches=rng.randint(1, 4))
    elif op == "extract":
        c.update(sp=rng.randint(10, 26), lf=round(rng.uniform(0.3, 0.9), 3), keys=keys,
                 frac=round(rng.uniform(0.0, 0.5), 3))
    elif op == "copy_if":
        c.update(n=_logint(rng, 1_000, 1 << 27), keep=round(rng.uniform(0.05, 0.95), 3),
                 rule=rng.choice(["lt", "maskeq", "flags"]))
    elif op == "scan":
        c.update(n=_logint(rng, 1_000, 1 << (28 if bits == 32 else 27)))
    else:
        lo = rng.randint(6, 11)
        c.update(bits=rng.choice([32, 32, 64]), maps=_logint(rng, 16, 1024), sp_lo=lo, sp_hi=rng.randint(lo + 1, 16),
                 lf=round(rng.uniform(0.4, 0.8), 3), frac=round(rng.uniform(0.1, 0.5), 3))
    return c


# ------------------------------------------------------------------ inputs
def _lsr(x, s):
    return (x >> s) & ((1 << (64 - s)) - 1)


def _mix(x):
    """The SplitMix64 finalizer on int64 bit patterns."""
    x = (x ^ _lsr(x, 30)) * (0xBF58476D1CE4E5B9 - (1 << 64))
    x = (x ^ _lsr(x, 27)) * (0x94D049BB133111EB - (1 << 64))
    return x ^ _lsr(x, 31)


def _mix_int(x):
    return int(_mix(torch.tensor([x], dtype=torch.int64))[0])


def _bij(x, bits):
    """A bijection of [0, 2^bits) (odd products and xor-shifts), bits <= 63."""
    m, h = (1 << bits) - 1, bits // 2
    x = x & m
    x = x ^ (x >> h)
    x = (x * (0x9E3779B97F4A7C15 - (1 << 64))) & m
    x = x ^ (x >> h)
    x = (x * (0xC2B2AE3D27D4EB4F - (1 << 64))) & m
    return x ^ (x >> h)


def _narrow(x, bits):
    """int64 in [0, 2^32) or any -> the tensor type that carries `bits`-bit patterns."""
    return x if bits == 64 else ((x + (1 << 31)) % (1 << 32) - (1 << 31)).to(torch.int32)


def _uniform(n, bits, seed, start):
    """n distinct keys of the upper half of the key space, none a sentinel:
    index ranges that do not overlap give keys that do not meet."""
    off = _mix_int(seed * 2 + 1) & ((1 << (bits - 1)) - 1)
    i = torch.arange(start, start + n + 2, dtype=torch.int64, device=DEV)
    k = _bij(i + off, bits - 1)
    k = k[k < (1 << (bits - 1)) - 2][:n]
    return k | (-(1 << 63)) if bits == 64 else _narrow(k | (1 << 31), 32)


def _runs(n, bits, seed, gen):
    """n distinct keys of the lower half: runs of 8..512 consecutive ids, each
    run in a block of 1,024 of its own."""
    lens = torch.randint(8, 513, (n // 8 + 2,), generator=gen, device=DEV)
    ends = torch.cumsum(lens, 0)
    r = int(torch.searchsorted(ends, n).item()) + 1
    lens = lens[:r].clone()
    lens[-1] -= ends[r - 1] - n
    b = bits - 11
    starts = _bij(torch.arange(r, dtype=torch.int64, device=DEV) + (_mix_int(seed * 2) & ((1 << b) - 1)), b) << 10
    first = torch.cumsum(lens, 0) - lens
    k = torch.repeat_interleave(starts - first, lens) + torch.arange(n, dtype=torch.int64, device=DEV)
    return _narrow(k, bits)


def _gen(seed, salt=0):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1_000_003 + salt) & 0x7FFFFFFF)
    return g


def _keys(n, c, seed):
    """n distinct keys in random order."""
    g = _gen(seed, 1)
    if c["keys"] == "uniform":
        return _uniform(n, c["bits"], seed, 0)
    nr = n // 2
    k = torch.cat([_uniform(n - nr, c["bits"], seed, 0), _runs(nr, c["bits"], seed, g)])
    return k[torch.randperm(n, generator=g, device=DEV)]


def _absent(m, n, c, seed):
    """m keys that _keys(n, c, seed) does not hold."""
    return _uniform(m, c["bits"], seed, n + 8)


def _vals(keys, bits, seed):
    v = _mix(keys.to(torch.int64) ^ _mix_int(seed + 77))
    return v if bits == 64 else v.to(torch.int32)


def _shuffle(t, gen):
    return t[torch.randperm(t.shape[0], generator=gen, device=DEV)]


def _fill(c):
    return min((1 << c["sp"]) - 1, max(1, int(c["lf"] * (1 << c["sp"]))))


def _resident(c, k, v, **kw):
    hm = Hashmap(c["sp"], c["bits"], **kw)
    hm.insert(k, v, targetLF=1.0)
    return hm


def _map_inputs(c, seed):
    n = _fill(c)
    k = _keys(n, c, seed)
    return n, k, _vals(k, c["bits"], seed)


def _step_inputs(c, seed):
    n, k, v = _map_inputs(c, seed)
    if c["form"] == "index":
        v = torch.arange(n, dtype=_IDT[c["bits"]], device=DEV)
    a = _absent(n, n, c, seed)
    p = torch.randperm(2 * n, generator=_gen(seed, 2), device=DEV)
    q = torch.cat([k, a])[p]
    return k, v, q, p


def _query_inputs(c, seed):
    n, k, v = _map_inputs(c, seed)
    g = _gen(seed, 3)
    nh = min(c["n"], int(c["n"] * c["hits"]))
    at = torch.randint(0, n, (nh,), generator=g, device=DEV)
    a = _absent(c["n"] - nh, n, c, seed)
    p = torch.randperm(c["n"], generator=g, device=DEV)
    q = torch.cat([k[at], a])[p]
    return k, v, q, at, p


def _update_inputs(c, seed):
    n, k, v = _map_inputs(c, seed)
    u = k[torch.randperm(n, generator=_gen(seed, 4), device=DEV)[: c["n"]]].contiguous()
    return k, v, u, _vals(u, c["bits"], seed + 5)


def _churn_inputs(c, seed):
    n, k, v = _map_inputs(c, seed)
    m = max(1, int(c["frac"] * n))
    q = _shuffle(k, _gen(seed, 6))[: 2 * m].contiguous()
    return k, v, k[:m].contiguous(), v[:m].contiguous(), q


def _pairs_inputs(c, seed):
    g = _gen(seed, 7)
    lo, hi = (-(1 << 31), (1 << 31) - 3) if c["bits"] == 32 else (-(1 << 63), (1 << 63) - 3)
    return torch.randint(lo, hi, (c["n"], 2), dtype=_IDT[c["bits"]], generator=g, device=DEV)


def _rule(c):
    """The rule of a copy_if case: value < limit, or some low bits of the value equal to zero."""
    if c["rule"] == "lt":
        return pred(HN_PRED_LT, 1, 0, min((1 << c["bits"]) - 1, int(c["keep"] * (1 << c["bits"]))))
    return pred(HN_PRED_MASKEQ, 1, 3, 0)


def _kept(c, pairs, flags):
    if c["rule"] == "flags":
        return flags != 0
    if c["rule"] == "maskeq":
        return (pairs[:, 1] & 3) == 0
    top = -(1 << (c["bits"] - 1))
    limit = min((1 << c["bits"]) - 1, int(c["keep"] * (1 << c["bits"]))) + top
    return (pairs[:, 1] ^ top) < limit


def _scan_input(c, seed):
    return torch.randint(0, 1 << 20, (c["n"],), dtype=_IDT[c["bits"]], generator=_gen(seed, 8), device=DEV)


def _batch_inputs(c, seed, grid=200, sigma=20.0):
    """Per map: distinct grid cells around a random centre, values, queries
    (the cells and as many absent ids, shuffled) and the cells to erase."""
    g = _gen(seed, 9)
    sps = np.random.default_rng(c["maps"]).integers(c["sp_lo"], c["sp_hi"] + 1, size=c["maps"])
    n = torch.from_numpy((c["lf"] * (1 << sps)).astype(np.int64)).to(DEV)
    m = torch.repeat_interleave(torch.arange(c["maps"], device=DEV), 3 * n + 64)
    centre = torch.randint(0, grid, (c["maps"], 3), generator=g, device=DEV)
    d = torch.randn((m.numel(), 3), generator=g, device=DEV) * sigma
    xyz = (centre[m] + d.round().to(torch.int64)) % grid
    cell = xyz[:, 0] + grid * xyz[:, 1] + grid * grid * xyz[:, 2]
    u = torch.unique(m * (1 << 32) + cell)
    # n[m] cells of each map, in random order: sort by (map, random) and keep the first n[m]
    m = u >> 32
    order = torch.argsort(m * (1 << 40) + torch.randint(0, 1 << 40, u.shape, generator=g, device=DEV))
    u, m = u[order], m[order]
    have = torch.bincount(m, minlength=c["maps"])
    first = torch.cumsum(have, 0) - have
    rank = torch.arange(u.numel(), device=DEV) - first[m]
    u = u[rank < n[m]]
    take = torch.minimum(n, have)
    if c["bits"] == 64:  # wide ids: the cell and the map it lies in
        key, far = u, u + (1 << 24)
    else:
        key, far = u & 0xFFFFFFFF, (u & 0xFFFFFFFF) + (1 << 24)
    m = u >> 32
    qk = torch.cat([key, far])
    qm = torch.cat([m, m])
    order = torch.argsort(qm * (1 << 40) + torch.randint(0, 1 << 40, qm.shape, generator=g, device=DEV))
    qk = qk[order]
    nd = np.uint32 if c["bits"] == 32 else np.uint64
    take = take.cpu().numpy()

    def lists(t, lens):
        return np.split(t.cpu().numpy().astype(nd), np.cumsum(lens)[:-1])

    ins = lists(key, take)
    vals = lists(_mix(key) & 0x7FFFFFFF, take)
    qry = lists(qk, 2 * take)
    ers = [k[: int(c["frac"] * len(k))] for k in ins]
    return sps, ins, vals, qry, ers


def prepare(case, seed):
    c = dict(case)
    s = {"case": c}
    op, dt = c["op"], _IDT[c["bits"]]
    if op == "step":
        k, v, q, _ = _step_inputs(c, seed)
        if c["form"] == "pairs":
            k, v, q = torch.stack([k, v], 1), None, torch.stack([q, torch.zeros_like(q)], 1)
        s.update(k=k, v=v, q=q)
    elif op == "retrieve":
        k, v, q, _, _ = _query_inputs(c, seed)
        kw = {} if c["order"] == "home" else {"auto_reorder": 0, "auto_build": 0, "merge_min": 0}
        s.update(map=_resident(c, k, v, **kw), q=q, vals=torch.zeros(c["n"], dtype=dt, device=DEV),
                 hit=torch.zeros(c["n"], dtype=torch.uint8, device=DEV))
    elif op == "update":
        k, v, u, uv = _update_inputs(c, seed)
        s.update(map=_resident(c, k, v), u=u, uv=uv)
    elif op == "churn":
        k, v, e, ev, q = _churn_inputs(c, seed)
        s.update(map=_resident(c, k, v), e=e, ev=ev, q=q)
    elif op == "grow":
        k = _keys(c["n"], c, seed)
        v = _vals(k, c["bits"], seed)
        step = -(-c["n"] // c["batches"])
        s.update(parts=[(k[i : i + step], v[i : i + step]) for i in range(0, c["n"], step)])
    elif op == "extract":
        n, k, v = _map_inputs(c, seed)
        m = _resident(c, k, v)
        m.erase(k[: int(c["frac"] * n)])
        s.update(map=m)
    elif op == "copy_if":
        s.update(pairs=_pairs_inputs(c, seed), out=torch.zeros((c["n"], 2), dtype=dt, device=DEV),
                 out_keys=torch.zeros(c["n"], dtype=dt, device=DEV))
        if c["rule"] == "flags":
            s.update(flags=(torch.rand(c["n"], generator=_gen(seed, 10), device=DEV) < c["keep"]).to(torch.uint8))
    elif op == "scan":
        s.update(x=_scan_input(c, seed))
    else:
        s.update(batch=BatchedMaps(*_batch_inputs(c, seed), key_bits=c["bits"]))
    return s


# ------------------------------------------------------------------ one pass
def run(state):
    c, op = state["case"], state["case"]["op"]
    if op == "step":
        hm = Hashmap(c["sp"], c["bits"])
        if c["form"] == "pairs":
            hm.insert(state["k"], targetLF=1.0)
            q, h = hm.retrieve(state["q"])
            return {"vals": q[:, 1], "hit": h, "buckets": hm.buckets}
        if c["form"] == "index":
            hm.insertIndex(state["k"], targetLF=1.0)
        else:
            hm.insert(state["k"], state["v"], targetLF=1.0)
        _, v, h = hm.retrieve(state["q"])
        return {"vals": v, "hit": h, "buckets": hm.buckets}
    if op == "retrieve":
        _, v, h = state["map"].retrieve(state["q"], state["vals"], state["hit"])
        return {"vals": v, "hit": h}
    if op == "update":
        state["map"].insert(state["u"], state["uv"], targetLF=1.0)
        _, v, h = state["map"].retrieve(state["u"])
        return {"vals": v, "hit": h}
    if op == "churn":
        hm = state["map"]
        hm.erase(state["e"])
        hm.clean_tombstones()
        _, v, h = hm.retrieve(state["q"])
        hm.insert(state["e"], state["ev"], targetLF=1.0)
        return {"vals": v, "hit": h, "buckets": hm.buckets}
    if op == "grow":
        hm = Hashmap(c["sp"], c["bits"])
        for k, v in state["parts"]:
            hm.insert(k, v)
        return {"buckets": hm.buckets}
    if op == "extract":
        return {"pairs": state["map"].extractPattern(), "keys": state["map"].extractAllKeys()}
    if op == "copy_if":
        # into the program's own buffers, the count left on the device
        if c["rule"] == "flags":
            out, n = copy_if_flags(state["pairs"], state["flags"], out=state["out"], sync=False)
            return {"pairs": out, "count": n}
        out, n = copy_if_pairs(state["pairs"], _rule(c), c["bits"], out=state["out"], sync=False)
        keys, m = copy_keys_if_pairs(state["pairs"], _rule(c), c["bits"], out=state["out_keys"], sync=False)
        return {"pairs": out, "count": n, "keys": keys, "key_count": m}
    if op == "scan":
        return {"out": split_prefix_scan(state["x"])}
    b = state["batch"]
    b.init()
    b.run()
    return {"vals": b.qry_vals, "hit": b.qry_hit, "fill": b.infos[:, 1], "tombstones": b.infos[:, 3]}


# ------------------------------------------------------------------ what a pass cannot do without
def work(case):
    """Inputs read once, outputs written once; of a resident table what its
    lookups touch, at 64 bytes each, or the whole of it where that is less."""
    c, op, w = case, case["op"], case["bits"] // 8
    if op in ("step", "retrieve", "update", "churn", "extract"):
        N, n = 1 << c["sp"], _fill(c)
        T = N * 2 * w
    if op == "step":
        b = n * (w if c["form"] == "index" else 2 * w) + T + min(T, 2 * n * 64) + 2 * n * (2 * w + 1)
    elif op == "retrieve":
        b = min(T, c["n"] * 64) + c["n"] * (2 * w + 1)
    elif op == "update":
        b = 2 * min(T, c["n"] * 64) + c["n"] * 2 * w + c["n"] * (2 * w + 1)
    elif op == "churn":
        m = max(1, int(c["frac"] * n))
        # erase: keys and their slots; clean: the table read, what moves written (about half of it);
        # retrieve: 2m queries; insert: the pairs and the table's new image
        b = m * w + min(T, m * 64) + T + T // 2 + min(T, 2 * m * 64) + 2 * m * (2 * w + 1) + m * 2 * w + 2 * T
    elif op == "grow":
        b, total = 0, 0
        step = -(-c["n"] // c["batches"])
        for i in range(0, c["n"], step):
            m = min(step, c["n"] - i)
            sp = max(c["sp"], math.ceil(math.log2(2 * (total + m))))
            b += m * 2 * w + total * 2 * w + (1 << sp) * 2 * w
            total += m
    elif op == "extract":
        live = n - int(c["frac"] * n)
        b = 2 * T + live * 3 * w
    elif op == "copy_if":
        keep = 0.25 if c["rule"] == "maskeq" else c["keep"]
        b = c["n"] * (2 * w + 1) + int(c["n"] * keep) * 2 * w
        if c["rule"] != "flags":
            b += c["n"] * (2 * w - 1) + int(c["n"] * keep) * w
    elif op == "scan":
        b = 2 * c["n"] * w
    else:
        spread = c["sp_hi"] - c["sp_lo"] + 1
        slots = c["maps"] * sum(1 << p for p in range(c["sp_lo"], c["sp_hi"] + 1)) / spread
        n = slots * c["lf"]
        # fresh tables written, pairs in, queries answered, keys erased, the cleaned tables written
        b = 2 * slots * 2 * w + n * 2 * w + 2 * n * (2 * w + 1) + c["frac"] * n * w
    return {"bytes": int(b), "flops": 0}


# ------------------------------------------------------------------ the same answers in plain torch
def exact(case, seed):
    """What ``run`` returns, from the inputs alone: values and hit flags of the
    lookups, selected pairs, sums.  Bucket arrays, extractions (their order is
    the table's) and batches have none."""
    c, op = case, case["op"]
    if op == "step":
        k, v, q, p = _step_inputs(c, seed)
        n = k.numel()
        both = torch.cat([v, torch.zeros_like(v)])
        return {"vals": both[p], "hit": (p < n).to(torch.uint8), "buckets": None}
    if op == "retrieve":
        k, v, q, at, p = _query_inputs(c, seed)
        nh = at.numel()
        both = torch.cat([v[at], torch.zeros(c["n"] - nh, dtype=v.dtype, device=DEV)])
        return {"vals": both[p], "hit": (p < nh).to(torch.uint8)}
    if op == "update":
        _, _, u, uv = _update_inputs(c, seed)
        return {"vals": uv, "hit": torch.ones(u.numel(), dtype=torch.uint8, device=DEV)}
    if op == "copy_if":
        pairs = _pairs_inputs(c, seed)
        flags = None
        if c["rule"] == "flags":
            flags = (torch.rand(c["n"], generator=_gen(seed, 10), device=DEV) < c["keep"]).to(torch.uint8)
        got = pairs[_kept(c, pairs, flags)]
        m = torch.tensor([got.shape[0]], device=DEV)
        out = torch.zeros_like(pairs)
        out[: got.shape[0]] = got
        r = {"pairs": out, "count": m}
        return r if c["rule"] == "flags" else dict(r, keys=out[:, 0].contiguous(), key_count=m)
    if op == "scan":
        x = _scan_input(c, seed).to(torch.int64)
        return {"out": _narrow((torch.cumsum(x, 0) - x) & ((1 << 32) - 1), 32) if c["bits"] == 32 else
                torch.cumsum(x, 0) - x}
    return None
