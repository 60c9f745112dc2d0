"""Performance cases of the dictionaries: what a program has them do.

Every case goes through the Python binding's public calls (GPULSMOpt,
FlixIndex, Server) on tensors that are on the GPU already.  The sizes are
those of the workloads this repository measures and tests (16 batches of 2^16
keys with 2^20 lookups; batches of 2^20 keys with a tenth tombstones; clustered
64-bit FliX keys; uneven Zipf request streams), scaled so that a pass takes
at most tens of milliseconds, plus small calls and odd sizes.

Kinds of case:

  lookup   point lookups against a dictionary that was filled before
  session  an empty dictionary takes update batches, then answers point
           lookups, range counts, range sums and successors (each optional)
  reads    range sums, range counts and successors against a dictionary of
           several runs, some of them tombstones
  load     a bulk build from unsorted keys, then the sorted export
  serve    requests of uneven sizes through the batching engine
  fbuild   a FliX index from unsorted keys, then lookups and successors
  fupdate  a FliX index that is in use takes a batch of inserts, answers
           lookups and range enumerations, and takes a batch of removes

Outputs are whole-number tensors, whole.  A pass leaves the contents that it
found (an update's keys are written again with the same values, or removed
again), so passes repeat.
"""

import math

import torch

import __graft_entry__ as entry

pkg = entry.load_package()

DEV = "cuda:0"


# ------------------------------------------------------------------- cases
def _case(name, kind, **kw):
    c = {"name": name, "kind": kind, "key_bytes": 4, "dist": "uniform"}
    c.update(kw)
    return c


def listed():
    return [
        # one small request against a small dictionary: latency and launches
        _case("lookup_small", "lookup", rows=1 << 20, batch=1 << 16,
              queries=1000, found=True, erase=0.0),
        # the query side of a large dictionary that takes updates (rows of
        # several sizes, tombstones on top), more queries than rows touched
        _case("lookup_large", "lookup", rows=(1 << 25) + 12345,
              batch=1 << 20, queries=1 << 23, found=False, erase=0.1),
        # many small updates, each followed by a few reads
        _case("session_trickle", "session", batches=24, batch=700,
              queries=700, counts=100, sums=0, succ=0, each=True, found=True,
              erase=0.2),
        # 2^20 keys in 16 batches, then reads of every type
        _case("session_medium", "session", batches=16, batch=1 << 16,
              queries=1 << 20, counts=1 << 14, sums=3000, succ=50000,
              each=False, found=False, erase=0.0, wlo=10, whi=16),
        # 2^26 updates in batches of 2^20, a tenth of them tombstones
        _case("session_large", "session", batches=64, batch=1 << 20,
              queries=1 << 25, counts=1 << 20, sums=0, succ=0, each=False,
              found=False, erase=0.1, wlo=4, whi=20),
        # 64-bit keys and values, odd batches
        _case("session_u64", "session", key_bytes=8, batches=12,
              batch=700001, queries=3000001, counts=40001, sums=20011,
              succ=100003, each=False, found=True, erase=0.1, wlo=38, whi=48),
        # analytic reads over several runs
        _case("reads_runs", "reads", rows=6000000, batch=1 << 19,
              counts=12000, sums=12000, succ=1 << 20, erase=0.1,
              wlo=4, whi=24),
        # a table loaded at once and written out in key order
        _case("load_u32", "load", rows=15000001),
        _case("load_u64", "load", key_bytes=8, rows=3000017,
              dist="clustered"),
        # uneven requests of skewed keys through the batching engine
        _case("serve_mixed", "serve", rows=1 << 22, requests=200, smin=32,
              smax=1 << 15, dist="zipf"),
        # 32-bit index, build and ordered reads
        _case("flix_build_u32", "fbuild", value_bytes=4, rows=1 << 23,
              queries=1 << 24, succ=1 << 20, sorted=True, slots=32, fill=50),
        # 64-bit clustered index in use: any-order updates and lookups,
        # range enumerations
        _case("flix_update_u64", "fupdate", key_bytes=8, value_bytes=8,
              rows=1 << 23, inserts=1500003, queries=1 << 21, ranges=1 << 15,
              sorted=False, slots=64, fill=75, dist="clustered"),
    ]


def _size(rng, lo, hi):
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(lo, min(hi, n))


def draw(rng):
    kind = rng.choice(["lookup", "session", "session", "reads", "load",
                       "serve", "fbuild", "fupdate", "fupdate"])
    kb = rng.choice([4, 8])
    dist = rng.choice(["uniform", "full", "clustered", "zipf"])
    erase = rng.choice([0.0, 0.1, 0.3])
    c = {"kind": kind, "key_bytes": kb, "dist": dist}
    # the key space is 2^31 (or, 64-bit keys but the skewed ones, 2^62) wide
    wl = rng.randint(4, 16) + (32 if kb == 8 and dist != "zipf" else 0)
    if kind == "lookup":
        rows = _size(rng, 1 << 14, 1 << 24)
        c.update(rows=rows, batch=_size(rng, max(1 << 10, rows >> 6), 1 << 20),
                 queries=_size(rng, 100, 1 << 22), found=rng.random() < 0.5,
                 erase=erase)
    elif kind == "session":
        batch = _size(rng, 300, 1 << 20)
        c.update(batches=rng.randint(1, 20), batch=batch,
                 queries=_size(rng, 300, 1 << 21), each=batch < 5000,
                 counts=_size(rng, 50, 1 << 16), sums=_size(rng, 50, 1 << 13),
                 succ=_size(rng, 50, 1 << 18), found=rng.random() < 0.5,
                 erase=erase, wlo=wl - 4, whi=wl)
    elif kind == "reads":
        rows = _size(rng, 1 << 16, 1 << 22)
        c.update(rows=rows, batch=_size(rng, rows >> 5, min(rows, 1 << 20)),
                 counts=_size(rng, 50, 1 << 15), sums=_size(rng, 50, 1 << 14),
                 succ=_size(rng, 50, 1 << 20), erase=erase, wlo=4, whi=wl + 4)
    elif kind == "load":
        c.update(rows=_size(rng, 1 << 12, 1 << 23))
    elif kind == "serve":
        c.update(rows=_size(rng, 1 << 16, 1 << 21),
                 requests=rng.randint(20, 150), smin=32,
                 smax=_size(rng, 1 << 10, 1 << 15))
    elif kind == "fbuild":
        c.update(value_bytes=rng.choice([4, 8]), rows=_size(rng, 1 << 12,
                                                             1 << 22),
                 queries=_size(rng, 300, 1 << 22), succ=_size(rng, 300,
                                                              1 << 18),
                 sorted=rng.random() < 0.5, slots=rng.choice([16, 32, 64]),
                 fill=rng.choice([50, 75]))
    else:
        rows = _size(rng, 1 << 14, 1 << 22)
        c.update(value_bytes=rng.choice([4, 8]), rows=rows,
                 inserts=_size(rng, 300, rows // 2), queries=_size(
                     rng, 300, 1 << 20), ranges=_size(rng, 50, 1 << 13),
                 sorted=rng.random() < 0.5, slots=rng.choice([16, 32, 64]),
                 fill=rng.choice([50, 75]))
    return c


# ------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _rand(g, n, lo, hi):
    return torch.randint(lo, hi, (n,), generator=g, device=DEV,
                         dtype=torch.int64)


def _cut(x, kb):
    """int64 tensor of key values -> the key width's tensor (same bits)."""
    return x.to(torch.int32) if kb == 4 else x


def _keys(g, n, kb, dist):
    """n keys as int64: 31- or 62-bit uniform, uniform over the whole
    width, runs of up to 4096 consecutive keys at random places in a random
    order, or skewed ranks (density 1/rank) scattered over 30 bits.  None is
    0 or 1 or one of the four largest (reserved by FliX)."""
    if dist == "full":
        if kb == 8:
            x = _rand(g, n, -(1 << 62), 1 << 62) * 2 + _rand(g, n, 0, 2)
        else:
            x = _rand(g, n, -(1 << 31), 1 << 31)
        return torch.where((x >= 0) & (x < 2) | (x < 0) & (x >= -4),
                           torch.full_like(x, 77), x)
    if dist == "clustered":
        runs = max(1, n >> 11)
        top = (1 << 31) - 5000 if kb == 4 else (1 << 62)
        starts = _rand(g, runs, 2, top)
        return starts[_rand(g, n, 0, runs)] + _rand(g, n, 0, 4096)
    if dist == "zipf":
        u = torch.rand(n, generator=g, device=DEV, dtype=torch.float64)
        rank = torch.exp(u * math.log(1 << 30)).to(torch.int64)
        return ((rank * 0x9E3779B1 + 0x5BD1E995) & ((1 << 30) - 1)) + 2
    return _rand(g, n, 2, 1 << (31 if kb == 4 else 62))


def _values(g, n, vb):
    """Values over the whole width: for the ranges' sums to wrap around."""
    if vb == 4:
        return _rand(g, n, -(1 << 31), 1 << 31).to(torch.int32)
    return _rand(g, n, -(1 << 62), 1 << 62)


def _empty(n, nbytes):
    dt = {1: torch.uint8, 4: torch.int32, 8: torch.int64}[nbytes]
    return torch.empty(n, dtype=dt, device=DEV)


def _batches(g, c, n_total):
    """Update batches: (keys, values, erase flags); an erased key is one of
    the earlier batches' keys."""
    kb = c["key_bytes"]
    keys = _keys(g, n_total, kb, c["dist"])
    vals = _values(g, n_total, kb)
    flags = torch.zeros(n_total, dtype=torch.uint8, device=DEV)
    b = c["batch"]
    if c["erase"] > 0 and n_total > b:
        hit = torch.rand(n_total, generator=g, device=DEV) < c["erase"]
        hit[:b] = False
        at = torch.arange(n_total, device=DEV)
        pick = (torch.rand(n_total, generator=g, device=DEV,
                           dtype=torch.float64) *
                (at // b * b).clamp(min=1)).to(torch.int64)
        keys = torch.where(hit, keys[pick], keys)
        flags = hit.to(torch.uint8)
    k = _cut(keys, kb)
    out = []
    for a in range(0, n_total, b):
        z = min(n_total, a + b)
        out.append((k[a:z].clone(), vals[a:z].clone(), flags[a:z].clone()))
    return keys, out


def _queries(g, c, n, keys, hit=0.7):
    """A share of stored keys, the rest from the same distribution."""
    q = _keys(g, n, c["key_bytes"], c["dist"])
    take = torch.rand(n, generator=g, device=DEV) < hit
    q = torch.where(take, keys[_rand(g, n, 0, keys.numel())], q)
    return _cut(q, c["key_bytes"])


def _ranges(g, c, n, keys):
    """lo at or near a stored key, widths log-uniform in 2^[wlo, whi]."""
    kb = c["key_bytes"]
    a, z = c.get("wlo", 4), c.get("whi", 16)
    lo = keys[_rand(g, n, 0, keys.numel())]
    u = torch.rand(n, generator=g, device=DEV, dtype=torch.float64)
    w = torch.exp2(a + u * (z - a)).to(torch.int64)
    if kb == 4:  # unsigned 32-bit bounds without a wrap-around
        lo = lo & 0xFFFFFFFF
        hi = (lo + w - 1).clamp(max=0xFFFFFFFF)
        return (lo - ((lo >> 31) << 32)).to(torch.int32), \
            (hi - ((hi >> 31) << 32)).to(torch.int32)
    hi = lo + w - 1
    return lo, torch.where((lo < 0) & (hi >= 0), torch.full_like(hi, -1), hi)


def _unsigned_order(x):
    """Sort key of a tensor that holds unsigned bits."""
    return x ^ (-(1 << 31) if x.dtype == torch.int32 else -(1 << 63))


def _sorted(x):
    return _unsigned_order(torch.sort(_unsigned_order(x))[0])


# ----------------------------------------------------------------- prepare
def prepare(case, seed):
    g = _gen(seed)
    s = {"lookup": _prep_lookup, "session": _prep_session,
         "reads": _prep_reads, "load": _prep_load, "serve": _prep_serve,
         "fbuild": _prep_fbuild, "fupdate": _prep_fupdate}[case["kind"]](
             g, case)
    s["kind"] = case["kind"]
    torch.cuda.synchronize()
    return s


def _filled(g, c):
    keys, batches = _batches(g, c, c["rows"])
    d = pkg.GPULSMOpt(max_elements=2 * c["rows"], batch_capacity=1 << 20,
                      key_bytes=c["key_bytes"])
    for k, v, e in batches:
        d.apply_mixed(k, v, e)
    return d, keys


def _prep_lookup(g, c):
    d, keys = _filled(g, c)
    n = c["queries"]
    return {"d": d, "q": _queries(g, c, n, keys),
            "out": _empty(n, c["key_bytes"]),
            "found": _empty(n, 1) if c["found"] else None}


def _prep_session(g, c):
    kb = c["key_bytes"]
    keys, batches = _batches(g, c, c["batches"] * c["batch"])
    d = pkg.GPULSMOpt(max_elements=2 * keys.numel(), batch_capacity=1 << 20,
                      key_bytes=kb)
    rounds = c["batches"] if c["each"] else 1
    outs = {"out": _empty(rounds * c["queries"], kb),
            "cnt": _empty(rounds * c["counts"], kb),
            "sum": _empty(rounds * c["sums"], kb),
            "sk": _empty(rounds * c["succ"], kb)}
    if c["found"]:
        outs["found"] = _empty(rounds * c["queries"], 1)
    s = {"d": d, "batches": batches, "each": c["each"], "erase": c["erase"],
         "reads": [], "outs": [t for t in outs.values() if t.numel()]}

    def part(name, i, n):
        return outs[name][i * n:(i + 1) * n]

    for i in range(rounds):
        r = {}
        if c["queries"]:
            r["q"] = _queries(g, c, c["queries"], keys)
            r["out"] = part("out", i, c["queries"])
            r["found"] = part("found", i, c["queries"]) if c["found"] else None
        if c["counts"]:
            r["clo"], r["chi"] = _ranges(g, c, c["counts"], keys)
            r["cnt"] = part("cnt", i, c["counts"])
        if c["sums"]:
            r["slo"], r["shi"] = _ranges(g, c, c["sums"], keys)
            r["sum"] = part("sum", i, c["sums"])
        if c["succ"]:
            r["sq"] = _queries(g, c, c["succ"], keys, 0.3)
            r["sk"] = part("sk", i, c["succ"])
        s["reads"].append(r)
    return s


def _prep_reads(g, c):
    kb = c["key_bytes"]
    d, keys = _filled(g, c)
    s = {"d": d}
    s["clo"], s["chi"] = _ranges(g, c, c["counts"], keys)
    s["slo"], s["shi"] = _ranges(g, c, c["sums"], keys)
    s["sq"] = _queries(g, c, c["succ"], keys, 0.3)
    s["cnt"], s["sum"] = _empty(c["counts"], kb), _empty(c["sums"], kb)
    s["sk"] = _empty(c["succ"], kb)
    return s


def _prep_load(g, c):
    kb, n = c["key_bytes"], c["rows"]
    keys = _keys(g, n, kb, c["dist"])
    return {"d": pkg.GPULSMOpt(max_elements=n, batch_capacity=1 << 20,
                               key_bytes=kb),
            "k": _cut(keys, kb), "v": _values(g, n, kb),
            # repeated keys leave the end of the export as it is
            "ok": torch.zeros_like(_empty(n, kb)),
            "ov": torch.zeros_like(_empty(n, kb))}


def _prep_serve(g, c):
    kb, n = c["key_bytes"], c["requests"]
    srv = pkg.Server(max_elements=1 << 24, batch_capacity=1 << 20,
                     key_bytes=kb)
    # a key's value is a function of the key, and the erased keys are odd
    # while the others are even: how requests are grouped into steps then
    # changes no answer

    def key(m):
        return _keys(g, m, kb, c["dist"]) & ~1 | 2

    def value(k):
        return _cut((k * 0x2545F491 + 12345) & 0x7FFFFFFF, kb)

    base = key(c["rows"])
    u = torch.rand(2 * n, generator=torch.Generator().manual_seed(
        int(_rand(g, 1, 0, 1 << 30).item()))).tolist()
    sizes = [int(c["smin"] * math.exp(x * math.log(c["smax"] / c["smin"])))
             for x in u[:n]]
    out = torch.zeros_like(_empty(n * c["smax"], kb))
    reqs = []
    for i in range(n):
        m, at = sizes[i], i * c["smax"]
        what = u[n + i]
        if what < 0.4:
            k = base[_rand(g, m, 0, base.numel())]
            reqs.append((srv.INSERT, _cut(k, kb), value(k), None))
        elif what < 0.5:
            reqs.append((srv.ERASE, _cut(key(m) | 1, kb), None, None))
        elif what < 0.9:
            take = torch.rand(m, generator=g, device=DEV) < 0.7
            q = torch.where(take, base[_rand(g, m, 0, base.numel())], key(m))
            reqs.append((srv.LOOKUP, _cut(q, kb), None, out[at:at + m]))
        else:
            lo, hi = _ranges(g, c, m, base)
            reqs.append((srv.RANGE_COUNT, lo, hi, out[at:at + m]))
    torch.cuda.synchronize()
    for a in range(0, base.numel(), 1 << 20):
        k = base[a:a + (1 << 20)]
        kk, vv = _cut(k, kb).clone(), value(k).clone()
        torch.cuda.synchronize()
        srv.wait(srv.submit(srv.INSERT, kk, vv))
    return {"srv": srv, "reqs": reqs, "out": out}


def _prep_fbuild(g, c):
    kb, vb = c["key_bytes"], c["value_bytes"]
    keys = _keys(g, c["rows"], kb, c["dist"])
    q = _queries(g, c, c["queries"], keys)
    return {"f": pkg.FlixIndex(kb, vb, node_slots=c["slots"],
                               fill_percent=c["fill"]),
            "k": _cut(keys, kb), "q": _sorted(q) if c["sorted"] else q,
            "sorted": c["sorted"],
            "sq": _sorted(_queries(g, c, c["succ"], keys, 0.3)),
            "out": _empty(c["queries"], vb), "sk": _empty(c["succ"], kb)}


def _prep_fupdate(g, c):
    kb, vb, n = c["key_bytes"], c["value_bytes"], c["inserts"]
    built = torch.unique(_keys(g, c["rows"], kb, c["dist"]))
    # new keys near the built ones and anywhere; the built ones are left out,
    # so that the removes restore the contents
    near = built[_rand(g, n, 0, built.numel())] + _rand(g, n, 1, 64)
    ins = torch.where(torch.rand(n, generator=g, device=DEV) < 0.5, near,
                      _keys(g, n, kb, c["dist"]))
    at = torch.searchsorted(built, ins).clamp(max=built.numel() - 1)
    ins = ins[(built[at] != ins) & ((ins > 1) | (ins < -4))]
    if kb == 4:
        ins = ins[(ins < (1 << 31)) & (ins >= -(1 << 31))]
    n = ins.numel()
    rem = ins[torch.randperm(n, generator=g, device=DEV)]
    k, r = _cut(ins, kb), _cut(rem, kb)
    f = pkg.FlixIndex(kb, vb, node_slots=c["slots"], fill_percent=c["fill"])
    f.build_bucket_layer_only(_cut(built, kb), max_size=2 * (built.numel() + n))
    q = _queries(g, c, c["queries"], torch.cat([built, ins]))
    # enumerations of 16 to 1024 neighbouring built keys
    m = c["ranges"]
    order = _sorted(_cut(built, kb))
    i = _rand(g, m, 0, order.numel())
    u = torch.rand(m, generator=g, device=DEV, dtype=torch.float64)
    w = torch.exp2(4 + 6 * u).to(torch.int64)
    j = (i + w).clamp(max=order.numel() - 1)
    lo, hi = order[i].clone(), order[j].clone()
    # at most 1024 built pairs each and 242 at the mean, the new keys between
    # them on top
    every = _unsigned_order(_sorted(torch.unique(
        torch.cat([_cut(built, kb), k]))))
    pairs = int((torch.searchsorted(every, _unsigned_order(hi), right=True) -
                 torch.searchsorted(every, _unsigned_order(lo))).sum().item())
    room = max(m * 512 + (1 << 16), pairs)
    return {"f": f, "k": _sorted(k) if c["sorted"] else k,
            "v": _values(g, n, vb), "r": _sorted(r) if c["sorted"] else r,
            "q": _sorted(q) if c["sorted"] else q, "sorted": c["sorted"],
            "lo": lo, "hi": hi, "out": _empty(c["queries"], vb),
            "offs": _empty(m + 1, 8),
            "pk": torch.zeros_like(_empty(room, kb)),
            "pv": torch.zeros_like(_empty(room, vb))}


# --------------------------------------------------------------------- run
def run(s):
    kind = s["kind"]
    if kind == "lookup":
        s["d"].lookup(s["q"], s["out"], s["found"])
        return [t for t in (s["out"], s["found"]) if t is not None]
    if kind == "session":
        return _run_session(s)
    if kind == "reads":
        d = s["d"]
        d.range_count(s["clo"], s["chi"], s["cnt"])
        d.range(s["slo"], s["shi"], s["sum"])
        d.successor(s["sq"], s["sk"])
        return [s["cnt"], s["sum"], s["sk"]]
    if kind == "load":
        d = s["d"]
        d.bulk_build(s["k"], s["v"])
        d.dump_sorted(s["ok"], s["ov"], s["ok"].numel())
        return [s["ok"], s["ov"]]
    if kind == "serve":
        srv = s["srv"]
        tickets = [srv.submit(op, a, b, out) for op, a, b, out in s["reqs"]]
        for t in tickets:
            srv.wait(t)
        return s["out"]
    f = s["f"]
    if kind == "fbuild":
        f.build_bucket_layer_only(s["k"])
        (f.lookups_ordered if s["sorted"] else f.lookup)(s["q"], s["out"])
        f.lookups_successor(s["sq"], s["sk"])
        return [s["out"], s["sk"]]
    f.insert(s["k"], s["v"])
    (f.lookups_ordered if s["sorted"] else f.lookup)(s["q"], s["out"])
    f.range(s["lo"], s["hi"], s["offs"])
    f.range(s["lo"], s["hi"], s["offs"], s["pk"], s["pv"])
    f.remove(s["r"], assume_sorted=s["sorted"])
    return [s["out"], s["offs"], s["pk"], s["pv"]]


def _run_session(s):
    d = s["d"]
    d.clear()
    for i, (k, v, e) in enumerate(s["batches"]):
        if s["erase"]:
            d.apply_mixed(k, v, e)
        else:
            d.insert(k, v)
        if s["each"]:
            _read(d, s["reads"][i])
    if not s["each"]:
        _read(d, s["reads"][0])
    return s["outs"]


def _read(d, r):
    if "q" in r:
        d.lookup(r["q"], r["out"], r["found"])
    if "clo" in r:
        d.range_count(r["clo"], r["chi"], r["cnt"])
    if "slo" in r:
        d.range(r["slo"], r["shi"], r["sum"])
    if "sq" in r:
        d.successor(r["sq"], r["sk"])


# -------------------------------------------------------------------- work
def work(case):
    """Bytes of one pass: each input read once, each output written once,
    and of the stored rows one per query (at most all of them)."""
    c = case
    kb = c["key_bytes"]
    row = 2 * kb
    kind = c["kind"]

    def reads(rows):
        b = 0
        q = c.get("queries", 0)
        b += q * (kb + kb + (1 if c.get("found") else 0)) + min(q, rows) * row
        b += c.get("counts", 0) * 3 * kb + min(2 * c.get("counts", 0),
                                               rows) * row
        b += c.get("sums", 0) * 3 * kb + min(2 * c.get("sums", 0), rows) * row
        b += c.get("succ", 0) * 2 * kb + min(c.get("succ", 0), rows) * row
        return b

    if kind in ("lookup", "reads"):
        b = reads(c["rows"])
    elif kind == "session":
        n = c["batches"] * c["batch"]
        b = n * (row + (1 if c["erase"] else 0)) + n * row
        b += reads(n) * (c["batches"] if c["each"] else 1)
    elif kind == "load":
        b = 2 * c["rows"] * row  # the batch in, the export out
    elif kind == "serve":
        mean = (c["smax"] - c["smin"]) / math.log(c["smax"] / c["smin"])
        b = int(c["requests"] * mean * (0.5 * 2 * row + 0.4 * 2 * row +
                                        0.1 * (3 * kb + 2 * row)))
    elif kind == "fbuild":
        pair = kb + c["value_bytes"]
        b = c["rows"] * (kb + pair)
        b += c["queries"] * pair + min(c["queries"], c["rows"]) * pair
        b += c["succ"] * 2 * kb + min(c["succ"], c["rows"]) * kb
    else:
        pair = kb + c["value_bytes"]
        b = c["inserts"] * (2 * pair + kb + pair)
        b += c["queries"] * 2 * pair
        b += c["ranges"] * (2 * kb + 8 + 173 * 2 * pair)
    return {"bytes": int(b), "flops": 0}
