"""The calls whose time matters to a user of the filter, as cases: building a
table, looking keys up, a window of keys that come and go, counting with
repeats, many small filters at once, a served mix of requests, dumping a
table and merging tables.  Sizes are those of the benchmark configurations
(2^16 .. 2^28 slots, loads 0.45 .. 0.95) and of the tests, odd ones included.

Every pass ends in the table's whole 81-byte-block image where it changed
the table (what a program writes to a file or sends to a replica), besides
the key arrays that the calls leave sorted and the counts.  Inputs that a
call overwrites are copied from the program's own array first.  All outputs
are whole numbers and bytes, so no case has an approximate value: exact()
gives None.
"""
import math

import torch

from cqf_amd import gqf, workloads

BLOCK = 81                 # bytes of one 64-slot block in the image
BATCH = 1 << 24            # keys per call when a large table is filled


class State(dict):
    """The tensors and filters of one case; closes the filters when dropped."""

    def __del__(self):
        if "group" in self:
            self["group"].close()
        for f in self.get("filters", ()):
            f.close()


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # one request's lookups in a small resident table: a launch and little else
        {"name": "get_q20_1000", "kind": "get", "nbits": 20, "load": 0.9, "n": 1000, "present": 0.5},
        # a served filter's ordinary update: a few thousand keys in, looked up, and out again
        {"name": "window_q24_5000", "kind": "window", "nbits": 24, "load": 0.85, "n": 5000},
        # the reference's smallest benchmark table, built with one call
        {"name": "fill_q20", "kind": "fill", "nbits": 20, "load": 0.9, "batch": 943718},
        # the load curve: a table filled in twentieths up to 95%, where clusters are long
        {"name": "fill_q26_steps", "kind": "fill", "nbits": 26, "load": 0.95, "batch": (1 << 26) // 20},
        # the headline table: 2^28 slots filled to 90% in calls of 2^24 keys
        {"name": "fill_q28", "kind": "fill", "nbits": 28, "load": 0.9, "batch": BATCH},
        # the headline lookups, present and absent keys mixed
        {"name": "get_q28", "kind": "get", "nbits": 28, "load": 0.9, "n": (1 << 26) + 13, "present": 0.5},
        # a sliding window over the headline table: a batch in, looked up, and out again
        {"name": "window_q28", "kind": "window", "nbits": 28, "load": 0.85, "n": 7549747},
        # counting a stream with heavy repeats (Zipf 1.5)
        {"name": "count_q26", "kind": "count", "nbits": 26, "ids": 1 << 23, "n": (1 << 26) + 12345},
        # one small filter per sample (k-mers), all samples inserted and looked up together
        {"name": "group_32", "kind": "group", "filters": 32, "q_lo": 16, "q_hi": 24},
        # one served batch of get / insert / delete requests in arrival order, and one that undoes it
        {"name": "requests_q24", "kind": "requests", "nbits": 24, "load": 0.8, "requests": 120, "median": 14},
        # a table read out whole: keys and counts, statistics, cluster lengths
        {"name": "dump_q26", "kind": "dump", "nbits": 26, "load": 0.9, "repeat": 0.1},
        # two tables counted apart and added up
        {"name": "merge_q25", "kind": "merge", "nbits": 25, "load": 0.42, "shared": 0.1},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["get", "window", "fill", "count", "group", "requests", "dump", "merge"])
    c = {"kind": kind}
    if kind == "group":
        c["filters"] = rng.randint(8, 40)
        c["q_lo"] = rng.randint(16, 20)
        c["q_hi"] = rng.randint(21, 24)
        return c
    if kind == "count":
        c["n"] = _log(rng, 1 << 18, 1 << 26) | 1
        c["ids"] = max(1000, int(c["n"] / _log(rng, 2, 64)))
        c["nbits"] = max(18, (2 * c["ids"]).bit_length())
        return c
    c["nbits"] = q = rng.randint(18, 28) if kind in ("get", "window") else rng.randint(18, 27)
    if kind == "requests":
        c["nbits"] = q = rng.randint(20, 26)
    if kind == "merge":
        c["nbits"] = rng.randint(18, 25)
        c["load"], c["shared"] = round(rng.uniform(0.2, 0.45), 3), round(rng.uniform(0.0, 0.5), 3)
        return c
    c["load"] = round(rng.uniform(0.5, 0.95 if kind in ("fill", "get", "dump") else 0.88), 3)
    if kind == "get":
        c["n"], c["present"] = _log(rng, 1000, 1 << 26), rng.choice([0.0, 0.5, 1.0])
    elif kind == "window":
        c["n"] = _log(rng, 500, max(1000, (1 << q) // 32))
    elif kind == "fill":
        n = int(c["load"] * (1 << q))
        c["batch"] = min(BATCH, n, _log(rng, max(50000, n // 24), n))
    elif kind == "requests":
        c["requests"], c["median"] = rng.randint(10, 200), rng.randint(10, 14)
    else:
        c["repeat"] = round(rng.uniform(0.0, 0.3), 3)
    return c


# ------------------------------------------------------- inputs, by the seed

def _keys(seed, n, stream=0):
    """n uniform 64-bit keys; streams of one seed do not meet."""
    return workloads.splitmix64(seed * 1000003 + 17, n, skip=stream << 40, device="cuda")


def _filled(nbits, keys, batch=BATCH):
    """A table that holds `keys`, with workspace for calls of `batch` keys."""
    f = gqf.GQF(nbits)
    f.reserve(max(batch, min(BATCH, keys.numel())))
    buf = keys.clone()
    for i in range(0, buf.numel(), BATCH):
        f.bulk_insert(buf[i:i + BATCH])
    return f


def _image(f):
    return torch.empty(f.nbytes, dtype=torch.uint8, device="cuda")


def _pick(seed, a, b, share):
    """a's value with probability `share`, else b's, place by place."""
    u = workloads.splitmix64(seed * 1000003 + 29, a.numel(), device="cuda")
    return torch.where((u >> 11 & ((1 << 30) - 1)) < int(share * (1 << 30)), a, b)


def _items(case):
    return int(case["load"] * (1 << case["nbits"]) * (1 - case["repeat"]))


def _group_sizes(case):
    return workloads.kmer_filter_params(case["filters"], 5, q_lo=case["q_lo"], q_hi=case["q_hi"])


def prepare(case, seed):
    s = State(case)
    kind = case["kind"]
    if kind == "group":
        # the filters' sizes come from the case, the reads from the seed
        params = _group_sizes(case)
        keys = torch.cat([workloads.kmers(n, genome, (seed + 1) * 1000003 + i, device="cuda")
                          for i, (_, _, n, genome) in enumerate(params)])
        offsets = [0]
        for p in params:
            offsets.append(offsets[-1] + p[2])
        s["filters"] = [gqf.GQF(q) for q, _, _, _ in params]
        s["group"] = gqf.GQFGroup(s["filters"])
        s["keys"], s["buf"], s["offsets"] = keys, torch.empty_like(keys), offsets
        s["counts"], s["images"] = torch.empty_like(keys), [_image(f) for f in s["filters"]]
        return s
    if kind == "count":
        _, draws, _ = workloads.zipf_workload(case["ids"], case["n"], 1.5, seed + 1,
                                              distinct_bits=case["nbits"] + 8, device="cuda")
        f = gqf.GQF(case["nbits"])
        f.reserve(case["n"])
        s["filters"], s["keys"], s["buf"], s["image"] = [f], draws, torch.empty_like(draws), _image(f)
        return s
    size = 1 << case["nbits"]
    if kind == "fill":
        f = gqf.GQF(case["nbits"])
        f.reserve(case["batch"])
        s["keys"] = _keys(seed, int(case["load"] * size))
        s["filters"], s["buf"], s["image"] = [f], torch.empty_like(s["keys"]), _image(f)
        return s
    n_base = int(case["load"] * size)
    base = _keys(seed, n_base)
    if kind == "dump":
        # a share of the insertions hits hashes that are there already
        n = _items(case)
        base = workloads.distinct_keys(seed * 1000003 + 17, n, case["nbits"] + 8, device="cuda")
        again = base[torch.remainder(_keys(seed, n_base - n, 1) >> 1, n)]
        s["filters"] = [_filled(case["nbits"], torch.cat([base, again]))]
    elif kind == "merge":
        other = _pick(seed, base, _keys(seed, n_base, 1), case["shared"])
        s["filters"] = [_filled(case["nbits"], base), _filled(case["nbits"], other), gqf.GQF(case["nbits"])]
        s["image"] = _image(s["filters"][2])
    elif kind == "get":
        n = case["n"]
        hit = base[torch.remainder(_keys(seed, n, 1) >> 1, n_base)]
        s["vals"] = _pick(seed, hit, _keys(seed, n, 2), case["present"])
        s["filters"], s["counts"] = [_filled(case["nbits"], base)], torch.empty_like(s["vals"])
    elif kind == "window":
        n = case["n"]
        s["new"] = _keys(seed, n, 1)
        s["vals"] = _pick(seed, s["new"], base[torch.remainder(_keys(seed, n, 2) >> 1, n_base)], 0.5)
        f = _filled(case["nbits"], base, n)
        s["filters"], s["image"] = [f], _image(f)
        s["ins"], s["outs"], s["counts"] = (torch.empty_like(s["new"]) for _ in range(3))
    elif kind == "requests":
        _prepare_requests(s, case, seed, base)
    return s


def _prepare_requests(s, case, seed, base):
    """A served batch: 60% gets, 30% inserts, 10% deletes of lognormal size;
    then the batch that takes its inserts out and puts its deletes back."""
    # who asks for what comes from the case, the keys from the seed
    _, reqs = workloads.serve_workload(case["requests"], 1, 6, median_log2=case["median"], max_log2=18)
    fresh, used, there = 0, 0, []
    for _, _, op, n, _ in reqs:
        if op == "insert":
            there.append((op, fresh, n))
            fresh += n
        elif op == "delete":
            n = min(n, base.numel() // 8 // case["requests"] + 1)
            there.append((op, used, n))
            used += n
        else:
            there.append((op, 0, n))
    new = _keys(seed, max(1, fresh), 1)
    batches = []
    for undo in (False, True):
        get_keys, get_ends, get_seqs, mut_keys, mut_ends, mut_tags = [], [], [], [], [], []
        got = muts = 0
        for i, (op, at, n) in enumerate(there):
            if op == "get":
                src = (base, new)[i % 2]
                get_keys.append(src[torch.remainder(_keys(seed, n, 3 + i) >> 1, src.numel())])
                got += n
                get_ends.append(got)
                get_seqs.append(i)
            else:
                mut_keys.append((new if op == "insert" else base)[at:at + n])
                muts += n
                mut_ends.append(muts)
                mut_tags.append(i << 1 | ((op == "delete") != undo))
        empty = torch.empty(0, dtype=torch.int64, device="cuda")
        gets, mut = torch.cat([empty] + get_keys), torch.cat([empty] + mut_keys)
        batches.append({"gets": gets, "get_ends": get_ends, "get_seqs": get_seqs, "mut": mut,
                        "buf": torch.empty_like(mut), "mut_ends": mut_ends, "mut_tags": mut_tags,
                        "counts": torch.empty_like(gets)})
    f = _filled(case["nbits"], base, max(1, batches[0]["mut"].numel()))
    s["filters"], s["image"], s["batches"] = [f], _image(f), batches


# ------------------------------------------------------------------ one pass

def run(s):
    kind, f = s["kind"], s["filters"][0]
    if kind == "get":
        return f.bulk_get(s["vals"], s["counts"])
    if kind == "fill":
        s["buf"].copy_(s["keys"])
        f.reset()
        for i in range(0, s["buf"].numel(), s["batch"]):
            f.bulk_insert(s["buf"][i:i + s["batch"]])
        return s["buf"], f.export_image_device(s["image"])
    if kind == "window":
        s["ins"].copy_(s["new"])
        f.bulk_insert(s["ins"])
        f.bulk_get(s["vals"], s["counts"])
        s["outs"].copy_(s["new"])
        f.bulk_delete(s["outs"])
        return s["ins"], s["counts"], s["outs"], f.export_image_device(s["image"])
    if kind == "count":
        s["buf"].copy_(s["keys"])
        f.reset()
        f.bulk_insert_reduce(s["buf"])
        return s["buf"], f.export_image_device(s["image"])
    if kind == "group":
        s["buf"].copy_(s["keys"])
        for g in s["filters"]:
            g.reset()
        s["group"].bulk_insert(s["buf"], s["offsets"])
        s["group"].bulk_get(s["keys"], s["offsets"], s["counts"])
        images = [g.export_image_device(i) for g, i in zip(s["filters"], s["images"])]
        return [s["buf"], s["counts"]] + images
    if kind == "requests":
        out = []
        for b in s["batches"]:
            if b["gets"].numel():
                f.bulk_get(b["gets"], b["counts"])
            if b["mut"].numel():
                b["buf"].copy_(b["mut"])
                f.mutate_seq(b["buf"], b["mut_ends"], b["mut_tags"])
                if b["gets"].numel():
                    f.get_seq_adjust(b["gets"], b["get_ends"], b["get_seqs"], b["counts"], b["buf"])
            out += [b["counts"], b["buf"]]
        return out + [f.export_image_device(s["image"])]
    if kind == "dump":
        keys, counts = f.enumerate(form=gqf.QF_ENUM_KEY)
        stats = f.stats()
        _, hist, longest = f.cluster_census(nbins=4096, lengths=False)
        return keys, counts, stats, hist, longest
    target = s["filters"][2]
    target.reset()
    moved = target.merge_from(s["filters"][0], s["filters"][1])
    return moved, target.export_image_device(s["image"])


# ------------------------------------------------- what a pass has to move

def _blocks(q):
    return ((1 << q) + int(10 * math.sqrt(1 << q)) + 63) // 64


def _touched(q, n):
    """Bytes of the distinct home blocks of n random hashes."""
    b = _blocks(q)
    return BLOCK * b * -math.expm1(-n / b)


def work(case):
    kind = case["kind"]
    if kind == "group":
        params = _group_sizes(case)
        n, table = sum(p[2] for p in params), sum(BLOCK * _blocks(p[0]) for p in params)
        # keys in and sorted out, every table built once, keys and counts of the lookups, the tables again for the images
        return {"bytes": 32 * n + 4 * table, "flops": 0}
    q = case["nbits"]
    table = BLOCK * _blocks(q)
    if kind == "get":
        return {"bytes": 16 * case["n"] + _touched(q, case["n"]), "flops": 0}
    if kind == "fill":
        n, m = int(case["load"] * (1 << q)), case["batch"]
        steps = sum(16 * min(m, n - i) + 2 * _touched(q, min(m, n - i)) for i in range(0, n, m))
        return {"bytes": 16 * n + steps + 3 * table, "flops": 0}
    if kind == "window":
        n = case["n"]
        return {"bytes": 32 * n + 32 * n + 16 * n + 5 * _touched(q, n) + 2 * table, "flops": 0}
    if kind == "count":
        return {"bytes": 32 * case["n"] + 4 * table, "flops": 0}
    if kind == "requests":
        n = case["requests"] * 2.0 ** case["median"] * math.exp(0.5)
        gets, muts = 0.6 * n, 0.4 * n
        return {"bytes": 2 * (16 * gets + 32 * muts + _touched(q, gets) + 2 * _touched(q, muts)) + 2 * table, "flops": 0}
    if kind == "dump":
        return {"bytes": 3 * table + 16 * _items(case), "flops": 0}
    return {"bytes": 2 * table + 2 * table + 2 * table, "flops": 0}


def exact(case, seed):
    """Every output is whole numbers or bytes, which stay equal bit for bit."""
    return None
