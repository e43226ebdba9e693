"""The work that users of this framework have it do, as cases to be timed.

Every case goes through the package's public entry points, as a program that
clusters or serves sequences calls them:

  step    one whole pass over a resident database: sketch, bucketing and the
          batched graph (Database.step), then the edge list (Database.edges)
  makedb  the makeDB half: signatures and bucketing, representative rows read
          back to the host, where they go into the packed DB file
  graph   the cluster half on host arrays as read from a packed DB file:
          upload, graph and edge list (Context.build_graph)
  fast    the fast mode (-m fast): clusters without a graph (Database.fast)
  align   the scoring seam: a list of (rep, tar) jobs on the host
          (Context.align)
  serve   a request of query sequences assigned to the clusters of a resident
          set (Serve.assign)

The sequence sets are those of the package's generator (gen_config): 1 is
proteins of 50-1,000 residues in large families, 2 log-normal proteins of
30-5,000, 3 DNA of 1,000-1,800 bases, 4 heavy-tailed proteins of up to 35,000
residues.  Record lengths are ragged in all of them.
"""
import math

import numpy as np

import ngia2_amd as ng

# Mean record length per set, for work().
_MEAN_LEN = {1: 340.0, 2: 397.0, 3: 1400.0, 4: 387.0}
# Distinct candidate pairs per record, for work(): a record shares a band with
# a few members of its family (proteins), or with most bands' chance hits in
# DNA, whose 8-mers repeat across families.
_PAIRS_PER_SEQ = {1: 7.0, 2: 4.5, 3: 40.0, 4: 4.0}


def listed():
    return [
        # The smallest whole call: a gene family of a few hundred proteins,
        # where launches and waits count.
        {"name": "step_500_i60", "kind": "step", "set": 1, "families": 10, "members": 50,
         "identity": 60, "bands": 64},
        # A bacterial proteome's worth of sequences.
        {"name": "step_10k_i70", "kind": "step", "set": 1, "families": 200, "members": 50,
         "identity": 70, "bands": 64},
        # An ordinary non-redundant set at a middle identity.
        {"name": "step_100k_i70", "kind": "step", "set": 2, "families": 5000, "members": 20,
         "identity": 70, "bands": 64},
        # A large set at a low identity: wide bands, millions of alignments.
        {"name": "step_1m_i50", "kind": "step", "set": 2, "families": 50000, "members": 20,
         "identity": 50, "bands": 64},
        # The headline workload: a million heavy-tailed proteins at -i 90.
        {"name": "step_heavy_1m_i90", "kind": "step", "set": 4, "families": 50000, "members": 20,
         "identity": 90, "bands": 64},
        # DNA (16S-like reads) at a high identity.
        {"name": "step_dna_200k_i97", "kind": "step", "set": 3, "families": 2000, "members": 100,
         "identity": 97, "bands": 64},
        # makeDB of a middling heavy-tailed set, rows read back for the file.
        {"name": "makedb_50k", "kind": "makedb", "set": 4, "families": 2500, "members": 20,
         "identity": 90, "bands": 64},
        # cluster on a packed DB just read from disk, with fewer bands than
        # the file holds (the -b option).
        {"name": "graph_100k_i80_b40", "kind": "graph", "set": 2, "families": 5000, "members": 20,
         "identity": 80, "bands": 40},
        # Quick clustering without the graph.
        {"name": "fast_100k_i90", "kind": "fast", "set": 2, "families": 5000, "members": 20,
         "identity": 90, "bands": 64},
        # A job list scored for a program with candidates of its own.
        {"name": "align_20k_i80", "kind": "align", "set": 1, "families": 150, "members": 41,
         "identity": 80, "bands": 64, "jobs": 20011},
        # One small interactive request against a resident set.
        {"name": "serve_16", "kind": "serve", "set": 4, "families": 5000, "members": 20,
         "identity": 90, "bands": 64, "queries": 16},
        # A bulk request against the same residents.
        {"name": "serve_20k", "kind": "serve", "set": 4, "families": 5000, "members": 20,
         "identity": 90, "bands": 64, "queries": 20000},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "makedb", "graph", "fast", "align", "serve"])
    sets = {"step": [1, 2, 3, 4], "makedb": [1, 2, 3, 4], "graph": [1, 2, 3, 4],
            "fast": [1, 2, 3], "align": [1, 2], "serve": [1, 2, 4]}[kind]
    s = rng.choice(sets)
    members = rng.randint(3, 60)
    top = {"step": 300000, "makedb": 200000, "graph": 100000, "fast": 60000, "align": 20000,
           "serve": 100000}[kind]
    if s == 3:
        top = min(top, 60000)
    n = _log_uniform(rng, 300, top)
    # very long pairs at low identities would pass the largest listed case
    identity = rng.randint(90, 98) if s == 3 else rng.randint(75 if s == 4 else 50, 96)
    case = {"kind": kind, "set": s, "families": max(1, n // members), "members": members,
            "identity": identity, "bands": 64 if rng.random() < 0.6 else rng.randint(16, 63)}
    if kind == "align":
        case["jobs"] = _log_uniform(rng, 50, 40000)
    if kind == "serve":
        case["bands"] = 64
        case["queries"] = _log_uniform(rng, 1, 20000)
    return case


def _records(case, seed):
    p = ng.gen_config(case["set"], 1.0, seed)
    p.n_families = case["families"]
    p.members = case["members"]
    return ng.gen_packed(p)


def prepare(case, seed):
    d = _records(case, seed)
    kind = case["kind"]
    ctx = ng.Context(0)
    st = {"case": case, "ctx": ctx, "d": d}
    if kind in ("step", "graph"):
        st["edges"] = _edge_buffer(case, d.n)
    if kind in ("step", "makedb"):
        st["db"] = ng.Database(ctx, d.packed, d.word_off, d.lengths)
        return st
    # the others start from a database that makeDB has sketched and bucketed
    db = ng.Database(ctx, d.packed, d.word_off, d.lengths)
    db.sketch()
    db.bucket()
    if kind == "fast":
        st["db"] = db
    elif kind == "graph":
        st["reps"] = db.reps()[:case["bands"]].copy()
        db.close()
    elif kind == "align":
        st["jobs"] = _candidate_jobs(db.reps(), case["jobs"], seed)
        db.close()
    else:
        db.graph(case["identity"], 64)
        part = ng.leiden(db.edges(), d.n, ng.resolution(case["identity"]))
        st["queries"] = ng.gen_queries(d.packed, d.word_off, case["queries"], mutated=0.7,
                                       sub=(0.0, 0.3), indel=0.01, len_median=300.0, len_sigma=0.5,
                                       len_min=30, len_max=5000, seed=seed + 1)
        st["serve"] = ng.Serve(db, part, case["identity"], int(part.max()) + 1,
                               grow_queries=1 << 16, grow_residues=1 << 27)
        db.close()
    return st


def _candidate_jobs(reps, count, seed):
    """`count` distinct (rep, tar) candidates in a shuffled order (repeated
    when the set has fewer), with a zero score column."""
    n = reps.shape[1]
    tar = np.broadcast_to(np.arange(n, dtype=np.uint64), reps.shape)
    has = reps != tar
    keys = np.unique((reps[has].astype(np.uint64) << np.uint64(32)) | tar[has])
    if len(keys) == 0:
        keys = np.array([min(1, n - 1)], dtype=np.uint64)
    pick = np.random.default_rng(seed).permutation(len(keys))
    keys = keys[pick[np.arange(count) % len(keys)]]
    jobs = np.zeros((count, 3), dtype=np.uint32)
    jobs[:, 0] = keys >> np.uint64(32)
    jobs[:, 1] = keys & np.uint64(0xFFFFFFFF)
    return jobs


def _edge_buffer(case, n):
    """The program's own edge list, with room for the edges of n records: a
    record has few representatives above the identity threshold (at most one
    per band and family member)."""
    per = min(case["bands"], case["members"], {1: 12, 2: 6, 3: 40, 4: 6}[case["set"]])
    return np.zeros((n * per, 3), dtype=np.int32)


def _edges(state, e):
    out = state["edges"]
    out[:len(e)] = e.view(np.int32).reshape(-1, 3)
    return {"count": len(e), "edges": out}


def run(state):
    case, d = state["case"], state["d"]
    kind = case["kind"]
    if kind == "step":
        state["db"].step(case["identity"], case["bands"])
        return _edges(state, state["db"].edges())
    if kind == "makedb":
        state["db"].sketch()
        state["db"].bucket()
        return {"reps": state["db"].reps()}
    if kind == "graph":
        e, _ = state["ctx"].build_graph(d.packed, d.word_off, d.lengths, state["reps"],
                                        case["bands"], case["identity"])
        return _edges(state, e)
    if kind == "fast":
        cl, total = state["db"].fast(case["identity"], case["bands"])
        return {"cluster": cl, "pairs": int(total)}
    if kind == "align":
        return {"jobs": state["ctx"].align(d.packed, d.word_off, state["jobs"],
                                           case["identity"] / 100.0)}
    # a session of one request: the snapshot goes back to the residents first
    state["serve"].reset()
    a, _ = state["serve"].assign(state["queries"])
    return {k: np.ascontiguousarray(a[k]) for k in ("cluster", "resident", "score", "candidates")}


def work(case):
    """Bytes: the packed records (4 bits per residue, offsets and lengths) read
    once, the results written once.  Operations: 17 integer operations per
    8-mer and band (the hash), and 4 per 32 cells of a candidate's band (the
    bit-parallel row update), for the expected number of candidates."""
    kind = case["kind"]
    m = _MEAN_LEN[case["set"]]
    n = case["families"] * case["members"]
    thr = case["identity"] / 100.0
    record = 16.0 * (m / 32.0 + 0.5) + 16.0
    sketch_ops = 17.0 * 64.0 * max(m - 7.0, 1.0)
    blocks = m / 32.0
    window = 2.0 * math.ceil(m * (1.0 - thr) / 32.0) + 1.0
    align_ops = 128.0 * blocks * min(window, blocks)
    pairs = n * min(_PAIRS_PER_SEQ[case["set"]], case["members"]) * case["bands"] / 64.0
    if kind == "step":
        return {"bytes": n * record + 12.0 * n * 0.5, "flops": n * sketch_ops + pairs * align_ops}
    if kind == "makedb":
        return {"bytes": n * record + 256.0 * n, "flops": n * sketch_ops}
    if kind == "graph":
        return {"bytes": n * (record + 4.0 * case["bands"]) + 12.0 * n * 0.5,
                "flops": pairs * align_ops}
    if kind == "fast":
        return {"bytes": n * (record + 4.0 * case["bands"] + 4.0), "flops": pairs * align_ops}
    if kind == "align":
        return {"bytes": n * record + 24.0 * case["jobs"], "flops": case["jobs"] * align_ops}
    q = case["queries"]
    return {"bytes": q * (m + 16.0 + record * 4.0), "flops": q * (sketch_ops + 4.0 * align_ops)}


def exact(case, seed):
    """No output is a rounded number: signatures, rows, scores and clusters are
    whole numbers, and an edge is the 12 bytes of its two indices and the
    weight score / 100, returned as three 32-bit words."""
    return None
