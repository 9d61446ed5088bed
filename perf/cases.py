"""What is timed of this framework: the calls its users make, over the sizes
they make them at.

Four kinds of call, each on inputs a seed alone determines (random RNAs and
their base-pair probabilities from the package's host folding, as in its
tests and benchmark):

  align  a batch of prepared pairs: lcg_batch_run (fill of D, top level,
         traceback), then score, alignment and structures of every pair
  pf     a batch of LocARNA-P pairs: lcg_batch_pf_run (inside and outside),
         then the probabilities, or the gradient of log Z for fitting
  fold   base-pair probabilities of single sequences (lcg_fold_run)
  whole  from texts or sequences to alignments in one go: mlocarna's
         all-pairs stage (preparation with device band and compaction, batch,
         run, results) or its default run (lcg_mlocarna_run)
"""
import concurrent.futures as cf
import ctypes
import math
import os
import random

import numpy as np
import torch

from locarna_amd import api, synth

_THREADS = 16


def listed():
    return [
        # locarna on two tRNA-sized sequences: one small pair, latency
        {"name": "align_pair_trna", "kind": "align", "count": 2, "pairing": "adjacent", "len_min": 71, "len_max": 77,
         "span": 100, "local": False, "graph": False},
        # all pairs of a small family of ragged sequences, sequence-local
        {"name": "align_all16_local", "kind": "align", "count": 16, "pairing": "all", "len_min": 35, "len_max": 149,
         "span": 100, "local": True, "graph": False},
        # the benchmark's all-pairs batch: 2016 pairs, replayed as a graph
        {"name": "align_all64", "kind": "align", "count": 64, "pairing": "all", "len_min": 60, "len_max": 200,
         "span": 100, "local": False, "graph": True},
        # a few long pairs: fewer pairs than compute units
        {"name": "align_long500", "kind": "align", "count": 8, "pairing": "adjacent", "len_min": 500, "len_max": 500,
         "span": 200, "local": False, "graph": True},
        # locarna_p on one pair: match probabilities
        {"name": "pf_pair", "kind": "pf", "count": 2, "pairing": "adjacent", "len_min": 85, "len_max": 95,
         "span": 100, "grad": False},
        # mlocarna --probabilistic's pairwise stage over 16 sequences
        {"name": "pf_all16x150", "kind": "pf", "count": 16, "pairing": "all", "len_min": 150, "len_max": 150,
         "span": 100, "grad": False},
        # one gradient step of a parameter fit over ragged pairs
        {"name": "pf_grad48", "kind": "pf", "count": 96, "pairing": "adjacent", "len_min": 80, "len_max": 250,
         "span": 100, "grad": True},
        # locarna_rnafold_pp on one tRNA-sized sequence
        {"name": "fold_one", "kind": "fold", "count": 1, "len_min": 71, "len_max": 77, "span": -1, "out": "probs"},
        # the input step of the benchmark's 64 sequences: pp texts
        {"name": "fold_all64", "kind": "fold", "count": 64, "len_min": 60, "len_max": 200, "span": 100, "out": "pp"},
        # two long sequences without a span limit
        {"name": "fold_long", "kind": "fold", "count": 2, "len_min": 700, "len_max": 800, "span": -1, "out": "probs"},
        # mlocarna's all-pairs stage from pp texts to alignments on the host
        {"name": "stage_all32", "kind": "whole", "what": "pairs", "count": 32, "len_min": 60, "len_max": 200,
         "span": 100},
        # mlocarna's default run from sequences to the multiple alignment
        {"name": "mlocarna12", "kind": "whole", "what": "mlocarna", "count": 12, "len_min": 60, "len_max": 130,
         "span": 100},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["align", "align", "pf", "pf", "fold", "whole"])
    if kind == "align":
        pairing = rng.choice(["all", "adjacent"])
        hi = _log(rng, 50, 200) if pairing == "all" else _log(rng, 50, 500)
        lo = max(30, int(hi * rng.uniform(0.3, 1.0)))
        count = _log(rng, 3, 56) if pairing == "all" else 2 * _log(rng, 1, 4 if hi > 200 else 64)
        return {"kind": kind, "count": count, "pairing": pairing, "len_min": lo, "len_max": hi,
                "span": rng.choice([100, 100, 120, 150 if hi < 400 else 200]), "local": rng.random() < 0.3,
                "graph": rng.random() < 0.5}
    if kind == "pf":
        pairing = rng.choice(["all", "adjacent"])
        hi = _log(rng, 50, 150) if pairing == "all" else _log(rng, 50, 250)
        lo = max(30, int(hi * rng.uniform(0.4, 1.0)))
        count = _log(rng, 3, 14) if pairing == "all" else 2 * _log(rng, 1, 40)
        return {"kind": kind, "count": count, "pairing": pairing, "len_min": lo, "len_max": hi, "span": 100,
                "grad": rng.random() < 0.4}
    if kind == "fold":
        hi = _log(rng, 50, 700)
        lo = max(30, int(hi * rng.uniform(0.3, 1.0)))
        return {"kind": kind, "count": _log(rng, 1, 64) if hi <= 200 else rng.randint(1, 2), "len_min": lo,
                "len_max": hi, "span": rng.choice([-1, 100, 150]), "out": rng.choice(["probs", "pp"])}
    what = rng.choice(["pairs", "mlocarna"])
    hi = _log(rng, 70, 200 if what == "pairs" else 130)
    return {"kind": "whole", "what": what, "count": rng.randint(5, 31 if what == "pairs" else 12),
            "len_min": max(40, int(hi * rng.uniform(0.4, 1.0))), "len_max": hi, "span": 100}


def _lengths(case):
    """The sequences' lengths: the case's own, so that outputs of every seed
    have one shape."""
    rng = random.Random("%(count)d %(len_min)d %(len_max)d" % case)
    return [rng.randint(case["len_min"], case["len_max"]) for _ in range(case["count"])]


def _sequences(case, seed):
    gc = (0.35, 0.65) if case["len_min"] < case["len_max"] else (0.5, 0.5)
    return [synth.sequences(seed * 1009 + k, 1, n, n, *gc)[0] for k, n in enumerate(_lengths(case))]


def _pp_texts(case, seed):
    seqs = _sequences(case, seed)
    with cf.ThreadPoolExecutor(min(_THREADS, os.cpu_count() or 1)) as ex:
        return list(ex.map(lambda k: synth.make_pp("s%03d" % k, seqs[k], case["span"]), range(len(seqs))))


def _ptr(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def _keep_text(state, key, texts, cap):
    """The texts one after the other in a buffer of `cap` bytes."""
    data = "".join(texts).encode()
    buf = state.setdefault(key, np.zeros(cap, np.uint8))
    buf[:len(data)] = np.frombuffer(data, np.uint8)
    return buf


def _alignment_buffers(lens):
    """Flat buffers for the alignments of all pairs, and one pair's offsets."""
    cap = [a + b + 2 for a, b in lens]
    at = np.concatenate([[0], np.cumsum(cap)])
    total = int(at[-1])
    buf = {"scores": np.zeros(len(lens), np.int64), "edges": np.zeros(len(lens), np.int64),
           "a": np.zeros(total, np.int32), "b": np.zeros(total, np.int32),
           "sa": np.zeros(total, np.uint8), "sb": np.zeros(total, np.uint8)}
    base = {k: buf[k].ctypes.data for k in ("a", "b", "sa", "sb", "scores")}
    where = []
    for k in range(len(lens)):
        o = int(at[k])
        where.append((base["a"] + 4 * o, base["b"] + 4 * o, cap[k],
                      ctypes.cast(base["sa"] + o, ctypes.c_char_p), ctypes.cast(base["sb"] + o, ctypes.c_char_p),
                      ctypes.cast(base["scores"] + 8 * k, ctypes.POINTER(ctypes.c_int64))))
    return buf, where


def _fetch_alignments(h, buf, where):
    L = api.lib()
    score, align, edges = L.lcg_batch_score, L.lcg_batch_alignment, buf["edges"]
    for k, (a, b, cap, sa, sb, sc) in enumerate(where):
        if score(h, k, sc) != 0:
            raise RuntimeError("lcg_batch_score")
        n = align(h, k, a, b, cap, sa, sb, cap)
        if n < 0:
            raise RuntimeError("lcg_batch_alignment (%d)" % n)
        edges[k] = n
    return buf


def prepare(case, seed):
    device = torch.cuda.current_device()
    state = {"case": case, "device": device}
    if case["kind"] == "fold":
        state["seqs"] = _sequences(case, seed)
        return state
    if case["kind"] == "whole" and case["what"] == "mlocarna":
        state["seqs"] = _sequences(case, seed)
        state["names"] = ["s%03d" % k for k in range(case["count"])]
        return state
    pps = _pp_texts(case, seed)
    idx = synth.pair_list(case["count"], case.get("pairing", "all"))
    texts = [(pps[a], pps[b]) for a, b in idx]
    if case["kind"] == "whole":
        state["texts"] = texts
        state["params"] = api.locarna_params(max_bp_span=case["span"])
        return state
    if case["kind"] == "align":
        params = api.locarna_params(max_bp_span=case["span"], sequ_local=1 if case["local"] else 0)
        pairs, _ = api.prepare_pairs(texts, params, device_compaction=True, device_band=True, threads=_THREADS,
                                     device=device)
        state["batch"] = api.Batch(pairs, device=device)
        state["out"], state["where"] = _alignment_buffers([(p.lenA, p.lenB) for p in pairs])
        return state
    params = api.locarna_p_params(max_bp_span=case["span"])
    pairs, _ = api.prepare_pairs(texts, params, threads=_THREADS, device=device)
    state["batch"] = api.Batch(pairs, device=device)
    n = len(pairs)
    out = {"Z": np.zeros(n), "openings": np.zeros(n)}
    if case["grad"]:
        rng = random.Random(seed)
        # score offsets of a fit under way: about one score unit in a hundred
        state["dtheta"] = [rng.gauss(0.0, 3.0) for _ in range(api.NTHETA)]
        out["grad"] = np.zeros((n, api.NTHETA))
    else:
        # room for the arc matches of any input of these lengths
        state["am_at"] = np.concatenate([[0], np.cumsum([200 * (p.lenA + p.lenB) for p in pairs])]).astype(int)
        state["bm_at"] = np.concatenate([[0], np.cumsum([(p.lenA + 1) * (p.lenB + 1) for p in pairs])]).astype(int)
        out["am"] = np.zeros(int(state["am_at"][-1]))
        out["bm"] = np.zeros(int(state["bm_at"][-1]))
    state["out"] = out
    return state


def _run_pf(state):
    L, batch, out = api.lib(), state["batch"], state["out"]
    grad = state["case"]["grad"]
    batch.pf_run(state.get("dtheta"))
    for k in range(len(batch.pairs)):
        out["Z"][k], out["openings"][k] = batch.pf_result(k)
        if grad:
            if L.lcg_batch_pf_grad(batch.h, k, _ptr(out["grad"][k]), api.NTHETA) < 0:
                raise RuntimeError("lcg_batch_pf_grad")
            continue
        a, b = out["am"][state["am_at"][k]:state["am_at"][k + 1]], out["bm"][state["bm_at"][k]:state["bm_at"][k + 1]]
        if not 0 <= L.lcg_batch_am_probs(batch.h, k, _ptr(a), a.size) <= a.size:
            raise RuntimeError("lcg_batch_am_probs")
        if L.lcg_batch_bm_probs(batch.h, k, 0, _ptr(b), b.size) < 0:
            raise RuntimeError("lcg_batch_bm_probs")
    return out


def _run_fold(state):
    case = state["case"]
    F = api.Fold(state["seqs"], max_bp_span=case["span"], min_prob=synth.BPCUT, device=state["device"])
    n = len(state["seqs"])
    out = {"log_z": np.array([F.log_z(k) for k in range(n)])}
    if case["out"] == "pp":
        out["pp"] = _keep_text(state, "pp", [F.pp(k, "s%03d" % k) for k in range(n)],
                               sum(400 * len(s) + 200 for s in state["seqs"]))
    else:
        both = [F.probs(k) for k in range(n)]
        out["P"] = [p for p, _ in both] if n <= 8 else np.concatenate([p.ravel() for p, _ in both])
        out["P2"] = [q for _, q in both] if n <= 8 else np.concatenate([q.ravel() for _, q in both])
    F.destroy()
    return out


def run(state):
    case = state["case"]
    if case["kind"] == "align":
        state["batch"].run(mode=2 if case["graph"] else 0, trace=True)
        return _fetch_alignments(state["batch"].h, state["out"], state["where"])
    if case["kind"] == "pf":
        return _run_pf(state)
    if case["kind"] == "fold":
        return _run_fold(state)
    if case["what"] == "pairs":
        pairs, _ = api.prepare_pairs(state["texts"], state["params"], device_compaction=True, device_band=True,
                                     threads=_THREADS, device=state["device"])
        batch = api.Batch(pairs, device=state["device"])
        batch.run(mode=0, trace=True)
        buf, where = _alignment_buffers([(p.lenA, p.lenB) for p in pairs])
        out = _fetch_alignments(batch.h, buf, where)
        batch.destroy()
        return out
    M = api.Mlocarna(state["names"], state["seqs"], max_bp_span=case["span"], device=state["device"])
    out = {"scores": np.array(M.scores()), "tree": np.array(M.tree()),
           "clustal": _keep_text(state, "clustal", [M.clustal()], 4000 + 40 * sum(len(s) + 40 for s in state["seqs"]))}
    M.destroy()
    return out


def work(case):
    """Estimates from the sizes: C cells of the arc-match regions and the top
    level inside the trace band (about 0.7 n^2 min(n, span) a pair on these
    inputs), K = 2.5 C arc terms; 11 C + 2 K integer operations, and three
    times 13 C + 2 K in double for LocARNA-P with its outside pass."""
    n = 0.5 * (case["len_min"] + case["len_max"])
    span = case["span"] if case["span"] > 0 else n
    count = case["count"]
    fold = {"bytes": count * (n + 16 * n * min(n, span)),
            "flops": count * 2.0 * n * min(n, span) * (0.37 * 2 * 496 + 2.0 * min(n, span))}
    if case["kind"] == "fold":
        return fold
    pairs = count // 2 if case.get("pairing") == "adjacent" else count * (count - 1) // 2
    cells = pairs * 0.7 * n * n * min(n, span)
    arcs = 40.0 * n * min(n, span) / 100.0 * pairs  # arc matches of a pair, about
    if case["kind"] == "pf":
        out = 8.0 * pairs * (api.NTHETA if case["grad"] else n * n) + (0 if case["grad"] else 8 * arcs)
        return {"bytes": 24 * arcs + out, "flops": 3 * 18 * cells}
    w = {"bytes": 24 * arcs + pairs * 40.0 * n, "flops": 16 * cells}
    if case.get("what") == "mlocarna":  # folding, all pairs, and as many profile merges as sequences
        w = {"bytes": w["bytes"] + fold["bytes"], "flops": w["flops"] * (1 + 2.0 / count) + fold["flops"]}
    return w


def tolerance(case):
    if case["kind"] == "pf":
        return {"rel": 1e-11, "max": 1e-9}
    if case["kind"] == "fold":
        # texts: 6 significant digits of a probability, one in a million of
        # which may round the other way
        return {"rel": 1e-11, "max": 1e-9, "differ": 1e-4}
    return "exact"


# ---- the same values in plain 64-bit torch

def exact(case, seed):
    if case["kind"] == "fold":
        n, span = case["len_max"], case["span"]
        if case["out"] == "pp" or case["count"] * n * min(n, span if span > 0 else n) > 30000:
            return None
        return _exact_fold(case, seed)
    if case["kind"] == "pf" and case["pairing"] == "adjacent" and case["count"] == 2 and case["len_max"] <= 110:
        return _exact_pf(case, seed)
    return None


def _exact_fold(case, seed):
    """McCaskill's partition function over the package's reduced energy model
    (kcal/mol at 37 C), inside by diagonals; the probabilities are derivatives
    of log Z."""
    kT = 0.0019872 * 310.15
    typ = {"AU": 1, "CG": 2, "GC": 3, "UA": 4, "GU": 5, "UG": 6}
    wc = {"AA/UU": -0.93, "AU/UA": -1.10, "UA/AU": -1.33, "CU/GA": -2.08, "CA/GU": -2.11, "GU/CA": -2.24,
          "GA/CU": -2.35, "CG/GC": -2.36, "GG/CC": -3.26, "GC/CG": -3.42}
    bases = {1: "AU", 2: "CG", 3: "GC", 4: "UA", 5: "GU", 6: "UG"}

    def bf(e):
        return math.exp(-e / kT)

    def stack(to, ti):
        (X, Xp), (Y, Yp) = bases[to], bases[ti]
        if to < 5 and ti < 5:
            return wc.get("%s%s/%s%s" % (X, Y, Xp, Yp), wc.get("%s%s/%s%s" % (Yp, Xp, Y, X), -1.0))
        if to >= 5 and ti >= 5:
            return -0.5
        return -1.4 if min(to, ti) in (2, 3) else -1.0

    def wk(t):
        return t in (1, 4, 5, 6)

    def loop(l1, l2, to, ti):
        s = l1 + l2
        if s == 0:
            return stack(to, ti)
        if l1 == 0 or l2 == 0:
            if s == 1:
                return 3.8 + stack(to, ti)
            e = [0, 0, 2.8, 3.2, 3.6, 4.0, 4.4][s] if s <= 6 else 4.4 + 1.75 * kT * math.log(s / 6.0)
            return e + 0.5 * wk(to) + 0.5 * wk(ti)
        e = [0, 0, 0.5, 1.6, 1.1, 2.0, 2.0][s] if s <= 6 else 2.0 + 1.08 * math.log(s / 6.0)
        return e + min(3.0, 0.6 * abs(l1 - l2)) + 0.7 * wk(to) + 0.7 * wk(ti)

    table = torch.zeros(31, 31, 7, 7, dtype=torch.float64)
    for l1 in range(31):
        for l2 in range(31 - l1):
            for to in range(1, 7):
                for ti in range(1, 7):
                    table[l1, l2, to, ti] = bf(loop(l1, l2, to, ti))
    branch = torch.tensor([0.0] + [bf(0.4 + 0.5 * wk(t)) for t in range(1, 7)], dtype=torch.float64)
    close = torch.tensor([0.0] + [bf(3.8 + 0.5 * wk(t)) for t in range(1, 7)], dtype=torch.float64)
    ext = torch.tensor([0.0] + [bf(0.5 * wk(t)) for t in range(1, 7)], dtype=torch.float64)

    def hairpin(L, t):
        e = [0, 0, 0, 5.4, 5.6, 5.7, 5.4, 6.0, 6.1, 6.2][L] if L <= 9 else 6.2 + 1.75 * kT * math.log(L / 9.0)
        return bf(e + 0.5 * wk(t))

    def one(s):
        n = len(s)
        W = n if case["span"] < 0 else min(n, case["span"])
        ty = torch.zeros(n, n, dtype=torch.long)
        for i in range(n):
            for j in range(i + 4, min(n, i + W)):
                ty[i, j] = typ.get(s[i] + s[j], 0)
        x = torch.zeros(n, n, dtype=torch.float64, requires_grad=True)   # log weight of a pair
        y = torch.zeros(n, n, dtype=torch.float64, requires_grad=True)   # log weight of a stack on (i, j)
        ex, ey = torch.exp(x), torch.exp(y)
        zero = torch.zeros(n, dtype=torch.float64)
        qb, qm, qm1 = {}, {}, {}  # diagonal d -> vector over i
        for d in range(W):
            m = n - d
            if d < 4:
                qb[d], qm[d], qm1[d] = zero[:m], zero[:m], zero[:m]
                continue
            t = torch.diagonal(ty, d)
            v = torch.tensor([0.0] + [hairpin(d - 1, k) for k in range(1, 7)], dtype=torch.float64)[t]
            for s2 in range(0, min(30, d - 6) + 1):
                dd = d - 2 - s2
                inner = qb[dd]                       # over k = i + 1 + l1
                l1 = torch.arange(s2 + 1)
                k = torch.arange(m)[:, None] + 1 + l1[None, :]
                tk = torch.diagonal(ty, dd)[k]
                f = table[l1[None, :], (s2 - l1)[None, :], t[:, None], tk]
                if s2 == 0:
                    f = f * torch.diagonal(ey, d)[:, None]
                v = v + (f * inner[k]).sum(1)
            mq = zero[:m]
            for a in range(4, d - 6):                # Qm(i+1, i+1+a) Qm1(i+2+a, j-1)
                b = d - 3 - a
                if b >= 4:
                    mq = mq + qm[a][1:1 + m] * qm1[b][2 + a:2 + a + m]
            v = (v + mq * close[t]) * (t > 0) * torch.diagonal(ex, d)
            qb[d] = v
            q1 = zero[:m]
            for a in range(4, d + 1):
                q1 = q1 + qb[a][:m] * branch[torch.diagonal(ty, a)[:m]]
            qm1[d] = q1
            q = q1
            for a in range(0, d - 4):                # unpaired or Qm(i, i+a), then Qm1(i+a+1, j)
                q = q + (1.0 + qm[a][:m]) * qm1[d - a - 1][a + 1:a + 1 + m]
            qm[d] = q
        z = [torch.ones((), dtype=torch.float64)]
        for j in range(1, n + 1):
            v = z[j - 1]
            for d in range(4, min(W, j)):
                i = j - d - 1                        # 0-based left end
                if ty[i, j - 1] > 0:
                    v = v + z[i] * qb[d][i] * ext[ty[i, j - 1]]
            z.append(v)
        lz = torch.log(z[n])
        gx, gy = torch.autograd.grad(lz, (x, y))
        P, P2 = np.zeros((n + 1, n + 1)), np.zeros((n + 1, n + 1))
        P[1:, 1:], P2[1:, 1:] = gx.numpy(), gy.numpy()
        return float(lz.detach()), P, P2

    got = [one(s) for s in _sequences(case, seed)]
    out = {"log_z": np.array([g[0] for g in got])}
    for name, k in (("P", 1), ("P2", 2)):
        out[name] = [g[k] for g in got] if len(got) <= 8 else np.concatenate([g[k].ravel() for g in got])
    return out


def _exact_pf(case, seed):
    """LocARNA-P's inside recursion over the prepared pair's scores, arc
    matches and band (the integers the host preparation gives), all left ends
    of B at once; probabilities and gradient are derivatives of log Z."""
    pps = _pp_texts(case, seed)
    params = api.locarna_p_params(max_bp_span=case["span"])
    pair = api.Pair(pps[0], pps[1], params)
    n, m = pair.lenA, pair.lenB
    mn, mx = pair.band()
    ams, scores = pair.arcmatches()
    sig, gapA, gapB, _, _ = pair.score_tables()
    T, ps = float(params.temperature_alipf), params.pf_scale
    if case["grad"]:
        return None  # offsets of the scores are the kernel's own parametrisation
    x = torch.zeros(len(ams), dtype=torch.float64, requires_grad=True)  # log weight of an arc match
    eo = math.exp(params.indel_opening / T)
    es = torch.zeros(n + 1, m + 1, dtype=torch.float64)
    for (i, j), v in sig.items():
        es[i, j] = math.exp(v / T)
    gA = [1.0] + [math.exp(gapA[i] / T) for i in range(1, n + 1)]
    gB = torch.tensor([0.0] + [gapB[j] / T for j in range(1, m + 1)], dtype=torch.float64)
    cum = torch.cumsum(gB, 0)
    k = torch.arange(m + 1)
    # a gap run opened right after column k and ending in column j > k
    run = torch.where(k[:, None] < k[None, :], eo * torch.exp(cum[None, :] - cum[:, None]),
                      torch.zeros((), dtype=torch.float64))
    w = torch.exp(torch.tensor(scores, dtype=torch.float64) / T)
    cols = torch.arange(m + 1)
    band = [((cols >= mn[i]) & (cols <= mx[i])).double() for i in range(n + 1)]
    by_right, by_left = {}, {}
    for t, (al, ar, bl, br) in enumerate(ams):
        by_right.setdefault(ar, []).append(t)
        by_left.setdefault(al, []).append(t)
    D = [None] * len(ams)

    def fill(al, origins, last):
        """Rows al .. last of the regions with origins (al, bl)."""
        G = len(origins)
        org = torch.tensor(origins)[:, None]
        first = (cols[None, :] == org).double() / ps
        first = first + (first @ run) * band[al][None, :]
        M = [first]
        E = torch.zeros(G, m + 1, dtype=torch.float64)
        col = torch.full((G,), eo / ps, dtype=torch.float64)
        open_ = torch.ones(G, dtype=torch.float64)
        at = (cols[None, :] == org).double()
        right = (cols[None, :] > org).double()
        for i in range(al + 1, last + 1):
            act = right * band[i][None, :]
            open_ = open_ * (torch.tensor(origins) >= mn[i]).double()
            col = col * gA[i]
            up = M[-1]
            E = (E * gA[i] * (1.0 - eo) + up * gA[i] * eo) * act
            dg = torch.zeros_like(up)
            dg[:, 1:] = up[:, :-1]
            s = (dg * es[i][None, :] + E) * act
            ts = [t for t in by_right.get(i, []) if ams[t][0] > al]
            if ts:
                p = torch.tensor([ams[t][0] - 1 - al for t in ts])
                q = torch.tensor([ams[t][2] - 1 for t in ts])
                j = torch.tensor([ams[t][3] for t in ts])
                rows = torch.stack(M)                     # row, region, column
                val = rows[p, :, q].T * torch.stack([D[t] for t in ts])[None, :] * ps
                s = s + torch.zeros_like(s).index_add(1, j, val) * act
            s = s + at * (col * open_)[:, None]           # column bl
            # F from column j-1 on: a run opened after s or continued, F itself being part of M
            M.append(s + (s @ run) * act)
        return M

    for al in range(n, 0, -1):
        mine = by_left.get(al)
        if not mine:
            continue
        origins = sorted({ams[t][2] for t in mine})
        M = fill(al, origins, max(ams[t][1] for t in mine) - 1)
        place = {b: g for g, b in enumerate(origins)}
        for t in mine:
            _, ar, bl, br = ams[t]
            D[t] = M[ar - 1 - al][place[bl], br - 1] * w[t] * torch.exp(x[t])
    Z = fill(0, [0], n)[n][0, m]
    am, = torch.autograd.grad(torch.log(Z), x)
    padded = np.zeros(200 * (n + m))
    padded[:len(ams)] = am.numpy()
    return {"Z": np.array([float(Z.detach())]), "openings": None, "am": padded, "bm": None}
