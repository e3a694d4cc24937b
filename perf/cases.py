"""The searches whose speed this repository is measured by.

Every case is a batch of trie beam searches as a serving program issues
them: the trie and its search context are created once and kept, the
requests' proposal rows are in host memory, and one pass takes them through
a public entry point to whole results in host memory.

  call "search"  ft_search of the C ABI (include/flashtrie_amd.h) on rows
                 and result arrays that the caller owns: what the C++ facade
                 calls, and the boundary that latency is quoted at
  call "lists"   flashtrie.bs_tbs_gpu on nested Python lists, results
                 collected into arrays as the caller of the module does
  call "numpy"   flashtrie.bs_tbs_gpu on numpy rows, collected likewise
  call "staged"  stage / launch / fetch of the module: a pool of requests
                 staged once per pass and searched in launches of `launch`

Tries (all of them made by the repository's generators from fixed seeds):
  small   100k keys over a 32k vocabulary, length 3-8
  mid     10M key draws over a 256k vocabulary, length 4-12
  large   800M unique keys over a 2.2M vocabulary, length 3-16
  long    200M key draws over a 2.2M vocabulary, length 16-32

Rows come from the proposal models of the repository's workloads:
"example" (one seeded key path per beam slot, forced tokens far above the
distractors) and "literal" (log-softmax of normal logits, 30% of the mass on
one key path).  A case has `beam` hypotheses a step (with `narrow`, a final
beam a third as wide), `topk` proposals a step, `steps` steps and `batch`
requests; `shuffled` rows come in no token order.
"""

import ctypes
import functools
import itertools
import os
import sys

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PACKAGE = os.path.join(ROOT, "flash-trie_amd")
if PACKAGE not in sys.path:
    sys.path.insert(0, PACKAGE)

import flashtrie as ft  # noqa: E402

ALPHA = 5.0  # length-norm exponent of every workload
VOCAB = {"small": 32768, "mid": 262144, "large": 2_200_000, "long": 2_200_000}
SIGMA = {"small": 2.0, "mid": 2.0, "large": 2.5, "long": 2.5}
# limits that a context reserves its workspace for
MAX_BATCH, MAX_TOPK, MAX_STEPS, MAX_BEAM = 64, 1024, 32, 1024


def _case(name, trie, call, batch, beam, topk, steps, model="example", early=False,
          narrow=False, shuffled=False, tok=-10.0, sent=-40.0, launch=0):
    c = dict(trie=trie, call=call, batch=batch, beam=beam, topk=topk, steps=steps, model=model,
             early=early, narrow=narrow, shuffled=shuffled, tok=tok, sent=sent, launch=launch)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest search: a short plan over a small catalogue, where
        # launch and synchronisation count
        _case("small beam 10 b1", "small", "search", 1, 10, 32, 8, "literal"),
        # an interactive request at the common width over a mid-sized trie
        _case("mid beam 100 b1", "mid", "search", 1, 100, 100, 12),
        # a few users at once with a ragged shape: odd widths, rows as the
        # model emits them (by score, not by token), a narrower final beam
        _case("mid beam 333 b3", "mid", "search", 3, 333, 777, 9, narrow=True, shuffled=True),
        # the production-sized trie at its three widths, one request: the
        # latency that a serving system quotes
        _case("large beam 100 b1", "large", "search", 1, 100, 100, 16),
        _case("large beam 500 b2", "large", "search", 2, 500, 500, 16),
        _case("large beam 1000 b1", "large", "search", 1, 1000, 1000, 16),
        # ... and the batch that its throughput is quoted at
        _case("large beam 1000 b8", "large", "search", 8, 1000, 1000, 16),
        # peaked proposals: most hypotheses die in the first steps
        _case("large literal b8", "large", "search", 8, 1000, 1000, 16, "literal"),
        # a full server: more requests than the device has dies
        _case("large beam 1000 b64", "large", "search", 64, 1000, 1000, 16),
        # long keys under early exit and tight thresholds: many steps of
        # hypotheses that only follow their own key
        _case("long early b8", "long", "search", 8, 1000, 1000, 32, early=True, tok=-4.0,
              sent=-20.0),
        # the Python module, called with the lists that a harness builds
        _case("mid lists b8", "mid", "lists", 8, 100, 100, 12),
        # offline scoring: a pool staged at once, searched in launches of 32
        _case("mid staged 128", "mid", "staged", 128, 250, 250, 12, launch=32),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    trie = rng.choice(["small", "mid", "large", "long"])
    call = rng.choice(["search", "search", "search", "numpy", "lists", "staged"])
    if trie not in ("small", "mid"):
        call = "search"
    beam = _log_int(rng, 8, 1000)
    batch = _log_int(rng, 1, 64)
    # (searches that return something: the long keys under early exit need
    # most of their steps, a single literal path all of them, and the paths
    # of a beam a row that holds their tokens)
    model = "example" if trie == "long" else rng.choice(["example", "example", "literal"])
    least = 16 if model == "literal" else max(16, beam)
    topk = least if rng.random() < 0.5 else _log_int(rng, least, 1000)
    early = trie == "long" or rng.random() < 0.2
    full = {"small": 8, "mid": 12, "large": 16, "long": 32}[trie]
    steps = full if model == "literal" else rng.randint(24 if trie == "long" else 6, full)
    tok, sent = (-4.0, -20.0) if trie == "long" else (-10.0, -40.0)
    narrow = rng.random() < 0.25
    # (no drawn case takes longer than the largest listed one)
    shuffled = rng.random() < 0.25 and batch * topk * steps <= 30_000
    return _case(None, trie, call, batch, beam, topk, steps, model, early, narrow, shuffled, tok,
                 sent, launch=max(1, batch // rng.choice([1, 2, 3])) if call == "staged" else 0)


# ---- tries and contexts: what a program creates once and keeps -----------------


@functools.lru_cache(maxsize=None)
def _trie(name):
    t = ft.Trie()
    if name == "small":
        t.build_arrays(*ft.synth_keys(100_000, 32768, 3, 8, 1.1, 0))
    elif name == "mid":
        ft.synth_paper_trie(t, 10_000_000, VOCAB[name], 1.1, 0, lmin=4, lmax=12)
    elif name == "large":
        ft.synth_paper_trie(t, 845_450_000, VOCAB[name], 1.05, 0, unique_keys=800_000_000)
    else:
        ft.synth_paper_trie(t, 200_000_000, VOCAB[name], 1.05, 1, lmin=16, lmax=32)
    return t


@functools.lru_cache(maxsize=None)
def _module_trie(name):
    """The trie with its GPU context, for the Python module's calls."""
    t = ft.Trie()
    t.map(_trie(name).image_view())
    t.init_tbs_gpu(MAX_BATCH, max_num_topk=MAX_TOPK, max_num_outpos=MAX_STEPS,
                   max_num_out_beams=MAX_BEAM, max_num_out_tokens=MAX_BEAM * MAX_STEPS,
                   max_num_inter_beams=MAX_BEAM * MAX_STEPS)
    ft.reserve_staging(t, 128)
    return t


class _Request(ctypes.Structure):
    _fields_ = [("beams", ctypes.c_void_p), ("num_beams", ctypes.c_uint32),
                ("num_steps", ctypes.c_uint32), ("topk", ctypes.c_uint32),
                ("topk_id", ctypes.c_void_p), ("topk_logp", ctypes.c_void_p),
                ("topk_id_rows", ctypes.c_void_p), ("topk_logp_rows", ctypes.c_void_p),
                ("token_logp_threshold", ctypes.c_float),
                ("sent_logp_threshold", ctypes.c_double), ("length_norm", ctypes.c_double),
                ("early_exit", ctypes.c_int)]


class _Result(ctypes.Structure):
    _fields_ = [("capacity", ctypes.c_uint32), ("token_stride", ctypes.c_uint32),
                ("count", ctypes.c_uint32), ("status", ctypes.c_int32),
                ("logp_norm", ctypes.c_void_p), ("length", ctypes.c_void_p),
                ("tokens", ctypes.c_void_p), ("device_ms", ctypes.c_double * 4),
                ("step_stats", ctypes.c_void_p)]


@functools.lru_cache(maxsize=None)
def _lib():
    lib = ctypes.CDLL(os.path.join(PACKAGE, "libflashtrie_amd.so"))
    size, ptr = ctypes.c_size_t, ctypes.c_void_p
    lib.ft_create.argtypes = [ptr, size, ctypes.c_int, ctypes.POINTER(ptr)]
    lib.ft_reserve.argtypes = [ptr] + [size] * 6
    lib.ft_search.argtypes = [ptr, ptr, size, ptr, ptr]
    lib.ft_last_error.restype = ctypes.c_char_p
    return lib


def _check(rc):
    if rc:
        raise RuntimeError("%d: %s" % (rc, _lib().ft_last_error().decode()))


@functools.lru_cache(maxsize=None)
def _context(name):
    """The trie's context of the C ABI."""
    image = _trie(name).image_view()
    ctx = ctypes.c_void_p()
    _check(_lib().ft_create(image.ctypes.data, image.size, 0, ctypes.byref(ctx)))
    _check(_lib().ft_reserve(ctx, MAX_BATCH, MAX_TOPK, MAX_STEPS, MAX_BEAM,
                             MAX_BEAM * MAX_STEPS, MAX_BEAM * MAX_STEPS))
    return ctx


# ---- one case --------------------------------------------------------------------


def _rows(case, seed):
    """The requests of a case: beams [B][T], ids and logps [B][T][K]."""
    B, T, K, beam = case["batch"], case["steps"], case["topk"], case["beam"]
    literal = case["model"] == "literal"
    ids, lps = ft.synth_requests(_trie(case["trie"]), 0, B, VOCAB[case["trie"]], T, K,
                                 1 if literal else beam, 0.3, SIGMA[case["trie"]], True, seed,
                                 threads=16, model=0 if literal else 1)
    if case["shuffled"]:
        at = np.argsort(np.random.default_rng(seed).random((B, T, K)), axis=2)
        ids, lps = np.take_along_axis(ids, at, 2), np.take_along_axis(lps, at, 2)
    beams = np.full((B, T), beam, dtype=np.uint32)
    if case["narrow"]:
        beams[:, -1] = max(1, beam // 3)
    return beams, np.ascontiguousarray(ids), np.ascontiguousarray(lps)


def prepare(case, seed):
    beams, ids, lps = _rows(case, seed)
    B, T = beams.shape
    F = int(beams[0, -1])
    s = dict(case=case, beams=beams, ids=ids, lps=lps)
    if case["call"] != "search":
        s["trie"] = _module_trie(case["trie"])
        if case["call"] == "lists":
            s["beams"], s["ids"], s["lps"] = beams.tolist(), ids.tolist(), lps.tolist()
        s["flat"] = _flat(B, F, T)
        return s
    s["ctx"] = _context(case["trie"])
    s["norms"] = np.zeros((B, F), dtype=np.float64)
    s["lengths"] = np.zeros((B, F), dtype=np.int32)
    s["tokens"] = np.zeros((B, F, T), dtype=np.int32)
    s["reqs"], s["res"] = (_Request * B)(), (_Result * B)()
    for i in range(B):
        s["reqs"][i] = _Request(beams[i].ctypes.data, T, T, case["topk"], ids[i].ctypes.data,
                                lps[i].ctypes.data, None, None, case["tok"], case["sent"], ALPHA,
                                int(case["early"]))
        s["res"][i] = _Result(F, T, 0, 0, s["norms"][i].ctypes.data,
                              s["lengths"][i].ctypes.data, s["tokens"][i].ctypes.data)
    # the counts, read in place of the results that the call fills
    words = np.frombuffer(s["res"], dtype=np.int32).reshape(B, -1)
    s["counts"] = words[:, _Result.count.offset // 4]
    return s


def _flat(B, F, T):
    """Arrays for the module's results, one after another: counts, norms,
    lengths, tokens."""
    return (np.zeros(B, dtype=np.int32), np.zeros(B * F, dtype=np.float64),
            np.zeros(B * F, dtype=np.int32), np.zeros(B * F * T, dtype=np.int32))


def _collect(flat, sents, norms):
    """The module's lists into those arrays."""
    seqs = list(itertools.chain.from_iterable(sents))
    for to, values in zip(flat, (map(len, sents), itertools.chain.from_iterable(norms),
                                 map(len, seqs), itertools.chain.from_iterable(seqs))):
        values = np.fromiter(values, dtype=to.dtype)
        to[:len(values)] = values
    return flat


def run(s):
    case = s["case"]
    if case["call"] == "search":
        _check(_lib().ft_search(s["ctx"], s["reqs"], case["batch"], s["res"], None))
        return s["counts"], s["norms"], s["lengths"], s["tokens"]
    if case["call"] == "staged":
        t, n, step = s["trie"], case["batch"], case["launch"]
        ft.stage(t, s["beams"], s["ids"], s["lps"], case["tok"], case["sent"], ALPHA,
                 case["early"])
        for first in range(0, n, step):
            ft.launch(t, first, min(step, n - first))
        counts, norms, lengths, tokens, _ = ft.fetch(t)
        return counts.view(np.int32), norms, lengths.view(np.int32), tokens.view(np.int32)
    sents, norms, _, _ = ft.bs_tbs_gpu(s["trie"], case["batch"], s["beams"], s["ids"], s["lps"],
                                       case["tok"], case["sent"], ALPHA, case["early"])
    return _collect(s["flat"], sents, norms)


def work(case):
    """Each proposal row read once; of the trie, a 16-byte record for each
    hypothesis that a full beam keeps over the first four steps (few live
    longer); each possible result written once.  No arithmetic to speak of:
    one 64-bit add and multiply a proposal that is taken."""
    B, T, K, beam = case["batch"], case["steps"], case["topk"], case["beam"]
    kept = beam * min(T, 4)
    final = max(1, beam // 3) if case["narrow"] else beam
    return {"bytes": float(B * (T * (8 * K + 4) + 16 * kept + final * (12 + 2 * T))),
            "flops": float(B * 2 * kept)}


def tolerance(case):
    """Scores are 64-bit sums in a fixed order, one multiply each: every
    correct implementation returns the same bits."""
    return "exact"


# ---- the same search in plain numpy ------------------------------------------------


def _image_arrays(name):
    """Records [N + 1][4] (first child, first token, tail offset, meta),
    parents [N] and tail tokens of a trie image."""
    img = _trie(name).image_view()
    head = np.frombuffer(img[:64].tobytes(), dtype="<u8")
    n, tail_len, rec_at, par_at, tail_at = (int(head[i]) for i in (1, 3, 4, 5, 6))
    return (img[rec_at:rec_at + 16 * (n + 1)].view(np.uint32).reshape(-1, 4),
            img[par_at:par_at + 4 * n].view(np.uint32),
            img[tail_at:tail_at + 4 * tail_len].view(np.uint32))


def _keep(norm, node, m):
    """Which pushes (in arrival order) a heap of m entries ends with: it
    drops the smallest (norm, node), and takes no push equal to its least
    norm."""
    if len(norm) <= m:
        return np.ones(len(norm), dtype=bool)
    least = np.partition(norm, len(norm) - m)[len(norm) - m]
    keep = norm > least
    at = np.flatnonzero(norm >= least)[:m]
    at = at[norm[at] == least]
    keep[at[np.argsort(node[at])][len(at) - (m - int(keep.sum())):]] = True
    return keep


def _search(arrays, case, beams, ids, lps):
    """One request: (sequences, norms) in ascending (norm, node) order."""
    recs, parents, tail = arrays
    T, final = len(beams), int(beams[-1])
    scale = [(6.0 / (5.0 + d)) ** ALPHA for d in range(T + 1)]

    def key_token(n, j):  # token j of the string that ends at node n
        while True:
            _, first, off, meta = (int(x) for x in recs[n])
            start = (meta & 0xFFFF) - ((meta >> 16) & 0x3FFF)
            if j >= start:
                return int(tail[off + j - start]) if meta & 0x40000000 else first
            n = int(parents[n])

    cur = [(0.0, 0, ())]  # (sum of logps, node, sequence)
    sel_s, sel_n, sel_q = [], [], []
    for t in range(T):
        if not cur or (case["early"] and len(sel_s) >= final):
            break
        cur.sort(key=lambda h: (h[0] * scale[t], h[1]))
        order = np.argsort(ids[t], kind="stable")
        row = ids[t][order]
        logp = lps[t].astype(np.float64)
        nxt_s, nxt_n, nxt_p, nxt_tok = [], [], [], []
        new_at = []  # pushes that also close a key, by position among all pushes
        for p, (score, node, _) in enumerate(cur):
            meta = int(recs[node, 3])
            depth = meta & 0xFFFF
            if meta & 0x80000000 and depth > t:
                tok = key_token(node, t)
                i = int(np.searchsorted(row, tok))
                at = order[i:i + 1] if i < len(row) and row[i] == tok else order[:0]
                child = np.full(len(at), node, dtype=np.int64)
                closes = np.full(len(at), depth == t + 1)
                goes = ~closes
            else:
                c0, c1 = int(recs[node, 0]), int(recs[node + 1, 0])
                labels = recs[c0:c1, 1]
                if c1 - c0 <= len(row):
                    i = np.searchsorted(row, labels)
                    hit = np.flatnonzero(row[np.minimum(i, len(row) - 1)] == labels)
                    at, child = order[i[hit]], c0 + hit
                else:
                    i = np.searchsorted(labels, row)
                    hit = np.flatnonzero(labels[np.minimum(i, c1 - c0 - 1)] == row)
                    at, child = order[hit], c0 + i[hit]
                by = np.argsort(at)
                at, child = at[by], child[by]
                m = recs[child, 3]
                closes = (m & 0x80000000 != 0) & (m & 0xFFFF == t + 1)
                goes = np.ones(len(at), dtype=bool)
            ok = ~((logp[at] <= np.float32(case["tok"])) | (score + logp[at] <= case["sent"]))
            for a, c, z, g in zip(at[ok], child[ok], closes[ok], goes[ok]):
                if z:
                    new_at.append((score + logp[a], int(c), cur[p][2] + (int(ids[t][a]),)))
                if g:
                    nxt_s.append(score + logp[a])
                    nxt_n.append(int(c))
                    nxt_p.append(p)
                    nxt_tok.append(int(ids[t][a]))
        if case["early"]:
            new_at = new_at[:final - len(sel_s)]
        for s, n, q in new_at:
            sel_s.append(s)
            sel_n.append(n)
            sel_q.append(q)
        if len(sel_s) > final:
            norm = np.array([s * scale[len(q)] for s, q in zip(sel_s, sel_q)])
            keep = _keep(norm, np.array(sel_n), final)
            sel_s, sel_n, sel_q = ([x for x, k in zip(v, keep) if k]
                                   for v in (sel_s, sel_n, sel_q))
        norm = np.array(nxt_s) * scale[t + 1]
        keep = np.flatnonzero(_keep(norm, np.array(nxt_n), int(beams[t])))
        cur = [(nxt_s[i], nxt_n[i], cur[nxt_p[i]][2] + (nxt_tok[i],)) for i in keep]
    done = sorted((s * scale[len(q)], n, q) for s, n, q in zip(sel_s, sel_n, sel_q))
    return [q for _, _, q in done], [s for s, _, _ in done]


def exact(case, seed):
    if case["batch"] * case["beam"] * case["topk"] > 16_000_000:
        return None  # over 20 seconds of plain Python
    beams, ids, lps = _rows(case, seed)
    arrays = _image_arrays(case["trie"])
    got = [_search(arrays, case, *r) for r in zip(beams, ids, lps)]
    B, T = beams.shape
    F = int(beams[0, -1])
    if case["call"] in ("lists", "numpy"):
        return _collect(_flat(B, F, T), [q for q, _ in got], [n for _, n in got])
    counts = np.array([len(q) for q, _ in got], dtype=np.int32)
    norms = np.zeros((B, F), dtype=np.float64)
    lengths = np.zeros((B, F), dtype=np.int32)
    tokens = np.zeros((B, F, T), dtype=np.int32)
    for b, (qs, ns) in enumerate(got):
        norms[b, :len(ns)] = ns
        for i, q in enumerate(qs):
            lengths[b, i] = len(q)
            tokens[b, i, :len(q)] = q
    return counts, norms, lengths, tokens
