"""Work that a serving program has this package do, as measurable cases.

Families (a case's "do"):

* ``step``     -- one decode step, SuffixGPUDrafter.propose_with_update: every
                  row's newest tokens are appended and the next draft is made
                  from the row itself and, with "corpus" > 0, from the global
                  memory.  With "graph" the step is captured once and a pass
                  replays it, as an engine's decode loop does; else a pass is
                  the call itself.
* ``harvest``  -- finished rows go to the global memory
                  (harvest_finished + poll), rebuilding it whenever the delta
                  reaches the rebuild threshold.
* ``sa``       -- build_suffix_array of a token sequence from scratch.
* ``local_op`` -- the operator boundary of the local matcher: match_back,
                  first_occurrences and expand_chain on one batch.
* ``sa_op``    -- the operator boundary of the global search: sa_search of
                  every suffix length of each row's tail.

Text is Zipf(1.1) tokens over a 128256-token vocabulary in short fresh spans,
mixed with copies of earlier spans of the same row ("copy" of the spans) and
with 64 template spans shared by all texts of a seed ("tmpl" of the spans),
which is what makes prompts and responses repeat themselves.
"""

import math

import numpy as np
import torch

from suffixgpu_amd import SuffixGPUDrafter, kernels
from suffixgpu_amd.suffix_array import (build_suffix_array,
                                        build_suffix_array_into)

VOCAB = 128256
SEP = -2
MAX_LEN = 32          # longest pattern, the drafter's default
DEV = "cuda"


# ------------------------------------------------------------------ cases
def _step(name, b, s, corpus=0, delta=0, fill=0.5, graph=True, tables=True,
          k=16, backoff=8, copy=0.4, tmpl=0.1):
    return {"name": name, "do": "step", "b": b, "s": s, "corpus": corpus,
            "delta": delta, "fill": fill, "graph": graph, "tables": tables,
            "k": k, "backoff": backoff, "copy": copy, "tmpl": tmpl}


def listed():
    return [
        # One chat request without global memory, called eagerly: what a
        # single user waits for besides the model.
        _step("step_b1_s2048_eager", 1, 2048, graph=False),
        # The headline decode step: 64 requests, the memory full of
        # templated responses, half a delta of newer ones.
        _step("step_b64_s8192_global", 64, 8192, 1 << 22, 1 << 16,
              copy=0.0, tmpl=0.1),
        # A large server's step: many long rows that quote themselves, a
        # nearly full delta, three times as many workgroups as the chip has
        # CUs.
        _step("step_b256_s16384_global", 256, 16384, 1 << 20, 1 << 16,
              fill=0.95),
        # The same server with the global memory off.
        _step("step_b256_s16384_local", 256, 16384),
        # A few long-context requests (documents, agents): rows that do not
        # fit a CU's LDS.
        _step("step_b8_s131072_global", 8, 131072, 1 << 20, 1 << 16),
        # The headline step with the small-footprint index (no key rows, no
        # n-gram table), for servers that cannot spare 1 GB.
        _step("step_b64_s8192_compact", 64, 8192, 1 << 22, 1 << 16,
              tables=False, copy=0.0, tmpl=0.1),
        # A few finished requests a step, rows and lengths on the device;
        # every seventh harvest or so starts a rebuild of a small memory.
        {"name": "harvest_4rows_device", "do": "harvest", "rows": 4,
         "s": 4096, "corpus": 1 << 18, "delta": 1 << 16, "lo": 256,
         "hi": 2048, "device": True},
        # Sixteen finished requests at once into a full-size memory: append,
        # evict, rebuild and swap in one go.
        {"name": "harvest_rebuild_4m", "do": "harvest", "rows": 16,
         "s": 8192, "corpus": 1 << 22, "delta": 1 << 16, "lo": 2048,
         "hi": 3800, "device": False},
        # Suffix arrays from scratch: of one long document, and of a whole
        # corpus.
        {"name": "sa_61k", "do": "sa", "n": 61003, "kind": "copy"},
        {"name": "sa_4m", "do": "sa", "n": 4193511, "kind": "template"},
        # The operators below the classes, as a program that keeps its own
        # drafter classes calls them.
        {"name": "op_local_b64_s8192", "do": "local_op", "b": 64, "s": 8192,
         "c": 8, "r": 128, "k": 16},
        {"name": "op_sa_search_2048_4m", "do": "sa_op", "b": 64,
         "n": 4193511},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    do = rng.choice(["step", "step", "step", "harvest", "sa", "local_op",
                     "sa_op"])
    if do == "step":
        s = _log(rng, 512, 131072)
        b = _log(rng, 1, max(1, min(256, (1 << 22) // s)))
        on = rng.random() < 0.6
        c = _step("", b, s, _log(rng, 1 << 14, 1 << 22) if on else 0,
                  _log(rng, 1 << 12, 1 << 16) if on else 0,
                  round(rng.uniform(0.1, 0.95), 3),
                  graph=rng.random() < 0.7,
                  tables=not on or rng.random() < 0.8,
                  k=rng.choice([4, 8, 16]), backoff=rng.choice([1, 4, 8]),
                  copy=round(rng.uniform(0.0, 0.5), 3),
                  tmpl=round(rng.uniform(0.02, 0.15), 3))
        del c["name"]
        return c
    if do == "harvest":
        rows = rng.randint(1, 32)
        delta = _log(rng, 1 << 13, 1 << 16)
        per = delta // rows
        # half of the draws rebuild at every harvest
        lo, hi = ((0.5, 0.93) if rng.random() < 0.5 else (0.03, 0.15))
        return {"do": "harvest", "rows": rows, "s": max(16, per),
                "corpus": _log(rng, 1 << 17, 1 << 22), "delta": delta,
                "lo": max(4, math.ceil(lo * per) + 1),
                "hi": max(5, int(hi * per)), "device": rng.random() < 0.5}
    if do == "sa":
        return {"do": "sa", "n": _log(rng, 1 << 11, 4193511),
                "kind": rng.choice(["template", "copy", "uniform"])}
    if do == "local_op":
        s = _log(rng, 512, 65536)
        return {"do": "local_op", "b": _log(rng, 1, min(128, (1 << 20) // s)),
                "s": s, "c": rng.choice([1, 4, 8]),
                "r": rng.choice([32, 128]), "k": rng.choice([4, 8, 16])}
    return {"do": "sa_op", "b": _log(rng, 1, 128),
            "n": _log(rng, 1 << 14, 4193511)}


# ------------------------------------------------------------------- text
class _Text:
    """Seeded text on the GPU (see the module's description)."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(int(seed) * 7919 + 17)
        w = torch.arange(1, VOCAB + 1, dtype=torch.float64,
                         device=DEV) ** -1.1
        self.cdf = torch.cumsum(w / w.sum(), 0)
        self.perm = torch.randperm(VOCAB, generator=self.g,
                                   device=DEV).to(torch.int32)
        self.tmpl_len = torch.randint(32, 257, (64,), generator=self.g,
                                      device=DEV)
        self.tmpl = self.zipf(64 * 256).view(64, 256)

    def rand(self, *shape):
        return torch.rand(*shape, generator=self.g, device=DEV)

    def zipf(self, n):
        u = torch.rand(n, generator=self.g, device=DEV, dtype=torch.float64)
        r = torch.searchsorted(self.cdf, u).clamp_(max=VOCAB - 1)
        return self.perm[r]

    def rows(self, b, s, copy, tmpl):
        """[b, s] int32: spans of 8-64 fresh tokens, copies of 16-64 earlier
        tokens of the row, and template spans."""
        nseg = s // 8 + 2
        u = self.rand(b, nseg)
        kind = torch.where(u < copy, 1, torch.where(u < copy + tmpl, 2, 0))
        tid = (self.rand(b, nseg) * 64).long().clamp_(max=63)
        short = 8 + (self.rand(b, nseg) * 57).long().clamp_(max=56)
        ln = torch.where(kind == 2, self.tmpl_len[tid],
                         torch.where(kind == 1, short.clamp(min=16), short))
        end = ln.cumsum(1)
        start = end - ln
        # a copy needs its whole source before it
        kind = torch.where((kind == 1) & (start < ln), 0, kind)
        src = (self.rand(b, nseg).double() * (start - ln + 1).clamp(min=1)
               ).long()
        pos = torch.arange(s, device=DEV).expand(b, s).contiguous()
        seg = torch.searchsorted(end, pos, right=True)
        k = kind.gather(1, seg)
        off = pos - start.gather(1, seg)
        tok = self.zipf(b * s).view(b, s)
        tok = torch.where(k == 2, self.tmpl[tid.gather(1, seg),
                                            off.clamp(max=255)], tok)
        if copy > 0:
            at = torch.where(k == 1, src.gather(1, seg) + off, pos)
            while True:  # a copy of a copy: follow it to its first token
                nxt = at.gather(1, at)
                if bool((nxt == at).all()):
                    break
                at = nxt
            tok = tok.gather(1, at)
        return tok.contiguous()

    def docs(self, n, copy=0.0, tmpl=0.1, lo=1024, hi=8192):
        """Documents of lo..hi tokens, separators included n at most."""
        out, used = [], 0
        if n <= 2 * lo:
            lo, hi = max(2, n // 4), max(3, n // 2)
        lens = (lo + self.rand(max(4, 2 * n // lo)) * (hi - lo)).long()
        for x in lens.tolist():
            if used + x + 1 > n:
                break
            out.append(x)
            used += x + 1
        if copy > 0:
            t = self.rows(len(out), max(out), copy, tmpl)
            return [t[i, :x] for i, x in enumerate(out)]
        t = self.rows(1, sum(out), 0.0, tmpl)[0]
        return list(t.split(out))


def _counts(t, b, lo, hi):
    return (lo + t.rand(b).double() * (hi - lo + 1)).long().clamp_(
        max=hi).to(torch.int32)


# ---------------------------------------------------------------- prepare
def _prepare_step(c, t):
    b, s, k = c["b"], c["s"], c["k"]
    T = k + 1
    on = c["corpus"] > 0
    d = SuffixGPUDrafter(
        k=k, device=DEV, max_pattern_len=MAX_LEN, max_occurrences=128,
        num_backoff=c["backoff"], max_spec_factor=2.0, min_token_prob=0.1,
        enable_global=on, global_capacity=max(1, c["corpus"]),
        delta_capacity=max(1, c["delta"]),
        rebuild_threshold=max(1, c["delta"]),
        global_search_tables=c["tables"])
    if on:
        d.global_index.load_documents(t.docs(c["corpus"] - 1, tmpl=c["tmpl"]))
        d.global_index.append_documents(
            t.docs(max(8, int(c["delta"] * c["fill"])), tmpl=c["tmpl"]))
    full = t.rows(b, s + T, c["copy"], c["tmpl"])
    tokens = full[:, :s].contiguous()
    nt = _counts(t, b, max(1, s // 4), s - T)
    # accepted tokens of the last verification: geometric, at least one
    acc = 1 + (torch.log(t.rand(b).clamp(min=1e-9))
               / math.log(0.7)).long().clamp_(max=T - 1)
    j = torch.arange(T, device=DEV)
    nxt = full.gather(1, nt.long()[:, None] + j)
    sampled = torch.where(j < acc[:, None], nxt, -1).to(torch.int32)
    st = {"d": d, "tokens": tokens, "nt": nt, "sampled": sampled}
    if c["graph"]:
        d.propose_with_update(nt, tokens, sampled)  # before the capture
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            st["out"] = d.propose_with_update(nt, tokens, sampled)
        st["g"] = g
    return st


def _prepare_harvest(c, t):
    d = SuffixGPUDrafter(
        k=16, device=DEV, max_pattern_len=MAX_LEN, max_occurrences=128,
        max_spec_factor=2.0, min_token_prob=0.1, enable_global=True,
        global_capacity=c["corpus"], delta_capacity=c["delta"],
        rebuild_stream=torch.cuda.Stream() if c["device"] else None)
    gi = d.global_index
    gi.load_documents(t.docs(c["corpus"] - 1))
    tokens = t.rows(c["rows"], c["s"], 0.2, 0.1)
    ln = _counts(t, c["rows"], c["lo"], c["hi"])
    at = torch.randperm(c["rows"], generator=t.g, device=DEV).to(torch.int32)
    if c["device"]:
        # swaps at the poll after the harvest that started the rebuild
        gi.blocking_poll = True
    else:
        ln, at = ln.tolist(), at.tolist()
    return {"d": d, "tokens": tokens, "rows": at, "lens": ln}


def _text(c, t):
    if c["kind"] == "uniform":
        return torch.randint(0, 32000, (c["n"],), generator=t.g,
                             device=DEV, dtype=torch.int32)
    w = 8192
    n = -(-c["n"] // w)
    copy = 0.4 if c["kind"] == "copy" else 0.0
    return t.rows(n, w, copy, 0.1).view(-1)[:c["n"]].contiguous()


def _match_back(rows, pat):
    """Plain torch: [B, S] leading tokens of pat[b] (newest first) that end
    at each position of rows[b]."""
    b, s = rows.shape
    pad = torch.full((b, pat.shape[1]), -1, dtype=rows.dtype, device=DEV)
    x = torch.cat([pad, rows], 1)
    mb = torch.zeros(b, s, dtype=torch.int32, device=DEV)
    run = torch.ones(b, s, dtype=torch.bool, device=DEV)
    for i in range(pat.shape[1]):
        st = pat.shape[1] - 1 - i
        run &= x[:, st:st + s] == pat[:, i:i + 1]
        mb += run
    return mb


def _first(mb, thr, r):
    """Plain torch first r columns with mb >= thr: (pos [N, r], cnt [N])."""
    n, c = thr.shape
    hit = (mb[:, None, :] >= thr[:, :, None]) & (thr[:, :, None] > 0)
    hit = hit.view(n * c, -1)
    at = hit.long().cumsum(1) - 1
    row, col = (hit & (at < r)).nonzero(as_tuple=True)
    pos = torch.zeros(n * c, r, dtype=torch.int64, device=DEV)
    pos[row, at[row, col]] = col
    return pos, hit.sum(1).clamp(max=r)


def _prepare_local_op(c, t):
    b, s, r, k = c["b"], c["s"], c["r"], c["k"]
    rows = t.rows(b, s, 0.5, 0.1)
    pat = rows[:, -MAX_LEN:].flip(1).contiguous()
    mb = _match_back(rows, pat)
    # largest length with 2^i occurrences, the local support thresholds
    cnt = torch.stack([(mb >= x).sum(1) for x in range(1, MAX_LEN + 1)], 1)
    thr = torch.stack([(cnt >= 2 ** i).sum(1) for i in range(c["c"])], 1)
    pos, occ = _first(mb, thr, r)
    at = pos[:, :, None] + torch.arange(k, device=DEV)
    own = rows.repeat_interleave(c["c"], 0)
    cont = own.gather(1, at.clamp(max=s - 1).view(b * c["c"], -1))
    cont = torch.where(at < s, cont.view_as(at), -1).to(torch.int32)
    return {"rows": rows, "pat": pat, "thr": thr.view(-1).contiguous(),
            "cont": cont.contiguous(), "occ": occ, "k": k, "c": c["c"],
            "r": r, "s": s, "cap": (2 * thr.view(-1)).clamp(max=k)}


def _prepare_sa_op(c, t):
    n = c["n"]
    corpus = t.rows(1, n, 0.0, 0.1)[0]
    sa = torch.empty(n, dtype=torch.int32, device=DEV)
    build_suffix_array_into(corpus, n, sa)
    # every suffix length of each row's tail, left-aligned; half of the
    # tails are quoted from the corpus
    tail = t.rows(c["b"], MAX_LEN, 0.0, 0.1)
    at = (t.rand(c["b"]).double() * (n - MAX_LEN)).long()
    quote = corpus[at[:, None] + torch.arange(MAX_LEN, device=DEV)]
    tail = torch.where((torch.arange(c["b"], device=DEV) % 2 == 0)[:, None],
                       quote, tail)
    ln = torch.arange(1, MAX_LEN + 1, device=DEV)
    j = torch.arange(MAX_LEN, device=DEV)
    src = (MAX_LEN - ln[:, None] + j).clamp(max=MAX_LEN - 1)
    pat = torch.where(j < ln[:, None], tail[:, src], -1)
    return {"sa": sa, "corpus": corpus,
            "pat": pat.view(-1, MAX_LEN).to(torch.int32).contiguous(),
            "plen": ln.repeat(c["b"]).contiguous()}


def prepare(case, seed):
    t = _Text(seed)
    if case["do"] == "step":
        st = _prepare_step(case, t)
    elif case["do"] == "harvest":
        st = _prepare_harvest(case, t)
    elif case["do"] == "sa":
        st = {"text": _text(case, t)}
    elif case["do"] == "local_op":
        st = _prepare_local_op(case, t)
    else:
        st = _prepare_sa_op(case, t)
    st["do"] = case["do"]
    return st


# -------------------------------------------------------------------- run
def run(state):
    do = state["do"]
    if do == "step":
        if "g" in state:
            state["g"].replay()
            out = state["out"]
        else:
            out = state["d"].propose_with_update(
                state["nt"], state["tokens"], state["sampled"])
        return {"draft": out[0], "num_valid": out[1], "counts": out[2],
                "tokens": state["tokens"]}
    if do == "harvest":
        d = state["d"]
        d.harvest_finished(state["rows"], state["lens"], state["tokens"])
        d.poll()
        gi = d.global_index
        return {"corpus": gi.corpus, "sa": gi.sa, "delta": gi.delta,
                "delta_len": gi.delta_len_t}
    if do == "sa":
        return build_suffix_array(state["text"])
    if do == "local_op":
        mb = kernels.match_back(state["rows"], state["pat"], state["s"])
        pos, cnt = kernels.first_occurrences(mb, state["thr"], state["c"],
                                             state["r"])
        out = kernels.expand_chain(state["cont"], state["occ"], state["k"],
                                   0.1, state["cap"])
        return {"mb": mb, "pos": pos, "cnt": cnt, "chain": out[0],
                "num_valid": out[1], "num_emit": out[2], "score": out[3]}
    return kernels.sa_search(state["sa"], state["corpus"], state["pat"],
                             state["plen"])


# ------------------------------------------------------------------- work
def work(case):
    do = case["do"]
    if do == "step":
        b, k = case["b"], case["k"]
        # the rows' committed tokens, the sampled ids, the draft; with
        # global memory one candidate's continuations per row
        n = 4 * b * (0.625 * case["s"] + 2 * (k + 1) + k + 3)
        if case["corpus"]:
            n += 4 * b * 128 * (k + 1)
        return {"bytes": n, "flops": 0}
    if do == "harvest":
        new = case["rows"] * (case["lo"] + case["hi"]) / 2
        full = min(1.0, new / (case["delta"] / 2))  # rebuilds per pass
        # the documents copied; corpus and suffix array of a rebuild
        return {"bytes": 8 * new + full * (8 + 4) * case["corpus"],
                "flops": 0}
    if do == "sa":
        return {"bytes": 12 * case["n"], "flops": 0}
    if do == "local_op":
        b, s, r = case["b"], case["s"], case["r"]
        bc = b * case["c"]
        return {"bytes": 12 * b * s + bc * (8 * r + 4 * r * case["k"]),
                "flops": 0}
    b = case["b"] * MAX_LEN
    return {"bytes": b * (4 * MAX_LEN + 24
                          + 16 * math.log2(case["n"])), "flops": 0}


def tolerance(case):
    # Token ids, positions and counts; the one floating output (the chain
    # score) is a fixed sequence of IEEE fp32 operations in depth order.
    return "exact"


# ------------------------------------------------------------------ exact
def _suffix_array(text):
    n = text.numel()
    _, rank = torch.unique(text, return_inverse=True)
    h = 1
    while True:
        nxt = torch.zeros_like(rank)
        nxt[:max(0, n - h)] = rank[h:] + 1
        key = rank * (n + 1) + nxt
        sa = torch.argsort(key, stable=True)
        ks = key[sa]
        new = torch.zeros(n, dtype=torch.int64, device=DEV)
        new[1:] = (ks[1:] != ks[:-1]).long().cumsum(0)
        rank = torch.empty_like(new)
        rank[sa] = new
        h *= 2
        if int(new[-1]) == n - 1:
            return sa


def _expand(cont, occ, k, min_prob, cap):
    """Majority-vote chains in 64 bits."""
    n, r, _ = cont.shape
    cont = cont.long()
    on = torch.arange(r, device=DEV) < occ[:, None]
    cum = torch.ones(n, dtype=torch.float64, device=DEV)
    score = torch.zeros_like(cum)
    chain = torch.full((n, k), -1, dtype=torch.int64, device=DEV)
    lowest = float(np.float32(min_prob)) * (1 - 1e-6)
    alive = torch.ones(n, dtype=torch.bool, device=DEV)
    for d in range(k):
        v = cont[:, :, d]
        act = on & (v != -1)
        votes = ((v[:, :, None] == v[:, None, :]) & act[:, None, :]).sum(2)
        votes = torch.where(act, votes, 0)
        top = votes.max(1).values
        tok = torch.where(act & (votes == top[:, None]), v,
                          2 ** 40).min(1).values
        cum = cum * (top.double() / act.sum(1).clamp(min=1))
        alive &= (top > 0) & (cum >= lowest)
        chain[:, d] = torch.where(alive, tok, -1)
        score += torch.where(alive & (cap > d), cum, 0.0)
        on = on & (v == tok[:, None]) & alive[:, None]
    nv = (chain != -1).sum(1)
    return chain, nv, torch.minimum(nv, cap.clamp(min=0)), score


def exact(case, seed):
    """The operators and suffix arrays in plain torch.  The steps' and the
    harvests' outputs are whole numbers that only a restatement of the whole
    drafter would give."""
    if case["do"] == "sa":
        return _suffix_array(_text(case, _Text(seed)))
    if case["do"] != "local_op":
        return None
    st = _prepare_local_op(case, _Text(seed))
    mb = _match_back(st["rows"], st["pat"])
    pos, cnt = _first(mb, st["thr"].view(case["b"], case["c"]), case["r"])
    out = _expand(st["cont"], st["occ"], st["k"], 0.1, st["cap"])
    return {"mb": mb, "pos": pos, "cnt": cnt, "chain": out[0],
            "num_valid": out[1], "num_emit": out[2], "score": out[3]}
