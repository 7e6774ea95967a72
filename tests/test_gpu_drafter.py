"""Whole drafter on gfx950 vs the oracle: local+global decode steps on the
synthetic workloads, HIP-graph capture and replay, serial vs parallel
paths, and the reference's speculative-loop verification tests."""

from __future__ import annotations

import random

import numpy as np
import pytest
import torch

from oracle.drafter import DrafterOracle
from suffixgpu_amd import synth

pytestmark = pytest.mark.gpu

I32 = np.int32


def T(a, dev, dtype=None):
    t = torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    return t if dtype is None else t.to(dtype)


def N(t):
    return t.cpu().numpy()


GLOBAL_KW = dict(k=16, max_pattern_len=32, max_occurrences=128,
                 num_backoff=8, max_spec_factor=2.0, min_token_prob=0.1,
                 enable_global=True, global_capacity=1 << 16,
                 delta_capacity=1 << 12, rebuild_threshold=1 << 30)


def _global_pair(gpu, seed=3, b=24, s=2048, **over):
    from suffixgpu_amd import SuffixGPUDrafter
    kw = dict(GLOBAL_KW)
    kw.update(over)
    w = synth.global_corpus(seed=seed, capacity=kw["global_capacity"],
                            delta_fill=kw["delta_capacity"] // 2, n_docs=40,
                            b=b, s=s, seq_hi=1500)
    d = SuffixGPUDrafter(device=gpu, **kw)
    o = DrafterOracle(**kw)
    d.global_index.load_documents([T(x, gpu) for x in w.active_docs])
    o.global_index.load_documents(w.active_docs)
    d.global_index.append_documents([T(x, gpu) for x in w.delta_docs])
    o.global_index.append_documents(w.delta_docs)
    return w, d, o


def test_global_step_split_delta_vs_oracle(gpu):
    """A 2^16 delta capacity splits every row's delta scan over several
    workgroups of the fused step (B=24 rows)."""
    w, d, o = _global_pair(gpu, seed=6, delta_capacity=1 << 16)
    assert d.global_index.delta_len > 20000
    bt = w.batch
    tg = T(bt.tokens, gpu)
    draft, nv, new = d.propose_with_update(T(bt.num_tokens, gpu), tg,
                                           T(bt.sampled, gpu))
    to = bt.tokens.copy()
    ed, env, enew = o.propose_with_update(bt.num_tokens, to, bt.sampled)
    np.testing.assert_array_equal(N(new), enew)
    np.testing.assert_array_equal(N(draft), ed)
    np.testing.assert_array_equal(N(nv), env)


def test_global_step_vs_oracle(gpu):
    w, d, o = _global_pair(gpu)
    bt = w.batch
    tg = T(bt.tokens, gpu)
    draft, nv, new = d.propose_with_update(T(bt.num_tokens, gpu), tg,
                                           T(bt.sampled, gpu))
    to = bt.tokens.copy()
    ed, env, enew = o.propose_with_update(bt.num_tokens, to, bt.sampled)
    np.testing.assert_array_equal(N(tg), to)
    np.testing.assert_array_equal(N(new), enew)
    np.testing.assert_array_equal(N(draft), ed)
    np.testing.assert_array_equal(N(nv), env)
    assert (env > 0).sum() > 0
    # plain propose with a mask, and max_model_len / valid counts
    mask = np.arange(bt.tokens.shape[0]) % 3 != 0
    draft, nv = d.propose(new, tg, T(mask, gpu))
    ed, env = o.propose(enew, to, mask)
    np.testing.assert_array_equal(N(draft), ed)
    np.testing.assert_array_equal(N(nv), env)
    vc = np.minimum((bt.sampled != -1).sum(1), 2).astype(np.int64)
    draft, nv, new = d.propose_with_update(new, tg, T(bt.sampled, gpu),
                                           T(vc, gpu), max_model_len=1500)
    ed, env, enew = o.propose_with_update(enew, to, bt.sampled, vc,
                                          max_model_len=1500)
    np.testing.assert_array_equal(N(tg), to)
    np.testing.assert_array_equal(N(draft), ed)
    np.testing.assert_array_equal(N(nv), env)
    np.testing.assert_array_equal(N(new), enew)


def test_global_step_patterns_past_key_rows_vs_oracle(gpu):
    """Patterns of up to 48 tokens against 32-token key rows: a search
    probe whose row ties with the pattern finishes the comparison in the
    corpus.  The template corpus has matches longer than the rows."""
    from oracle.sa import suffix_match_backoff
    p = 48
    w, d, o = _global_pair(gpu, seed=5, max_pattern_len=p, num_backoff=5)
    bt = w.batch
    gi = o.global_index
    # the SA match lengths of the rows' tails, as the step will see them
    # after the update: some pass the key rows' 32 tokens
    q = np.zeros((bt.tokens.shape[0], p), dtype=np.int32)
    ql = np.zeros(bt.tokens.shape[0], dtype=np.int64)
    for i in range(bt.tokens.shape[0]):
        acc = int((bt.sampled[i] != -1).sum())
        ctx = np.concatenate([bt.tokens[i, :bt.num_tokens[i]],
                              bt.sampled[i, :acc]])
        n = min(len(ctx), p)
        q[i, :n] = ctx[len(ctx) - n:]
        ql[i] = n
    sa_len, _, _ = suffix_match_backoff(gi.sa, gi.corpus, q, ql, p,
                                        np.array([p], dtype=np.int64))
    assert (sa_len[:, 0] > 32).sum() >= 4, sa_len[:, 0]
    tg = T(bt.tokens, gpu)
    draft, nv, new = d.propose_with_update(T(bt.num_tokens, gpu), tg,
                                           T(bt.sampled, gpu))
    to = bt.tokens.copy()
    ed, env, enew = o.propose_with_update(bt.num_tokens, to, bt.sampled)
    np.testing.assert_array_equal(N(new), enew)
    np.testing.assert_array_equal(N(draft), ed)
    np.testing.assert_array_equal(N(nv), env)


def test_serial_equals_parallel_paths(gpu):
    w, d, o = _global_pair(gpu)
    d2, _, _ = None, None, None
    from suffixgpu_amd import SuffixGPUDrafter
    kw = dict(GLOBAL_KW)
    d2 = SuffixGPUDrafter(device=gpu, parallel_paths=False, **kw)
    d2.global_index.load_documents([T(x, gpu) for x in w.active_docs])
    d2.global_index.append_documents([T(x, gpu) for x in w.delta_docs])
    bt = w.batch
    outs = []
    for dr in (d, d2):
        tg = T(bt.tokens, gpu)
        outs.append([N(x) for x in dr.propose_with_update(
            T(bt.num_tokens, gpu), tg, T(bt.sampled, gpu))] + [N(tg)])
    for a, b in zip(*outs):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("enable_global", [False, True])
def test_graph_capture_replay(gpu, enable_global):
    """A captured propose_with_update step replays identically to eager,
    across replays with eager work and syncs in between."""
    kw = {} if enable_global else dict(enable_global=False)
    w, d, o = _global_pair(gpu, **kw) if enable_global else (None, None, None)
    if not enable_global:
        from suffixgpu_amd import SuffixGPUDrafter
        wl = synth.local_zipf(seed=2, b=16, s=4096)
        kwl = dict(GLOBAL_KW)
        kwl["enable_global"] = False
        d = SuffixGPUDrafter(device=gpu, **kwl)
        tokens, nt, sampled = wl.tokens, wl.num_tokens, wl.sampled
    else:
        tokens, nt = w.batch.tokens, w.batch.num_tokens
        sampled = w.batch.sampled
    buf = T(tokens, gpu)
    ntg = T(nt, gpu)
    sg = T(sampled, gpu)
    # eager reference on a copy
    ref_buf = buf.clone()
    ref = d.propose_with_update(ntg.clone(), ref_buf, sg)
    ref = [N(x) for x in ref]
    # warm up on scratch state, then capture
    for _ in range(2):
        d.propose_with_update(ntg.clone(), buf.clone(), sg)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    nt_static = ntg.clone()
    with torch.cuda.graph(g):
        out = d.propose_with_update(nt_static, buf, sg)
    for rep in range(4):
        nt_static.copy_(ntg)
        buf.copy_(T(tokens, gpu))
        g.replay()
        torch.cuda.synchronize()
        for a, b in zip(out, ref):
            np.testing.assert_array_equal(N(a), b, err_msg=f"replay {rep}")
        np.testing.assert_array_equal(N(buf), N(ref_buf))
        _ = torch.arange(1000, device=gpu).sum().item()  # eager work


# ------------------------------------------- reference verification loops
def _make(gpu, enable_global=True):
    from suffixgpu_amd import SuffixGPUDrafter
    return SuffixGPUDrafter(k=4, device=gpu, max_pattern_len=8,
                            max_occurrences=16, enable_global=enable_global,
                            global_capacity=1 << 16, delta_capacity=1 << 12,
                            rebuild_threshold=1 << 10)


def _adapter_propose(d, buf, nts, pending):
    n = len(pending)
    buf[0, nts:nts + n] = torch.tensor(pending, dtype=torch.int32,
                                       device=buf.device)
    return d.propose(torch.tensor([nts + n], dtype=torch.int32,
                                  device=buf.device), buf)


def _repetitive_doc(seed, n_blocks=12):
    g = random.Random(seed)
    blocks = [[g.randint(0, 5) for _ in range(6)] for _ in range(4)]
    doc = []
    for _ in range(n_blocks):
        doc.extend(g.choice(blocks))
    return doc


def _nonrepeating_doc(seed, n=30):
    g = random.Random(seed)
    doc = []
    while len(doc) < n:
        t = g.randint(0, 15)
        if len(doc) >= 2 and any(doc[i] == doc[-2] and doc[i + 1] == doc[-1]
                                 and doc[i + 2] == t
                                 for i in range(len(doc) - 2)):
            continue
        doc.append(t)
    return doc


def _spec_loop(d, doc, prompt_len, gpu):
    prompt = doc[:prompt_len]
    target = len(doc) - prompt_len
    buf = torch.zeros(1, len(doc) + 12, dtype=torch.int32, device=gpu)
    buf[0, :prompt_len] = torch.tensor(prompt, dtype=torch.int32)
    gen, pending, steps, acc = [], [doc[prompt_len]], 0, 0
    while len(gen) < target:
        steps += 1
        assert steps < 10000
        draft, nv = _adapter_propose(d, buf, prompt_len + len(gen), pending)
        gen.extend(pending)
        if len(gen) >= target:
            break
        base = prompt_len + len(gen)
        a = 0
        dl = N(draft)[0]
        while a < int(nv[0]) and base + a < len(doc) and dl[a] == doc[base + a]:
            a += 1
        acc += a
        pending = [int(dl[i]) for i in range(a)]
        if base + a < len(doc):
            pending.append(doc[base + a])
        else:
            gen.extend(pending)
            break
    return gen[:target], steps, acc, buf


def test_spec_loop_exact_local(gpu):
    doc = _repetitive_doc(7)
    gen, steps, acc, _ = _spec_loop(_make(gpu, False), doc, 4, gpu)
    assert gen == doc[4:]
    assert steps < len(doc) - 4 and acc > 0


@pytest.mark.parametrize("seed", [0, 1, 2])
def test_spec_loop_exact_random(gpu, seed):
    doc = _nonrepeating_doc(seed, 48)
    gen, _, _, _ = _spec_loop(_make(gpu, False), doc, 6, gpu)
    assert gen == doc[6:]


def test_global_warmup_improves_acceptance(gpu):
    d = _make(gpu)
    doc = _nonrepeating_doc(11, 32)
    accs = []
    for _ in range(2):
        gen, _, acc, buf = _spec_loop(d, doc, 4, gpu)
        assert gen == doc[4:]
        d.harvest_rows([buf[0]], [4 + len(gen)])
        accs.append(acc)
    assert accs[1] > accs[0] and accs[1] >= 8


def test_ingest_then_cross_request_draft(gpu):
    from suffixgpu_amd import SuffixGPUDrafter
    d = SuffixGPUDrafter(k=4, device=gpu, max_pattern_len=8,
                         max_occurrences=8, enable_global=True,
                         global_capacity=1024, delta_capacity=256,
                         rebuild_threshold=100000)
    phrase = [11, 12, 13, 14, 15, 16, 17, 18]
    resp = torch.tensor(phrase * 8, dtype=torch.int32, device=gpu)
    d.ingest_active(["a"], [resp], [len(resp)], chunk=16)
    buf = torch.zeros(1, 32, dtype=torch.int32, device=gpu)
    cur = [99, 98] + phrase[:6]
    buf[0, :len(cur)] = torch.tensor(cur, dtype=torch.int32)
    draft, nv = d.propose(torch.tensor([len(cur)], dtype=torch.int32,
                                       device=gpu), buf,
                          torch.ones(1, dtype=torch.bool, device=gpu))
    n = int(nv[0])
    assert n > 0 and N(draft)[0, :n].tolist() == (phrase[6:] + phrase)[:n]


@pytest.mark.parametrize("enable_global", [False, True])
def test_step_long_rows_vs_oracle(gpu, enable_global):
    """Rows of 40000 tokens, which do not fit LDS, with and without the
    global index (with it they take the match launch, without it the
    1024-thread local-only kernel streams them): rows are windows of the
    document stream at committed lengths around the 16384-position chunk
    boundaries of a streamed row."""
    from suffixgpu_amd import SuffixGPUDrafter
    s, t = 40000, 17
    w, d, o = _global_pair(gpu, seed=9, b=4, s=2048)
    if not enable_global:
        kw = dict(GLOBAL_KW, enable_global=False)
        d, o = SuffixGPUDrafter(device=gpu, **kw), DrafterOracle(**kw)
    stream = np.concatenate(w.active_docs + w.delta_docs).astype(I32)
    rng = np.random.default_rng(9)
    q_list = [0, 3, 16384, 16385, 20000, 39990, s - t, s]
    b = len(q_list)
    rows = np.zeros((b, s), dtype=I32)
    sampled = np.full((b, t), -1, dtype=I32)
    for i, q in enumerate(q_list):
        off = int(rng.integers(0, stream.shape[0] - s - t))
        rows[i] = stream[off:off + s]
        acc = int(rng.integers(0, t + 1))
        sampled[i, :acc] = stream[off + q:off + q + acc][:acc]
    nt = np.array(q_list, dtype=I32)
    tg = T(rows, gpu)
    draft, nv, new = d.propose_with_update(T(nt, gpu), tg, T(sampled, gpu))
    to = rows.copy()
    ed, env, enew = o.propose_with_update(nt, to, sampled)
    np.testing.assert_array_equal(N(tg), to)
    np.testing.assert_array_equal(N(new), enew)
    np.testing.assert_array_equal(N(draft), ed)
    np.testing.assert_array_equal(N(nv), env)
    assert (env > 0).sum() > 0


@pytest.mark.parametrize("entry", ["step", "noalloc", "rows"])
def test_long_rows_with_index_by_entry_point(gpu, entry):
    """Rows of 40000 tokens with an index through each entry point of the
    step -- without scratch one workgroup streams a row, with it the match
    launch spreads them -- against the oracle."""
    from suffixgpu_amd import _lib
    L = _lib.lib()
    s, t = 40000, 17
    w, d, o = _global_pair(gpu, seed=9, b=4, s=2048)
    stream = np.concatenate(w.active_docs + w.delta_docs).astype(I32)
    rng = np.random.default_rng(10)
    nt = np.array([0, 4096, 16384, 20000, s - t, s], I32)
    b = len(nt)
    rows = np.zeros((b, s), dtype=I32)
    sampled = np.full((b, t), -1, dtype=I32)
    for i, q in enumerate(nt):
        off = int(rng.integers(0, stream.shape[0] - s - t))
        rows[i] = stream[off:off + s]
        acc = int(rng.integers(1, t + 1))
        sampled[i, :acc] = stream[off + q:off + q + acc]
    to = rows.copy()
    exp = o.propose_with_update(nt, to, sampled)
    dev = T(rows, gpu)
    bt, keep = _lib.make_batch(dev, T(nt, gpu), sampled=T(sampled, gpu),
                               limit=s)
    out = [torch.full((b, d.k), -9, dtype=torch.int32, device=gpu),
           torch.full((b,), -9, dtype=torch.int32, device=gpu),
           torch.full((b,), -9, dtype=torch.int32, device=gpu)]
    args = [d._params, d.global_index.index_struct(), bt,
            *[x.data_ptr() for x in out]]
    cur = torch.cuda.current_stream().cuda_stream
    ws = d._workspace(b, cur)
    n = int(L.sfx_row_scratch_size(d._params, b, s))
    scratch = torch.full((n,), 0x5b, dtype=torch.uint8, device=gpu)
    if entry == "noalloc":
        rc = L.sfx_propose_step_noalloc(*args, cur)
    elif entry == "step":
        rc = L.sfx_propose_step(*args, ws.data_ptr(), ws.numel(), cur)
    else:
        rc = L.sfx_propose_step_rows(*args, ws.data_ptr(), ws.numel(),
                                     scratch.data_ptr(), n, cur)
    assert rc == 0 and n > 0
    torch.cuda.synchronize()
    del keep
    for g, e in zip((*out, dev), (*exp, to)):
        np.testing.assert_array_equal(N(g), e)
    assert (exp[1] > 0).sum() >= 3


@pytest.mark.parametrize("s", [8192, 16384])
def test_step_dense_grid_vs_oracle(gpu, s):
    """B=100 rows with global memory on make a grid of 300 workgroups,
    more than the CUs: the step then sizes every role for two workgroups
    per CU (at S=16384 the local role streams its row)."""
    w, d, o = _global_pair(gpu, seed=11, b=100, s=s)
    bt = w.batch
    tg = T(bt.tokens, gpu)
    draft, nv, new = d.propose_with_update(T(bt.num_tokens, gpu), tg,
                                           T(bt.sampled, gpu))
    to = bt.tokens.copy()
    ed, env, enew = o.propose_with_update(bt.num_tokens, to, bt.sampled)
    np.testing.assert_array_equal(N(tg), to)
    np.testing.assert_array_equal(N(new), enew)
    np.testing.assert_array_equal(N(draft), ed)
    np.testing.assert_array_equal(N(nv), env)
    assert (env > 0).sum() > 10


@pytest.mark.parametrize("b", [180, 256])
def test_step_wave_grid_split_delta_vs_oracle(gpu, b):
    """Batches whose grid runs in waves (3 B > 512) split a 2^16-capacity
    delta over several parts within 1024 workgroups (B=180: 3 parts, 900
    workgroups; B=256: 2 parts, 1024), dispatched by role."""
    w, d, o = _global_pair(gpu, seed=12, b=b, s=2048,
                           delta_capacity=1 << 16)
    assert d.global_index.delta_len > 30000
    bt = w.batch
    tg = T(bt.tokens, gpu)
    draft, nv, new = d.propose_with_update(T(bt.num_tokens, gpu), tg,
                                           T(bt.sampled, gpu))
    to = bt.tokens.copy()
    ed, env, enew = o.propose_with_update(bt.num_tokens, to, bt.sampled)
    np.testing.assert_array_equal(N(tg), to)
    np.testing.assert_array_equal(N(new), enew)
    np.testing.assert_array_equal(N(draft), ed)
    np.testing.assert_array_equal(N(nv), env)
    assert (env > 0).sum() > b // 2


def _rows_step(gpu, p, tokens, nt, sampled, mask, scratch):
    """One local-only step through the C ABI, with or without row scratch."""
    from suffixgpu_amd import _lib
    L = _lib.lib()
    b, s = tokens.shape
    rows = T(tokens, gpu)
    bt, keep = _lib.make_batch(
        rows, T(nt, gpu), sampled=None if sampled is None else T(sampled, gpu),
        mask=None if mask is None else T(mask, gpu), limit=s)
    out = [torch.full((b, p.k), -9, dtype=torch.int32, device=gpu),
           torch.full((b,), -9, dtype=torch.int32, device=gpu),
           torch.full((b,), -9, dtype=torch.int32, device=gpu)]
    n = int(L.sfx_row_scratch_size(p, b, s))
    assert n > 0, "the rows fit LDS"
    # whatever the memory held before must not matter
    ws = torch.full((n,), 0x5b, dtype=torch.uint8, device=gpu)
    cur = torch.cuda.current_stream().cuda_stream
    rc = L.sfx_propose_step_rows(
        p, None, bt, *[o.data_ptr() for o in out], None, 0,
        ws.data_ptr() if scratch else None, n if scratch else 0, cur)
    assert rc == 0
    torch.cuda.synchronize()
    del keep
    return [N(o) for o in out] + [N(rows)]


@pytest.mark.parametrize("s,P,R,C", [
    (40960, 32, 128, 8), (40963, 32, 128, 8), (70001, 1, 16, 8),
    (36866, 3, 128, 8), (40960, 5, 4, 1), (40960, 64, 128, 8),
    (40960, 65, 128, 32), (36865, 255, 300, 8), (12290, 32, 2000, 8),
    (266240, 32, 128, 8), (300001, 7, 2, 8)])
def test_split_rows_match_streamed(gpu, s, P, R, C):
    """Rows split over the chip against the same rows streamed by one
    workgroup each: counts at the edges of parts, sampled ids across an
    edge and with gaps, row lengths off the 4-token grid, more than one
    chunk of 64 parts, matches of every length up to P."""
    from suffixgpu_amd import _lib
    rng = np.random.default_rng(s + P)
    p = _lib.make_params(16, P, R, 1, [1 << min(i, 14) for i in range(C)],
                         (), 2.0, 0.0, 0.1, 0.0)
    part = 4096
    nt = np.array([0, 1, part - 3, part, part + 1, 2 * part - 2, 3 * part,
                   s - 17, s - 5, s, s // 2], I32)
    b = len(nt)
    tokens = rng.integers(0, 3, size=(b, s)).astype(I32)
    tokens[3] = 7                                  # one token throughout
    tokens[4] = np.arange(s) % 5                   # periodic
    tokens[5] = rng.integers(0, 1 << 30, size=s)   # no matches
    half = rng.integers(0, 50, size=900)
    tokens[7] = np.resize(half, s)                 # long repeats
    tokens[10, : s // 3] = 9
    sampled = np.full((b, 17), -1, I32)
    for i in range(b):
        n = rng.integers(1, 17)
        sampled[i, :n] = tokens[i, rng.integers(0, s - 20):][:n]
    sampled[2, 5] = -1
    sampled[6] = -1                                # nothing accepted
    for smp, mask in ((sampled, None),
                      (None, np.arange(b) % 4 != 2), (None, None)):
        got = _rows_step(gpu, p, tokens, nt, smp, mask, True)
        exp = _rows_step(gpu, p, tokens, nt, smp, mask, False)
        for g, e in zip(got, exp):
            np.testing.assert_array_equal(g, e)
    assert (exp[1] > 0).sum() >= 4


@pytest.mark.parametrize("over", [-1, 0])
def test_local_rows_around_the_split_length(gpu, over):
    """A local-only drafter on either side of the row length from which its
    steps take the match launch, against the oracle."""
    from suffixgpu_amd import SuffixGPUDrafter
    from suffixgpu_amd.proposer import SPLIT_MIN_LOCAL
    s = SPLIT_MIN_LOCAL + over
    rng = np.random.default_rng(s)
    kw = dict(k=8, max_pattern_len=16, max_occurrences=32, num_backoff=6,
              max_spec_factor=2.0, min_token_prob=0.05)
    d = SuffixGPUDrafter(device=gpu, **kw)
    o = DrafterOracle(**kw)
    assert (s >= d._split_seq) == (over == 0)
    rows = np.resize(rng.integers(0, 40, 7000), (3, s)).astype(I32)
    rows[1] = rng.integers(0, 5, s)
    nt = np.array([s - 20, s // 2, 4097], I32)
    sampled = np.full((3, 9), -1, I32)
    sampled[0, :4] = rows[0, nt[0]:nt[0] + 4]
    sampled[1, :2] = 3
    sampled[2, :1] = rows[2, nt[2]]
    dev = T(rows, gpu)
    draft, nv, cnt = d.propose_with_update(T(nt, gpu), dev, T(sampled, gpu))
    exp_rows = rows.copy()
    exp = o.propose_with_update(nt, exp_rows, sampled)
    for g, e in zip((draft, nv, cnt), exp):
        np.testing.assert_array_equal(N(g), e)
    np.testing.assert_array_equal(N(dev), exp_rows)


@pytest.mark.parametrize("s,scratch", [(9000, False), (40960, False),
                                       (40960, True)])
def test_local_step_counts_in_place(gpu, s, scratch):
    """Local-only steps whose new counts are written over the counts they
    start from: rows in LDS, streamed and split, drafting and masked.  The
    only occurrence of each row's tail ends at the row's last tokens, so a
    count taken twice shows in the draft."""
    from suffixgpu_amd import _lib
    L = _lib.lib()
    rng = np.random.default_rng(s)
    kw = dict(k=8, max_pattern_len=16, max_occurrences=32, num_backoff=6,
              max_spec_factor=2.0, min_token_prob=0.05)
    p = _lib.make_params(8, 16, 32, 1, [1 << i for i in range(6)], (), 2.0,
                         0.0, 0.05, 0.0)
    b = 24
    rows = np.tile(np.arange(s), (b, 1)).astype(I32)
    nt = rng.integers(s // 2, s - 10, b).astype(I32)
    sampled = np.full((b, 9), -1, I32)
    for i in range(b):
        n = i % 4                       # none accepted: masked
        rows[i, nt[i] - 4:nt[i]] = s + np.arange(4)
        sampled[i, :n] = s + np.arange(n)
    exp_rows = rows.copy()
    exp = DrafterOracle(**kw).propose_with_update(nt, exp_rows, sampled)
    dev, counts = T(rows, gpu), T(nt, gpu)
    bt, keep = _lib.make_batch(dev, counts, sampled=T(sampled, gpu), limit=s)
    assert bt.num_tokens == counts.data_ptr()
    draft = torch.full((b, 8), -9, dtype=torch.int32, device=gpu)
    nv = torch.full((b,), -9, dtype=torch.int32, device=gpu)
    n = int(L.sfx_row_scratch_size(p, b, s))
    assert (n > 0) == (s > 30000)
    ws = torch.empty(n if scratch else 0, dtype=torch.uint8, device=gpu)
    _lib.check(L.sfx_propose_step_rows(
        p, None, bt, draft.data_ptr(), nv.data_ptr(), counts.data_ptr(),
        None, 0, _lib.ptr(ws) if scratch else None, ws.numel(),
        torch.cuda.current_stream().cuda_stream), "step")
    torch.cuda.synchronize()
    del keep
    for g, e in zip((draft, nv, counts, dev), (*exp, exp_rows)):
        np.testing.assert_array_equal(N(g), e)


def test_split_rows_share_the_match_launch(gpu):
    """More parts than the match launch has workgroups: each takes several
    parts of its row, over rows from empty to full, against the same rows
    streamed by one workgroup each."""
    from suffixgpu_amd import _lib
    b, s = 300, 40962
    rng = np.random.default_rng(b)
    p = _lib.make_params(16, 32, 128, 1, [1 << i for i in range(8)], (), 2.0,
                         0.0, 0.1, 0.0)
    tokens = rng.integers(0, 3, size=(b, s)).astype(I32)
    tokens[::7] = np.resize(rng.integers(0, 50, size=900), s)
    nt = rng.integers(0, s - 20, b).astype(I32)
    nt[:5] = (0, 1, 4096, 8193, s)
    sampled = np.full((b, 17), -1, I32)
    for i in range(b):
        n = rng.integers(0, 17)
        sampled[i, :n] = tokens[i, rng.integers(0, s - 20):][:n]
    got = _rows_step(gpu, p, tokens, nt, sampled, None, True)
    exp = _rows_step(gpu, p, tokens, nt, sampled, None, False)
    for g, e in zip(got, exp):
        np.testing.assert_array_equal(g, e)
    assert (exp[1] > 0).sum() > b // 2


@pytest.mark.parametrize("enable_global", [False, True])
def test_split_seq_is_the_callers_choice(gpu, enable_global):
    """A drafter told never to take the match launch streams the rows that
    it would split, eagerly and in a capture, with equal results."""
    s = 50000
    w, d, o = _global_pair(gpu, seed=9, b=4, s=2048)
    if not enable_global:
        from suffixgpu_amd import SuffixGPUDrafter
        d = SuffixGPUDrafter(device=gpu, **dict(GLOBAL_KW,
                                                enable_global=False))
    assert d.split_seq <= s
    rng = np.random.default_rng(s)
    rows = np.resize(rng.integers(0, 40, 7000), (3, s)).astype(I32)
    nt = np.array([s - 20, s // 2, 4097], I32)
    sampled = np.full((3, 9), -1, I32)
    for i in range(3):
        sampled[i, :4] = rows[i, nt[i]:nt[i] + 4]
    dev = [T(x, gpu) for x in (nt, rows, sampled)]
    exp = [N(x) for x in d.propose_with_update(*dev)]
    graphs = []
    for seq in (d.split_seq, 1 << 30):
        d.split_seq = seq
        for g, e in zip(d.propose_with_update(*dev), exp):
            np.testing.assert_array_equal(N(g), e)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            out = d.propose_with_update(*dev)
        graphs.append((g, out))
    # replays over other rows than the captured ones, in turn
    for shift in (1, 2, 3):
        cur = np.roll(rows, shift, axis=0)
        for g, out in graphs:
            dev[1].copy_(T(cur, gpu))
            g.replay()
            torch.cuda.synchronize()
            fresh = d.propose_with_update(dev[0], T(cur, gpu), dev[2])
            for a, e in zip(out, fresh):
                np.testing.assert_array_equal(N(a), N(e))
    assert (exp[1] > 0).any()


@pytest.mark.parametrize("b,s", [(12, 40000), (100, 28000), (180, 27002)])
def test_rows_held_and_split_in_one_step(gpu, b, s):
    """Rows on either side of the length that a step with split rows holds
    in LDS, in one batch with an index, at one, two and three workgroups per
    CU: against the same rows without scratch."""
    from suffixgpu_amd import _lib
    L = _lib.lib()
    w, d, o = _global_pair(gpu, seed=9, b=4, s=2048)
    t = 17
    rng = np.random.default_rng(b)
    stream = np.concatenate(w.active_docs + w.delta_docs).astype(I32)
    stream = np.resize(stream, max(stream.shape[0], 2 * s))
    rows = np.zeros((b, s), I32)
    sampled = np.full((b, t), -1, I32)
    nt = rng.integers(0, s - t, b).astype(I32)
    nt[:11] = (0, 1, 4095, 4096, 4097, 8175, 8190, 8191, 8192, 8193, s - t)
    nt[11:b // 2] = rng.integers(1, 8300, max(0, b // 2 - 11))
    for i in range(b):
        off = int(rng.integers(0, stream.shape[0] - s))
        rows[i] = stream[off:off + s]
        acc = int(rng.integers(0, t + 1))
        sampled[i, :acc] = rows[i, nt[i]:nt[i] + acc]
    cur = torch.cuda.current_stream().cuda_stream
    n = int(L.sfx_row_scratch_size(d._params, b, s))
    assert n > 0
    results = []
    for scratch in (n, 0):
        dev = T(rows, gpu)
        bt, keep = _lib.make_batch(dev, T(nt, gpu), sampled=T(sampled, gpu),
                                   limit=s)
        out = [torch.full((b, d.k), -9, dtype=torch.int32, device=gpu),
               torch.full((b,), -9, dtype=torch.int32, device=gpu),
               torch.full((b,), -9, dtype=torch.int32, device=gpu)]
        ws = d._workspace(b, cur)
        mem = torch.full((n,), 0x5b, dtype=torch.uint8, device=gpu)
        _lib.check(L.sfx_propose_step_rows(
            d._params, d.global_index.index_struct(), bt,
            *[x.data_ptr() for x in out], ws.data_ptr(), ws.numel(),
            mem.data_ptr(), scratch, cur), "step")
        torch.cuda.synchronize()
        del keep
        results.append([N(x) for x in (*out, dev)])
    for g, e in zip(*results):
        np.testing.assert_array_equal(g, e)
    assert (results[0][1] > 0).sum() > b // 3
