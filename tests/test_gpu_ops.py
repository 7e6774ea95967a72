"""HIP operators vs the oracle: scatter, match_back, first occurrences,
SA build and search, majority-vote expansion (bit-exact; weighted-vote
scores within rtol 1e-5, the tolerance the path is held to; the
reference's own test allows 1e-4)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import naive
from oracle.drafter import DrafterOracle
from oracle.expand import expand_chain as o_expand
from oracle.local import first_occurrences as o_first_occ
from oracle.local import match_back as o_match_back
from oracle.local import newest_first_pattern
from oracle.sa import build_suffix_array as o_build_sa
from oracle.sa import search_interval as o_search
from tests.conftest import golden

pytestmark = pytest.mark.gpu

I32 = np.int32


def T(a, dev, dtype=None):
    t = torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    return t if dtype is None else t.to(dtype)


def N(t):
    return t.cpu().numpy()


def test_scatter_append(gpu):
    from suffixgpu_amd import SuffixGPUDrafter
    rng = np.random.default_rng(0)
    b, s, t = 33, 64, 9
    tok = rng.integers(0, 50, size=(b, s)).astype(I32)
    nt = rng.integers(0, s + 5, size=b).astype(I32)
    samp = rng.integers(-1, 50, size=(b, t)).astype(I32)
    samp[3] = -1
    d = SuffixGPUDrafter(k=4, device=gpu, max_pattern_len=8)
    o = DrafterOracle(k=4, max_pattern_len=8)
    for vc in (None, rng.integers(0, t + 1, size=b).astype(np.int64)):
        tg = T(tok, gpu)
        new = d.update_state(T(nt, gpu), tg, T(samp, gpu),
                             None if vc is None else T(vc, gpu))
        to = tok.copy()
        exp = o.update_state(nt, to, samp, vc)
        np.testing.assert_array_equal(N(tg), to)
        np.testing.assert_array_equal(N(new), exp)


def test_match_back_rows_and_shared(gpu):
    from suffixgpu_amd import kernels
    rng = np.random.default_rng(1)
    tok = rng.integers(0, 3, size=(7, 300)).astype(I32)
    q = rng.integers(0, 320, size=7)
    pat = newest_first_pattern(tok, q, 12, -2)
    got = kernels.match_back(T(tok, gpu), T(pat, gpu), 300)
    np.testing.assert_array_equal(N(got), o_match_back(tok, pat, 300))
    delta = rng.integers(-2, 3, size=500).astype(I32)
    got = kernels.match_back(T(delta, gpu), T(pat, gpu), 501)
    np.testing.assert_array_equal(N(got), o_match_back(delta, pat, 501))


def test_first_occurrences(gpu):
    from suffixgpu_amd import kernels
    rng = np.random.default_rng(2)
    mb = rng.integers(0, 6, size=(5, 3000)).astype(I32)
    thr = rng.integers(0, 7, size=(5, 4)).astype(np.int64)
    for r in (1, 7, 128, 600):
        pos, cnt = kernels.first_occurrences(T(mb, gpu), T(thr.reshape(-1),
                                                           gpu), 4, r)
        ep, ec = o_first_occ(mb, thr, r)
        np.testing.assert_array_equal(N(pos), ep.reshape(-1, r))
        np.testing.assert_array_equal(N(cnt), ec.reshape(-1))


@pytest.mark.parametrize("n", [1, 3, 4, 255, 4095, 4096, 4099, 12289])
def test_first_occurrences_edges(gpu, n):
    """Row lengths around four columns a thread and 4096 a pass (odd rows:
    every alignment), sparse and dense hits, more and fewer than max_occ,
    thresholds that nothing or everything reaches and past 32 bits."""
    from suffixgpu_amd import kernels
    rng = np.random.default_rng(n)
    mb = np.where(rng.random((3, n)) < 0.01, rng.integers(0, 30, (3, n)),
                  rng.integers(0, 3, (3, n))).astype(I32)
    mb[0, -1] = 31
    thr = np.array([[31, 1, 2, 20, -1, 1 << 33]] * 3, np.int64)
    for r in (1, 64, 5000):
        pos, cnt = kernels.first_occurrences(
            T(mb, gpu), T(thr.reshape(-1), gpu), 6, r)
        ep, ec = o_first_occ(mb, thr, r)
        np.testing.assert_array_equal(N(pos), ep.reshape(-1, r))
        np.testing.assert_array_equal(N(cnt), ec.reshape(-1))


@pytest.mark.parametrize("n", [256, 257, 1025, 4095, 4096, 6000, 9001])
@pytest.mark.parametrize("rows,c", [(1, 1), (32, 8), (33, 8), (128, 8),
                                    (1025, 1)])
def test_first_occurrences_workgroup_sizes(gpu, n, rows, c):
    """Row lengths and counts of threshold rows on either side of each
    workgroup size, with hits that are rare, common and everywhere."""
    from suffixgpu_amd import kernels
    rng = np.random.default_rng(n + rows)
    p = np.resize([0.002, 0.1, 1.0], rows)[:, None]
    mb = np.where(rng.random((rows, n)) < p, rng.integers(1, 9, (rows, n)),
                  0).astype(I32)
    thr = rng.integers(0, 9, (rows, c))
    pos, cnt = kernels.first_occurrences(T(mb, gpu), T(thr.reshape(-1), gpu),
                                         c, 40)
    ep, ec = o_first_occ(mb, thr, 40)
    np.testing.assert_array_equal(N(pos), ep.reshape(-1, 40))
    np.testing.assert_array_equal(N(cnt), ec.reshape(-1))


@pytest.mark.parametrize("n,vocab", [(1, 3), (2, 2), (7, 2), (64, 3),
                                     (4095, 4), (4097, 50), (20000, 3),
                                     (70000, 30000)])
def test_build_suffix_array(gpu, n, vocab):
    from suffixgpu_amd.suffix_array import build_suffix_array
    rng = np.random.default_rng(n)
    t = rng.integers(-2, vocab, size=n).astype(I32)
    got = build_suffix_array(T(t, gpu))
    np.testing.assert_array_equal(N(got), o_build_sa(t))


@pytest.mark.parametrize("n", [5000, 70000])
def test_build_suffix_array_wide_tokens(gpu, n):
    """Tokens spanning 2^31 values (no pair keys: the token round keys
    each position by its own token, signed order), over several radix
    tiles, with runs that need several doubling rounds."""
    from suffixgpu_amd.suffix_array import build_suffix_array
    rng = np.random.default_rng(n)
    vals = np.array([-2 ** 31, -5, 0, 7, 2 ** 30, 2 ** 31 - 2], np.int64)
    t = vals[rng.integers(0, len(vals), size=n)].astype(I32)
    t[n // 3:n // 3 + 900] = np.tile(t[:30], 30)  # a long repeat
    got = build_suffix_array(T(t, gpu))
    np.testing.assert_array_equal(N(got), o_build_sa(t))


def test_build_suffix_array_structured(gpu):
    from suffixgpu_amd.suffix_array import build_suffix_array
    for toks in ([1, 2, 3, 1, 2, 3, 1, 2], [5] * 5000, [0],
                 [3, -2, 2147483647, 3, -2, 0, 2147483647],
                 [-2147483648, 0, -2147483648, 5, -2147483648],
                 [1, 2] * 3000 + [1]):
        got = build_suffix_array(T(np.array(toks, I32), gpu))
        if len(toks) <= 64:
            assert N(got).tolist() == naive.suffix_array(toks)
        np.testing.assert_array_equal(N(got), o_build_sa(np.array(toks)))


def test_build_suffix_array_template_corpus(gpu):
    """Sequences sharing template spans: long repeats, many rounds, most
    suffixes finished early (the active set shrinks round by round)."""
    from suffixgpu_amd import synth
    from suffixgpu_amd.suffix_array import build_suffix_array
    tc = synth.TemplateCorpus(seed=11)
    docs = [np.append(tc.sequence(lo=1024, hi=4096), -2) for _ in range(90)]
    t = np.concatenate(docs + [np.array([2147483647])]).astype(I32)
    t = np.concatenate([t, t[:5000]])  # one 5000-token exact repeat
    got = build_suffix_array(T(t, gpu))
    np.testing.assert_array_equal(N(got), o_build_sa(t))


def _planted_bigram_text(count: int, seed: int) -> np.ndarray:
    """Random large-alphabet text where the bigram (1, 2) occurs exactly
    `count` times, after the suffixes starting with 0: the group of
    suffixes starting with (1, 2) -- the largest after the token round --
    occupies SA positions from there to there + count, across a
    4096-position tile boundary (asserted)."""
    rng = np.random.default_rng(seed)
    n = 3 * count + 6000
    t = rng.integers(3, 60000, size=n).astype(I32)
    t[rng.choice(n, 4000, replace=False)] = 0
    slots = rng.choice(n // 3 - 1, count, replace=False) * 3
    t[slots] = 1
    t[slots + 1] = 2
    zeros = int(np.sum(t == 0))
    assert zeros < 4096 < zeros + count
    return t


@pytest.mark.parametrize("extra", [0, 1])
def test_build_suffix_array_group_cap(gpu, extra):
    """A round whose largest group has sfx_sa_group_cap() suffixes sorts it
    inside one workgroup (following it into the next tile); one more takes
    the radix path.  The state's radix mask records which path round 1
    took."""
    from suffixgpu_amd import _lib
    from suffixgpu_amd.suffix_array import (build_suffix_array_into,
                                            read_build_state,
                                            sa_workspace_bytes)
    cap = int(_lib.lib().sfx_sa_group_cap())
    count = cap + extra
    t = _planted_bigram_text(count, count)
    exp = o_build_sa(t)
    assert np.sum((t[:-1] == 1) & (t[1:] == 2)) == count
    for adaptive in (True, False):
        ws = torch.empty(sa_workspace_bytes(t.shape[0]), dtype=torch.uint8,
                         device=gpu)
        out = torch.empty(t.shape[0], dtype=torch.int32, device=gpu)
        build_suffix_array_into(T(t, gpu), t.shape[0], out, ws,
                                adaptive=adaptive)
        np.testing.assert_array_equal(N(out), exp)
        st = read_build_state(ws, t.shape[0])
        assert st.done and not st.stalled
        assert bool(st.radix_mask & 2) == (count > cap)


def test_build_suffix_array_stall_and_resume(gpu):
    """Rounds enqueued without the radix path stop at the first round that
    needs it (the state names the round, the rest return at once); the
    same rounds enqueued again from there with the radix path finish the
    array."""
    from suffixgpu_amd import _lib
    from suffixgpu_amd.suffix_array import (build_suffix_array_rounds,
                                            enqueue_rounds, read_build_state,
                                            sa_workspace_bytes)
    t = _planted_bigram_text(5000, 3)
    m = t.shape[0]
    ws = torch.empty(sa_workspace_bytes(m), dtype=torch.uint8, device=gpu)
    out = torch.empty(m, dtype=torch.int32, device=gpu)
    L = _lib.lib()
    total = int(L.sfx_sa_build_rounds_total(m))
    build_suffix_array_rounds(T(t, gpu), m, out, ws, total, radix_mask=0)
    st = read_build_state(ws, m)
    assert not st.done and st.stalled == 1 and st.radix_mask == 1
    enqueue_rounds(m, 1, total, 1 << 1, ws.data_ptr(), ws.numel(),
                   _lib.stream_of(gpu))
    _lib.check(L.sfx_sa_build_finish(m, m, out.data_ptr(), 0, ws.data_ptr(),
                                     ws.numel(), _lib.stream_of(gpu)), "sa")
    st = read_build_state(ws, m)
    assert st.done and not st.stalled and st.radix_mask == 3
    np.testing.assert_array_equal(N(out), o_build_sa(t))


def test_build_suffix_array_stall_stops_every_launch(gpu):
    """Rounds behind a stalled one, with and without radix launches, leave
    the whole workspace as it is, and the build resumes from there."""
    from suffixgpu_amd import _lib
    from suffixgpu_amd.suffix_array import (enqueue_rounds, read_build_state,
                                            sa_workspace_bytes)
    m = 6001
    t = np.full(m, 7, I32)              # every round has a large group
    L = _lib.lib()
    st = _lib.stream_of(gpu)
    text = T(t, gpu)
    ws = torch.zeros(sa_workspace_bytes(m), dtype=torch.uint8, device=gpu)
    out = torch.full((m,), -9, dtype=torch.int32, device=gpu)
    args = (ws.data_ptr(), ws.numel(), st)
    _lib.check(L.sfx_sa_build_begin(text.data_ptr(), m, *args), "begin")
    enqueue_rounds(m, 1, 2, 1 << 1, *args)
    assert read_build_state(ws, m).stalled == 2
    before = N(ws)
    enqueue_rounds(m, 3, 3, 1 << 3 | 1 << 4, *args)
    _lib.check(L.sfx_sa_build_finish_if_final(
        m, 1, 5, m, out.data_ptr(), 0, *args), "finish")
    np.testing.assert_array_equal(N(ws), before)
    assert (N(out) == -9).all()
    total = int(L.sfx_sa_build_rounds_total(m))
    enqueue_rounds(m, 2, total - 1, -1, *args)
    _lib.check(L.sfx_sa_build_finish(m, m, out.data_ptr(), 0, *args),
               "finish")
    np.testing.assert_array_equal(N(out), np.arange(m)[::-1])


@pytest.mark.parametrize("period,n", [(0, 2), (0, 900), (2, 9), (3, 400),
                                      (40, 5000), (3000, 9001), (1, 5000)])
def test_build_suffix_array_adaptive_batches(gpu, period, n):
    """The adaptive build over texts whose last round falls on either side
    of a batch's end, from none (distinct tokens) to every round (one
    repeated token, whose rounds also need the radix path), and the output
    that waits for a batch's end: untouched before it, whole after it."""
    from suffixgpu_amd import _lib
    from suffixgpu_amd.suffix_array import (build_suffix_array_into,
                                            enqueue_rounds, read_build_state,
                                            sa_workspace_bytes)
    rng = np.random.default_rng(5)
    t = (rng.permutation(n) if period == 0 else
         np.resize(rng.permutation(period), n)).astype(I32)
    exp = o_build_sa(t)
    out = torch.full((n + 3,), -9, dtype=torch.int64, device=gpu)
    build_suffix_array_into(T(t, gpu), n, out, adaptive=True)
    np.testing.assert_array_equal(
        N(out), np.concatenate([exp, [n, n + 1, n + 2]]))

    L = _lib.lib()
    st = _lib.stream_of(gpu)
    ws = torch.empty(sa_workspace_bytes(n), dtype=torch.uint8, device=gpu)
    dt = T(t, gpu)
    total = int(L.sfx_sa_build_rounds_total(n))
    _lib.check(L.sfx_sa_build_begin(dt.data_ptr(), n, ws.data_ptr(),
                                    ws.numel(), st), "begin")
    outs = []
    for r in range(1, total + 1):
        enqueue_rounds(n, r, 1, -1, ws.data_ptr(), ws.numel(), st)
        o = torch.full((n,), -9, dtype=torch.int32, device=gpu)
        _lib.check(L.sfx_sa_build_finish_if_final(
            n, r, r, n, o.data_ptr(), 0, ws.data_ptr(), ws.numel(), st),
            "finish")
        outs.append(N(o))
    s = read_build_state(ws, n)
    # the round that left no group (a later one records that it found none)
    last = max(s.needed, 1) if s.done else total
    for r, o in enumerate(outs, 1):
        np.testing.assert_array_equal(o, exp if r == last else -9)


def test_build_suffix_array_stalls_in_a_row(gpu, monkeypatch):
    """One repeated token needs the radix path in every round: the stalls
    hand it out to more and more rounds, and no batch is wasted behind one
    after the first; random tokens of two values stall once more than the
    rounds that need it beyond the first."""
    from suffixgpu_amd import suffix_array as sa
    batches = []
    enqueue = sa.enqueue_rounds
    monkeypatch.setattr(sa, "enqueue_rounds",
                        lambda m, first, n, *a: (batches.append((first, n)),
                                                 enqueue(m, first, n, *a)))
    n = 70000
    out = torch.empty(n, dtype=torch.int32, device=gpu)
    sa.build_suffix_array_into(torch.full((n,), 7, dtype=torch.int32,
                                          device=gpu), n, out, adaptive=True)
    np.testing.assert_array_equal(N(out), np.arange(n)[::-1])
    # 16 rounds, 15 of them beyond the one given the path at first
    assert len(batches) <= 12, batches
    batches.clear()
    t = np.random.default_rng(1).integers(0, 2, n).astype(I32)
    sa.build_suffix_array_into(T(t, gpu), n, out, adaptive=True)
    _check_suffix_order(t, N(out).astype(np.int64))
    assert len(batches) <= 5, batches


@pytest.mark.parametrize("size", [511, 512, 513, 1000, 2048])
@pytest.mark.parametrize("at", [0, 2500, 4090])
def test_build_suffix_array_merged_windows(gpu, size, at):
    """A two-token group on both sides of the size from which a tile's
    windows are merged, `at` positions into its tile (so that it also runs
    on into the next one), beside small groups, with few distinct keys (runs
    of equal ones) and with many, over several rounds."""
    from suffixgpu_amd.suffix_array import build_suffix_array_into
    rng = np.random.default_rng(size + at)
    for keys in (3, 400):
        # the pair (10, 10) sorts behind `at` positions of small groups
        small = rng.integers(0, 9, size=at).astype(I32)
        cont = np.stack([np.full(size, 10), np.full(size, 10),
                         11 + rng.integers(0, keys, size)], 1)
        t = np.concatenate([small, cont.reshape(-1)]).astype(I32)
        out = torch.empty(t.shape[0], dtype=torch.int64, device=gpu)
        build_suffix_array_into(T(t, gpu), t.shape[0], out, adaptive=True)
        np.testing.assert_array_equal(N(out), o_build_sa(t))


@pytest.mark.parametrize("n", [2047, 2049, 131072, 131073, 524288, 524289])
def test_build_suffix_array_tile_sizes(gpu, n):
    """Both sides of a local tile, of the longest text whose radix passes
    are one launch each and of the longest that takes the small tile: few
    tokens (groups above the cap, radix rounds), runs of one token and a
    long repeat."""
    from suffixgpu_amd.suffix_array import build_suffix_array_into
    rng = np.random.default_rng(n)
    t = rng.integers(0, 20, n).astype(I32)
    t[n // 3:n // 3 + n // 8] = t[:n // 8]
    t[n // 2:n // 2 + min(n // 8, 3000)] = 7
    out = torch.empty(n, dtype=torch.int64, device=gpu)
    build_suffix_array_into(T(t, gpu), n, out, adaptive=True)
    got = N(out)
    # sorted by definition: a permutation, each suffix below the next
    assert np.array_equal(np.sort(got), np.arange(n))
    rank = np.empty(n + 1, np.int64)
    rank[got], rank[n] = np.arange(n), -1
    a, b = got[:-1], got[1:]
    assert np.all((t[a] < t[b]) |
                  ((t[a] == t[b]) & (rank[a + 1] < rank[b + 1])))


def _check_suffix_order(t, got):
    """Sorted by definition: a permutation, each suffix below the next."""
    n = t.shape[0]
    assert np.array_equal(np.sort(got), np.arange(n))
    rank = np.empty(n + 1, np.int64)
    rank[got], rank[n] = np.arange(n), -1
    a, b = got[:-1], got[1:]
    assert np.all((t[a] < t[b]) |
                  ((t[a] == t[b]) & (rank[a + 1] < rank[b + 1])))


def _past_small_tiles(t, top):
    """t with distinct larger tokens behind it (finished after the token
    round), so that the text takes the 4096-position local tile and t's
    suffixes come first in it."""
    fill = np.random.default_rng(0).permutation(1 << 19).astype(I32)
    return np.concatenate([t, top + 1 + fill]).astype(I32)


@pytest.mark.parametrize("size", [511, 512, 513, 2047, 2048, 2049])
@pytest.mark.parametrize("at", [0, 2500, 4090, 4096])
def test_build_suffix_array_groups_in_large_tiles(gpu, size, at):
    """A two-token group of a size on either side of the merge and of the
    cap, `at` positions into a 4096-position tile (past 2500 it runs on into
    the next one), beside small groups, with few distinct keys and many."""
    from suffixgpu_amd.suffix_array import build_suffix_array_into
    rng = np.random.default_rng(size + at)
    for keys in (3, 400):
        small = rng.integers(0, 9, size=at).astype(I32)
        cont = np.stack([np.full(size, 10), np.full(size, 10),
                         11 + rng.integers(0, keys, size)], 1)
        t = _past_small_tiles(np.concatenate([small, cont.reshape(-1)]), 500)
        out = torch.empty(t.shape[0], dtype=torch.int64, device=gpu)
        build_suffix_array_into(T(t, gpu), t.shape[0], out, adaptive=True)
        _check_suffix_order(t, N(out))


@pytest.mark.parametrize("period", [1, 2, 700])
@pytest.mark.parametrize("n", [2049, 5000, 9001])
def test_build_suffix_array_repeats_in_large_tiles(gpu, period, n):
    """A repeat that needs the radix path in no, some or every round (stalls
    and their resumption) and many batches of rounds, in a text of 4096-
    position tiles, adaptively and with every round enqueued."""
    from suffixgpu_amd.suffix_array import build_suffix_array_into
    rep = np.resize(np.random.default_rng(n).permutation(period), n)
    t = _past_small_tiles(rep, period)
    out = torch.empty(t.shape[0], dtype=torch.int64, device=gpu)
    for adaptive in (True, False):
        out.fill_(-9)
        build_suffix_array_into(T(t, gpu), t.shape[0], out,
                                adaptive=adaptive)
        _check_suffix_order(t, N(out))


def test_build_suffix_array_long_radix_list(gpu):
    """A radix list of more tiles than its launches have workgroups, so that
    every list kernel takes a second tile: all of 2.3M tokens of 8 values
    lie in groups above the cap after the token round."""
    from suffixgpu_amd.suffix_array import (build_suffix_array_rounds,
                                            read_build_state,
                                            sa_workspace_bytes)
    n = 2_300_000
    t = np.random.default_rng(8).integers(0, 8, n).astype(I32)
    pairs = np.bincount(t[:-1] * 8 + t[1:], minlength=64)
    listed = int(pairs[pairs > 2048].sum())
    assert listed > 512 * 4096
    ws = torch.empty(sa_workspace_bytes(n), dtype=torch.uint8, device=gpu)
    out = torch.empty(n, dtype=torch.int32, device=gpu)
    build_suffix_array_rounds(T(t, gpu), n, out, ws, 12, radix_mask=-1)
    st = read_build_state(ws, n)
    assert st.done and st.radix_mask & 2
    _check_suffix_order(t, N(out))


@pytest.mark.parametrize("n", [4097, 131072])
@pytest.mark.parametrize("vocab", [2, 511, 1000, 200000])
def test_build_suffix_array_few_digits(gpu, n, vocab):
    """One-launch radix passes over digits of one, two and many values (the
    counts of a wave's equal digits are added together)."""
    from suffixgpu_amd.suffix_array import build_suffix_array_into
    t = np.random.default_rng(n + vocab).integers(0, vocab, n).astype(I32)
    out = torch.empty(n, dtype=torch.int64, device=gpu)
    build_suffix_array_into(T(t, gpu), n, out, adaptive=True)
    _check_suffix_order(t, N(out))


@pytest.mark.parametrize("final_from", [1, 2, 4])
def test_build_suffix_array_expect_final_flag(gpu, final_from):
    """Rounds flagged as expected to find the array final (a rebuild's
    margin rounds) give the same array whether the flag is right or wrong:
    from round 1 every round is flagged, including the token pairs' radix
    round and the rounds that still have groups to sort."""
    from suffixgpu_amd.suffix_array import (build_suffix_array_rounds,
                                            read_build_state,
                                            sa_workspace_bytes)
    rng = np.random.default_rng(11)
    period = rng.integers(0, 5, size=37).astype(I32)
    texts = [_planted_bigram_text(5000, 3),
             np.concatenate([np.tile(period, 300),
                             rng.integers(0, 5, size=900).astype(I32)])]
    for t in texts:
        m = t.shape[0]
        ws = torch.empty(sa_workspace_bytes(m), dtype=torch.uint8,
                         device=gpu)
        out = torch.empty(m, dtype=torch.int32, device=gpu)
        build_suffix_array_rounds(T(t, gpu), m, out, ws, 40,
                                  radix_mask=(1 << 40) - 2,
                                  final_from=final_from)
        st = read_build_state(ws, m)
        assert st.done and not st.stalled
        np.testing.assert_array_equal(N(out), o_build_sa(t))


def test_build_suffix_array_identity_tail(gpu):
    from suffixgpu_amd.suffix_array import build_suffix_array_into
    rng = np.random.default_rng(4)
    t = rng.integers(0, 9, size=1000).astype(I32)
    out = torch.empty(1500, dtype=torch.int32, device=gpu)
    build_suffix_array_into(T(t, gpu), 600, out)
    exp = np.concatenate([o_build_sa(t[:600]), np.arange(600, 1500)])
    np.testing.assert_array_equal(N(out), exp)


@pytest.mark.parametrize("seed", range(3))
def test_sa_search(gpu, seed):
    from suffixgpu_amd.sa_search import search_interval
    rng = np.random.default_rng(seed)
    n = 3000
    toks = rng.integers(0, 4, size=n).astype(I32)
    sa = o_build_sa(toks).astype(I32)
    pats = np.zeros((200, 10), I32)
    lens = np.zeros(200, np.int64)
    for i in range(200):
        m = int(rng.integers(0, 11))
        st = int(rng.integers(0, n - m + 1))
        pats[i, :m] = toks[st:st + m]
        if i % 5 == 0:
            pats[i, :m] = rng.integers(0, 5, size=m)
        lens[i] = m
    s, e = search_interval(T(sa, gpu), T(toks, gpu), T(pats, gpu),
                           T(lens, gpu))
    es, ee = o_search(sa, toks, pats, lens)
    np.testing.assert_array_equal(N(s), es)
    np.testing.assert_array_equal(N(e), ee)


def _rand_expand(rng, b, r, k, vocab=9):
    cont = rng.integers(0, vocab, size=(b, r, k)).astype(I32)
    tail = rng.integers(0, k + 1, size=(b, r))
    cont = np.where(np.arange(k)[None, None, :] < tail[:, :, None], cont, -1)
    occ = rng.integers(0, r + 1, size=b).astype(np.int64)
    cap = rng.integers(-1, k + 2, size=b).astype(np.int64)
    return cont.astype(I32), occ, cap


@pytest.mark.parametrize("n", [1, 2, 37, 3000])
@pytest.mark.parametrize("width", [1, 4, 31, 32, 33, 70])
def test_sa_search_widths_and_batches(gpu, n, width):
    """Patterns shorter and longer than the 32 tokens an octet compares,
    running past the end of the corpus, on both lane counts (up to 8192
    patterns and past it)."""
    from suffixgpu_amd import kernels
    rng = np.random.default_rng(n * 100 + width)
    corpus = rng.integers(0, 2, size=n).astype(I32)
    corpus[n // 2:] = corpus[:n - n // 2]  # long repeats
    sa = o_build_sa(corpus)
    b = 40
    pat = np.full((b, width), -1, I32)
    plen = rng.integers(0, width + 1, size=b)
    for i in range(b):
        st = rng.integers(0, n)
        seg = corpus[st:st + plen[i]]
        pat[i, :seg.shape[0]] = seg
        pat[i, seg.shape[0]:plen[i]] = rng.integers(0, 2)
        if i % 4 == 0 and plen[i]:
            pat[i, plen[i] - 1] = rng.integers(-1, 3)
    es, ee = o_search(sa, corpus, pat, plen)
    for rows in (b, 8192, 8193):
        rep = np.arange(rows) % b
        lo, hi = kernels.sa_search(T(sa.astype(I32), gpu), T(corpus, gpu),
                                   T(pat[rep], gpu), T(plen[rep], gpu))
        np.testing.assert_array_equal(N(lo), es[rep])
        np.testing.assert_array_equal(N(hi), ee[rep])


@pytest.mark.parametrize("rows", [1, 64, 4096, 4097])
@pytest.mark.parametrize("width", [1, 2, 4, 5, 8, 9])
def test_sa_search_short_patterns(gpu, rows, width):
    """Patterns that a lane compares by itself and the first that an octet
    does, side by side in a wave (lengths 0 .. width), over few tokens with a
    pad among them, many of them at the corpus' end (past which a token
    compares as -1, the least here, so the order is one); on both lane counts
    (up to 4096 patterns of at most 4 tokens and past it)."""
    from suffixgpu_amd import kernels
    rng = np.random.default_rng(rows * 10 + width)
    n = 1500
    corpus = rng.choice(np.array([0, 1, 2, 3, 2**31 - 1], I32), n)
    sa = o_build_sa(corpus)
    b = min(rows, 200)
    plen = rng.integers(0, width + 1, size=b)
    pat = np.full((b, width), -1, I32)
    for i in range(b):
        at = n - rng.integers(1, 12) if i % 2 else rng.integers(0, n)
        seg = corpus[at:at + plen[i]]
        pat[i, :seg.shape[0]] = seg
        if i % 5 == 0 and plen[i]:
            pat[i, rng.integers(0, plen[i])] = rng.integers(-3, 4)
    es, ee = o_search(sa, corpus, pat, plen)
    rep = np.arange(rows) % b
    lo, hi = kernels.sa_search(T(sa.astype(I32), gpu), T(corpus, gpu),
                               T(pat[rep], gpu), T(plen[rep], gpu))
    np.testing.assert_array_equal(N(lo), es[rep])
    np.testing.assert_array_equal(N(hi), ee[rep])


@pytest.mark.parametrize("r", [1, 4, 30, 128, 256, 700])
@pytest.mark.parametrize("minp", [0.0, 0.1])
def test_expand_chain(gpu, r, minp):
    from suffixgpu_amd.expand import expand_chain
    rng = np.random.default_rng(1234 + r)
    for k, vocab in ((16, 9), (5, 3), (12, 2000)):
        cont, occ, cap = _rand_expand(rng, 37, r, k, vocab)
        got = expand_chain(T(cont, gpu), T(occ, gpu), k,
                           min_token_prob=minp, cap=T(cap, gpu))
        exp = o_expand(cont, occ, k, min_token_prob=minp, cap=cap)
        for g, e in zip(got, exp):
            np.testing.assert_array_equal(N(g), e)


@pytest.mark.parametrize("sentinel", [-7, -2, 0, 4])
def test_expand_chain_other_sentinels(gpu, sentinel):
    """A sentinel other than -1 pads the continuations and -1 is then a
    real token (expand.py:59-66, 107-147): the chain, counts and scores
    equal the oracle's, with and without weights, and int64 blocks keep
    their dtype."""
    from suffixgpu_amd.expand import expand_chain
    rng = np.random.default_rng(77 + sentinel)
    b, r, k = 41, 48, 10
    for lo, hi in ((-3, 6), (sentinel - 2, sentinel + 3)):
        cont = rng.integers(lo, hi, size=(b, r, k))
        tail = rng.integers(0, k + 1, size=(b, r))
        cont = np.where(np.arange(k)[None, None, :] < tail[:, :, None], cont,
                        sentinel)
        occ = rng.integers(0, r + 1, size=b).astype(np.int64)
        cap = rng.integers(-1, k + 2, size=b).astype(np.int64)
        w = rng.random((b, r)).astype(np.float32) + 0.05
        for dt, weights in ((I32, None), (np.int64, None), (I32, w)):
            c = cont.astype(dt)
            got = expand_chain(T(c, gpu), T(occ, gpu), k, sentinel=sentinel,
                               min_token_prob=0.05, cap=T(cap, gpu),
                               weights=None if weights is None
                               else T(weights, gpu))
            exp = o_expand(c, occ, k, sentinel=sentinel, min_token_prob=0.05,
                           cap=cap, weights=weights)
            assert got[0].dtype == T(c, gpu).dtype
            for g, e in zip(got[:3], exp[:3]):
                np.testing.assert_array_equal(N(g), e)
            if weights is None:
                np.testing.assert_array_equal(N(got[3]), exp[3])
            else:
                np.testing.assert_allclose(N(got[3]), exp[3], rtol=1e-5,
                                           atol=0)


@pytest.mark.parametrize("i", range(4))
def test_expand_alpha_weights_golden(gpu, i):
    from suffixgpu_amd.expand import expand_chain
    z = golden("expand_alpha_weights")
    cont, occ, cap = z[f"cont_{i}"], z[f"occ_{i}"], z[f"cap_{i}"]
    k = cont.shape[2]
    got = expand_chain(T(cont, gpu), T(occ, gpu), k, min_token_prob=0.05,
                       cap=T(cap, gpu), alpha=float(z[f"alpha_{i}"]))
    for g, key in zip(got, ("chain", "nv", "emit", "score")):
        np.testing.assert_array_equal(N(g), z[f"{key}_{i}"], err_msg=key)
    got = expand_chain(T(cont, gpu), T(occ, gpu), k, min_token_prob=0.05,
                       cap=T(cap, gpu), weights=T(z[f"w_{i}"], gpu))
    for g, key in zip(got[:3], ("wchain", "wnv", "wemit")):
        np.testing.assert_array_equal(N(g), z[f"{key}_{i}"], err_msg=key)
    np.testing.assert_allclose(N(got[3]), z[f"wscore_{i}"], rtol=1e-5,
                               atol=0)


def test_expand_division_table(gpu):
    """Every vote fraction v/n, 1 <= v <= n <= 128, is the IEEE fp32
    quotient: a one-depth chain of n occurrences with v equal tokens."""
    from suffixgpu_amd.expand import expand_chain
    rows = [(v, n) for n in range(1, 129) for v in range(1, n + 1)]
    b = len(rows)
    cont = np.full((b, 128, 1), -1, I32)
    occ = np.zeros(b, np.int64)
    for i, (v, n) in enumerate(rows):
        cont[i, :n, 0] = np.arange(1000, 1000 + n)
        cont[i, :v, 0] = 7
        occ[i] = n
    for alpha in (0.0, 0.5):
        _, _, _, score = expand_chain(T(cont, gpu), T(occ, gpu), 1,
                                      alpha=alpha)
        exp = np.array([np.float32(v) / (np.float32(max(n, 1)) +
                                         np.float32(alpha))
                        for v, n in rows], np.float32)
        np.testing.assert_array_equal(N(score), exp)


@pytest.mark.parametrize("start,n", [(1, 39999), (100, 30000), (8191, 8192),
                                     (20000, 20000), (0, 123), (5, 0)])
def test_delta_shift_in_place(gpu, start, n):
    """delta[:n] = delta[start:start + n] in place, overlapping windows
    included, and the device length set to n; the rest is untouched."""
    from suffixgpu_amd import _lib
    rng = np.random.default_rng(start + n)
    cap = 40000
    host = rng.integers(0, 1 << 30, size=cap).astype(I32)
    dl = torch.full((), -7, dtype=torch.int64, device=gpu)
    d = torch.from_numpy(host).to(gpu)
    rc = _lib.lib().sfx_delta_shift(d.data_ptr(), cap, start, n,
                                    dl.data_ptr(),
                                    torch.cuda.current_stream(gpu).cuda_stream)
    assert rc == 0
    want = host.copy()
    want[:n] = host[start:start + n]
    np.testing.assert_array_equal(d.cpu().numpy(), want)
    assert int(dl.item()) == n


def test_delta_append_groups(gpu):
    """150 documents (three launches of at most 64) at host-chosen offsets,
    a zero-length one among them; each followed by SEP, length set."""
    from suffixgpu_amd import _lib
    rng = np.random.default_rng(3)
    cap = 30000
    d = torch.full((cap,), 77, dtype=torch.int32, device=gpu)
    dl = torch.zeros((), dtype=torch.int64, device=gpu)
    want = np.full(cap, 77, dtype=I32)
    srcs, descs, off = [], [], 0
    for i in range(150):
        n = 0 if i == 17 else int(rng.integers(1, 150))
        x = rng.integers(0, 1000, size=n).astype(I32)
        t = torch.from_numpy(x).to(gpu)
        srcs.append(t)
        descs.append(_lib.SfxAppendDoc(t.data_ptr(), n, off))
        want[off:off + n] = x
        want[off + n] = -2
        off += n + 1
    arr = (_lib.SfxAppendDoc * len(descs))(*descs)
    rc = _lib.lib().sfx_delta_append(arr, len(descs), d.data_ptr(), cap,
                                     dl.data_ptr(), off,
                                     torch.cuda.current_stream(gpu).cuda_stream)
    assert rc == 0
    np.testing.assert_array_equal(d.cpu().numpy(), want)
    assert int(dl.item()) == off


@pytest.mark.parametrize("weighted", [False, True])
def test_majority_token_vs_oracle(gpu, weighted):
    """expand._majority_token (a one-depth expansion) against the oracle's
    pairwise vote.  Weights are multiples of 1/8, so every weight sum is
    exact in fp32 whatever the summation order, and tokens and counts
    compare exactly."""
    from oracle.expand import majority_token as o_major
    from suffixgpu_amd.expand import _majority_token
    rng = np.random.default_rng(17)
    b, r = 96, 40
    vals = rng.integers(0, 6, size=(b, r)).astype(np.int64)
    act = rng.random((b, r)) < 0.7
    act[:4] = False  # rows with no active entry
    w = ((rng.integers(1, 9, size=(b, r)) / 8).astype(np.float32)
         if weighted else None)
    tok, cnt = _majority_token(T(vals, gpu), T(act, gpu), -5,
                               None if w is None else T(w, gpu))
    etok, ecnt = o_major(vals, act, -5, w)
    np.testing.assert_array_equal(N(tok), etok)
    np.testing.assert_array_equal(N(cnt), ecnt)
