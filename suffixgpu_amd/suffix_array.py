"""Suffix-array construction (public API).

Mirrors suffix_gpu/suffix_array.py:15-63.  The GPU build (csrc/sa_build.hip)
is prefix doubling that stops on the device once all ranks are distinct:
a round whose unsorted groups fit a workgroup sorts them there in one
launch, a round with a larger group takes LSD radix sorts.  The suffix
array is unique, so it equals the reference's.
"""

from __future__ import annotations

from collections import deque

import torch

from suffixgpu_amd._lib import (SA_ROUNDS_EXPECT_FINAL, SA_ROUNDS_RADIX,
                                check, lib, require_gpu, stream_of,
                                unrelated_to_captures)


def sa_workspace_bytes(n: int) -> int:
    return int(lib().sfx_sa_build_workspace_size(int(n)))


# Doubling rounds enqueued between two reads of the build's state in the
# adaptive build.
SA_CHECK_ROUNDS = 3

# int32 words of the build's state block a host copy reads, and the
# default rounds that enqueue the radix path (round 1: on natural text its
# two-token groups exceed a workgroup)
STATE_WORDS = 16
DEFAULT_RADIX_MASK = 1 << 1
# the words an adaptive build copies after a batch: past the state block's
# first words, [MAX_GROUP_WORD + r] is the largest group entering round r
MAX_GROUP_WORD = 16
BATCH_STATE_WORDS = 64


def _workspace_ok(workspace: torch.Tensor | None, text: torch.Tensor,
                  need: int) -> torch.Tensor:
    """The caller's byte workspace, or a new one when it is None or short.
    A workspace must be a contiguous uint8 tensor on the text's device:
    its numel() is the byte count and the state block is sliced by byte
    offset."""
    if workspace is not None:
        if (workspace.dtype != torch.uint8 or not workspace.is_contiguous()
                or workspace.device != text.device):
            raise ValueError("workspace must be a contiguous uint8 tensor on "
                             f"{text.device}")
        if workspace.numel() >= need:
            return workspace
    return torch.empty(max(need, 1), dtype=torch.uint8, device=text.device)


def build_suffix_array_into(text: torch.Tensor, m: int, out: torch.Tensor,
                            workspace: torch.Tensor | None = None,
                            adaptive: bool = False) -> None:
    """out[:m] = SA(text[:m]); out[m:] = m .. len(out)-1 (int32 or int64).

    adaptive=False (the default) enqueues the fixed launch sequence for
    every doubling round the length allows, with no host read: launches
    after the finishing round return at their first instruction, and the
    call can be captured in a graph or run in the background.
    adaptive=True enqueues the rounds SA_CHECK_ROUNDS at a time, one batch
    ahead of the host's reads of the build state, and returns when the host
    has seen the array final, so the build stops within a few launches of
    the round that finished it (the reference's build synchronises too, on
    torch.unique in suffix_gpu/suffix_array.py)."""
    require_gpu(text, out)
    if text.dtype != torch.int32 or not text.is_contiguous():
        raise ValueError("text must be a contiguous int32 tensor")
    if out.dtype not in (torch.int32, torch.int64) or not out.is_contiguous():
        raise ValueError("out must be a contiguous int32/int64 tensor")
    if m > text.shape[0] or m > out.shape[0]:
        raise ValueError("m exceeds the text or output length")
    workspace = _workspace_ok(workspace, text, sa_workspace_bytes(m))
    if adaptive and m > 1:
        _build_adaptive(text, m, out, workspace)
        return
    check(lib().sfx_sa_build(text.data_ptr(), m, out.shape[0],
                             out.data_ptr(), int(out.dtype == torch.int64),
                             workspace.data_ptr(), workspace.numel(),
                             stream_of(text.device)), "build_suffix_array")


@unrelated_to_captures()
def _build_adaptive(text: torch.Tensor, m: int, out: torch.Tensor,
                    workspace: torch.Tensor,
                    radix_mask: int = DEFAULT_RADIX_MASK) -> BuildState:
    """The adaptive build of m > 1 positions: rounds go out SA_CHECK_ROUNDS
    at a time, each batch followed by a state copy and an output that is
    written only if that batch finished the array, and the host waits for a
    batch with the next one already enqueued, so the GPU never waits for the
    host between rounds.  ``radix_mask``: rounds expected to need the radix
    path (any other that does stalls the build and is enqueued again with
    it).

    What runs behind a stall is wasted, so the batch that resumes a stalled
    build goes out alone, and a text of long repeats, which needs the path
    for many rounds in a row, is given it for 1, 1, 2, 4, 8 ... rounds by
    the stalls of a row (a round that is given it and needs none has 16 idle
    launches, so two stalls in a row, as 1,500,000 random tokens of two
    values have them, still get one round each).  One repeated token,
    1,500,000 positions: 3.10 ms; 3.45 with a round a stall and a batch
    behind each.

    Returns the state that found the array final."""
    L = lib()
    st = stream_of(text.device)
    ws, nbytes = workspace.data_ptr(), workspace.numel()
    is64 = int(out.dtype == torch.int64)
    total = int(L.sfx_sa_build_rounds_total(m))
    state = state_view(workspace, m, BATCH_STATE_WORDS)
    flags = torch.empty(2, BATCH_STATE_WORDS, dtype=torch.int32,
                        pin_memory=True)
    check(L.sfx_sa_build_begin(text.data_ptr(), m, ws, nbytes, st),
          "build_suffix_array")
    stream = torch.cuda.current_stream(text.device)
    pending: deque = deque()  # (event, last round, pinned state words)
    first = 1
    sent = 0
    ahead = 2           # batches in flight
    row, behind = 0, 0  # stalls in a row; the round behind the last one's
    while True:
        while len(pending) < ahead and first <= total:
            n = min(SA_CHECK_ROUNDS, total - first + 1)
            last = first + n - 1
            enqueue_rounds(m, first, n, radix_mask, ws, nbytes, st)
            words = flags[sent & 1]
            sent += 1
            words.copy_(state, non_blocking=True)
            ev = torch.cuda.Event()
            ev.record(stream)
            check(L.sfx_sa_build_finish_if_final(
                m, first, last, out.shape[0], out.data_ptr(), is64, ws,
                nbytes, st), "build_suffix_array")
            pending.append((ev, last, words))
            first = last + 1
        ev, last, words = pending.popleft()
        ev.synchronize()
        w = words.tolist()
        s = BuildState.of(w)
        if s.stalled:
            # the batch behind it returned at once; resume from the round
            first = s.stalled
            row = row + 1 if first == behind else 1
            run = 1 << max(0, row - 2)
            behind = first + run
            radix_mask |= ((1 << run) - 1) << first
            ahead = 1
            pending.clear()
            continue
        ahead = 2
        if s.done:
            return s
        elif w[MAX_GROUP_WORD + last + 1] == 0:  # round last left no group
            none = next(r for r in range(1, last + 2)
                        if w[MAX_GROUP_WORD + r] == 0)
            return BuildState(True, none, 0, s.radix_mask)
        elif last == total:  # (h has reached m: cannot hold a group)
            raise RuntimeError("suffix array not final after every round")


def build_suffix_array(tokens: torch.Tensor) -> torch.Tensor:
    """Suffix array (int64) of a 1-D token sequence; negatives allowed."""
    require_gpu(tokens)
    tokens = tokens.reshape(-1).to(torch.int32).contiguous()
    n = tokens.shape[0]
    out = torch.empty(n, dtype=torch.int64, device=tokens.device)
    if n == 0:
        return out
    build_suffix_array_into(tokens, n, out, adaptive=True)
    return out


def build_suffix_array_rounds(text: torch.Tensor, m: int, out: torch.Tensor,
                              workspace: torch.Tensor, rounds: int,
                              radix_mask: int = DEFAULT_RADIX_MASK,
                              final_from: int = 0) -> None:
    """The build with only its first ``rounds`` doubling rounds enqueued
    (then the output copy): the background rebuild's first chunk.  Rounds
    whose bit is set in ``radix_mask`` enqueue the radix path too; rounds
    from ``final_from`` on (0: none) are enqueued as expected to find the
    array final (see :func:`enqueue_rounds`).  The result is final iff
    :func:`build_state` says so afterwards."""
    require_gpu(text, out, workspace)
    workspace = _workspace_ok(workspace, text, sa_workspace_bytes(m))
    L = lib()
    st = stream_of(text.device)
    ws, nbytes = workspace.data_ptr(), workspace.numel()
    check(L.sfx_sa_build_begin(text.data_ptr(), m, ws, nbytes, st),
          "SA build")
    enqueue_rounds(m, 1, max(0, rounds), radix_mask, ws, nbytes, st,
                   final_from)
    check(L.sfx_sa_build_finish(m, out.shape[0], out.data_ptr(),
                                int(out.dtype == torch.int64), ws, nbytes,
                                st), "SA build")


def enqueue_rounds(m: int, first: int, count: int, radix_mask: int,
                   ws: int, nbytes: int, stream, final_from: int = 0) -> None:
    """Doubling rounds first .. first+count-1 on ``stream``: a round r with
    bit r of ``radix_mask`` set enqueues the radix path too, the others
    only the local launch (a round that needs the radix path then stalls
    the build, see :class:`BuildState`).  Rounds r >= ``final_from`` (when
    it is positive) are flagged as expected to find the array final, as a
    rebuild's margin rounds are: their launches check the build state
    before reading their tiles.  The flag changes no result."""
    L = lib()

    def flags(r: int) -> int:
        f = SA_ROUNDS_RADIX if (radix_mask >> r) & 1 else 0
        if 0 < final_from <= r:
            f |= SA_ROUNDS_EXPECT_FINAL
        return f

    r, end = first, first + count
    while r < end:
        f = flags(r)
        r2 = r + 1
        while r2 < end and flags(r2) == f:
            r2 += 1
        check(L.sfx_sa_build_rounds(m, r, r2 - r, f, ws, nbytes, stream),
              "SA build")
        r = r2


def state_view(workspace: torch.Tensor, m: int,
               words: int = STATE_WORDS) -> torch.Tensor:
    """The device words of a build's state block (a view of the byte
    workspace)."""
    off = int(lib().sfx_sa_build_flag_offset(m))
    return workspace[off:off + 4 * words].view(torch.int32)


class BuildState:
    """A build's state words: done (the array is final), found_none (the
    round that found no unsorted group), stalled (the round that needs the
    radix path it was not given, 0 for none) and radix_mask (bit r for each
    round that took the radix path; bit 0 is the token round)."""

    def __init__(self, done: bool, found_none: int, stalled: int,
                 radix_mask: int):
        self.done = done
        self.found_none = found_none
        self.stalled = stalled
        self.radix_mask = radix_mask

    @classmethod
    def of(cls, words: list[int]) -> "BuildState":
        return cls(bool(words[0]), int(words[2]), int(words[7]),
                   int(words[8]) & 0xffffffff)

    @property
    def needed(self) -> int:
        """Doubling rounds the array needed (-1 while not final)."""
        return max(self.found_none - 1, 0) if self.done else -1


def read_build_state(workspace: torch.Tensor, m: int) -> BuildState:
    """The state of a build (synchronises the current stream)."""
    if m <= 1:
        return BuildState(True, 1, 0, 0)
    return BuildState.of(state_view(workspace, m).cpu().tolist())


def build_state(workspace: torch.Tensor, m: int) -> tuple[bool, int]:
    """(final, rounds the array needed) from a build's workspace; reads the
    device (synchronises the current stream)."""
    s = read_build_state(workspace, m)
    return s.done, (s.needed if m > 1 else 0)
