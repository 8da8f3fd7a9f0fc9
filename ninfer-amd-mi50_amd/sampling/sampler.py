"""Sampling of next tokens from logits rows on the device.

Policy as the reference's `sample_logits` (src/runtime/engine.cpp:18-82):
repetition penalty over prompt + generated tokens, greedy if temperature
<= 0, else temperature, top-k, softmax, top-p, one draw. The reference seeds
`mt19937_64(seed + step)` per step (:166-169); here the uniform number of a
draw is a counter hash of (seed, request key, draw index), so a request's
tokens do not depend on what it was batched with. Seed 0 means "not fixed":
the request gets a seed from the operating system when it is added.
"""
from __future__ import annotations

import os
from array import array
from itertools import accumulate
from operator import attrgetter
from typing import Dict, Iterable, List, Optional, Sequence, Tuple

import numpy as np
import torch

from .params import SamplingParams

_MASK = (1 << 64) - 1
# Tokens of a vocabulary beyond which rows that top-k does not cut go through four launches by the whole GPU (one row of
# 9,000, us so and by one block: 29 and 36, with top-p 1 23 and 19; 32,000 30 and 74, 23 and 33), and greedy ones with
# a penalty through two (32,000 tokens 11 and 10, 64 rows 12 and 13; 151,936 11 and 25, 21 and 33)
SPREAD_TOKENS = 12288
FEW_GREEDY_TOKENS = 32768
_OPTIONS = attrgetter("temperature", "top_p", "repetition_penalty", "top_k")
_STREAM = attrgetter("seed", "key", "draw")


def _splitmix64(x: int) -> int:
    x = (x + 0x9E3779B97F4A7C15) & _MASK
    x = ((x ^ (x >> 30)) * 0xBF58476D1CE4E5B9) & _MASK
    x = ((x ^ (x >> 27)) * 0x94D049BB133111EB) & _MASK
    return x ^ (x >> 31)


def uniform(seed: int, key: int, draw: int) -> float:
    """A number in [0, 1) with 24 random bits from (seed, key, draw)."""
    h = _splitmix64(_splitmix64(_splitmix64(seed & _MASK) ^ (key & _MASK)) ^ (draw & _MASK))
    return (h >> 40) / float(1 << 24)


def _streams(rows: Sequence["SampleRow"]) -> List[array]:
    """The rows' seeds, keys and draws as arrays of 64-bit numbers."""
    def u64s(vs):
        try:
            return array("Q", vs)
        except (OverflowError, TypeError):   # (of other sizes or signs: their last 64 bits)
            return array("Q", [v & _MASK for v in vs])
    return [u64s(vs) for vs in zip(*map(_STREAM, rows))]


def uniforms(rows: Sequence["SampleRow"]) -> np.ndarray:
    """`uniform` of every row's (seed, key, draw) at once, in 32-bit floats (24 bits each: exact)."""
    u64 = np.uint64

    def mix(x):
        x = x + u64(0x9E3779B97F4A7C15)
        x = (x ^ (x >> u64(30))) * u64(0xBF58476D1CE4E5B9)
        x = (x ^ (x >> u64(27))) * u64(0x94D049BB133111EB)
        return x ^ (x >> u64(31))

    seed, key, draw = (np.frombuffer(v, dtype=u64) for v in _streams(rows))
    return (mix(mix(mix(seed) ^ key) ^ draw) >> u64(40)).astype(np.float32) / np.float32(1 << 24)


def fresh_seed() -> int:
    return int.from_bytes(os.urandom(8), "little") | 1


class History:
    """How often a request has seen each token (prompt + generated), for the
    repetition penalty. Kept as two growing arrays (distinct tokens, counts), so
    that a step hands them to the device as they are: the work per generated
    token does not grow with the length of the history."""

    def __init__(self, tokens: Iterable[int] = ()):
        toks, counts = np.unique(np.asarray(list(tokens), dtype=np.int64), return_counts=True)
        n = int(toks.shape[0])
        self._both = np.zeros((2, max(64, 2 * n)), np.int32)   # tokens, then counts
        self._both[0, :n] = toks
        self._both[1, :n] = counts
        self._n = n
        self._where: Optional[Dict[int, int]] = None   # token -> index, made at the first add

    def add(self, token: int) -> None:
        if self._where is None:
            self._where = {int(t): i for i, t in enumerate(self._both[0, :self._n])}
        i = self._where.get(token)
        if i is not None:
            self._both[1, i] += 1
            return
        if self._n == self._both.shape[1]:
            self._both = np.concatenate([self._both, np.zeros_like(self._both)], axis=1)
        self._both[0, self._n] = token
        self._both[1, self._n] = 1
        self._where[token] = self._n
        self._n += 1

    def arrays(self) -> Tuple[np.ndarray, np.ndarray]:
        """(distinct tokens, their counts), int32 views of equal length."""
        return self._both[0, :self._n], self._both[1, :self._n]

    def both(self) -> np.ndarray:
        """`arrays` as the two rows of one view."""
        return self._both[:, :self._n]

    def count(self, token: int) -> int:
        toks, cnts = self.arrays()
        hit = np.nonzero(toks == token)[0]
        return int(cnts[hit[0]]) if hit.size else 0

    def __len__(self) -> int:
        return self._n


class SampleRow:
    """What the sampler needs of one row: options, history counts, RNG stream."""

    def __init__(self, params: SamplingParams, history: History, key: int, draw: int, seed: int):
        self.params = params
        self.history = history if isinstance(history, History) else History(
            t for t, c in dict(history).items() for _ in range(c))
        self.key = key
        self.draw = draw
        self.seed = seed


class Sampler:
    def __init__(self, ops, device):
        self.ops = ops
        self.device = device
        self._free: List[tuple] = []   # pinned buffers that no call uses

    def _staged(self, n: int) -> tuple:
        """(a buffer of at least n ints in pinned memory, the same memory as an array), which no other call uses until
        it is given back. The rows' parameters are written into it and fetched from it behind the step that makes
        the logits, while the host goes on (a copy out of pageable memory makes the host wait until the device has
        reached it, and the sampling kernel would then be launched only after the step has ended)."""
        try:
            slot = self._free.pop()
        except IndexError:
            slot = None
        if slot is None or slot[0].numel() < n:
            buffer = torch.empty(max(n if slot is None else 2 * n, 1024), dtype=torch.int32).pin_memory()
            slot = (buffer, buffer.numpy())
        return slot

    def sample(self, logits: torch.Tensor, rows: Sequence[SampleRow]) -> List[int]:
        """One token per row of `logits` [R, vocab]."""
        r = len(rows)
        assert logits.shape[0] == r
        # Everything the kernel needs of the rows travels in one array and one copy: four
        # 32-bit floats and one int per row, the offsets of the penalties, then their tokens
        # and counts. (Copies queue behind the step that makes the logits, one after the other:
        # every further one would add its latency to the step.)
        temps, tops, penalties, top_ks = zip(*map(_OPTIONS, (row.params for row in rows))) if r else ((),) * 4
        listed = [len(row.history) if penalty != 1.0 else 0 for row, penalty in zip(rows, penalties)]
        n_pen = sum(listed)
        o = 5 * r
        n = o + (r + 1 + 2 * n_pen if n_pen > 0 else 0)
        cuda = self.device.type == "cuda"
        if cuda:
            at = (n + 3) // 4 * 4   # (the tokens come behind the parameters)
            slot = pinned, packed = self._staged(at + r)
        else:
            packed = np.empty(n, np.int32)
        floats = packed[:4 * r].view(np.float32).reshape(4, r)
        floats[0] = temps
        floats[1] = tops
        floats[2] = penalties
        drawn = [row for row, t in zip(rows, temps) if t > 0]   # (greedy rows draw nothing)
        if len(drawn) < r:
            floats[3] = 0.0
        if drawn:
            to = floats[3] if len(drawn) == r else np.empty(len(drawn), np.float32)
            # (us one by one 1.5 a row; in the library 5.5 to 6.6 for 1 to 8; as whole arrays 31 for 16 rows, 34 for 24)
            if len(drawn) <= (3 if cuda else 20):
                to[:] = [uniform(row.seed, row.key, row.draw) for row in drawn]
            elif cuda:
                self.ops.uniforms(*_streams(drawn), to)
            else:
                to[:] = uniforms(drawn)
            if len(drawn) < r:
                floats[3, [i for i, t in enumerate(temps) if t > 0]] = to
        packed[4 * r:o] = top_ks
        if n_pen > 0:
            packed[o:o + r + 1] = list(accumulate(listed, initial=0))
            o += r + 1
            np.concatenate([row.history.both() for row, n_row in zip(rows, listed) if n_row], axis=1,
                           out=packed[o:n].reshape(2, n_pen))
        # rows that are greedy, keep few tokens (the reference's default is top_k = 50) or cut nothing by top-k take
        # the paths that read the logits with the whole GPU
        path = {}
        most, vocab = getattr(self.ops, "FEW_TOKENS", 0), logits.shape[1]
        # (greedy rows without a penalty stay with the one launch: it is short as it is)
        if most and (drawn or n_pen > 0 and vocab > FEW_GREEDY_TOKENS):
            if all(t <= 0 or 1 <= k <= most for t, k in zip(temps, top_ks)):
                path["few"] = True
            elif vocab > SPREAD_TOKENS and all(t <= 0 or k <= most or k >= vocab for t, k in zip(temps, top_ks)):
                path["spread"] = True
        if cuda:
            self.ops.sample_rows(logits, r, pinned, n, n_pen, **path)
            tokens = packed[at:at + r].tolist()
            self._free.append(slot)   # (a call that failed keeps its buffer)
            return tokens
        dev = torch.from_numpy(packed)
        f = dev[:4 * r].view(torch.float32)
        pen = {}
        if n_pen > 0:
            pen = dict(pen_offsets=dev[o - r - 1:o], pen_tokens=dev[o:o + n_pen],
                       pen_counts=dev[o + n_pen:n])
        out = torch.empty(r, dtype=torch.int32, device=self.device)
        self.ops.sample(logits, f[:r], f[3 * r:4 * r], out, top_k=dev[4 * r:5 * r], top_p=f[r:2 * r],
                        rep_penalty=f[2 * r:3 * r], **pen, **path)
        return out.tolist()
