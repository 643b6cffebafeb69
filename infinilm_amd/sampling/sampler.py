"""From rows of logits to tokens: argmax for greedy rows, temperature / top-k / top-p otherwise.

Reference: one `random_sample_(out, row, random_val, top_p, top_k, temperature)` call per request
in a host loop, random_val from a `std::mt19937` seeded by `std::random_device`
(csrc/engine/rank_worker.cpp:27,467-513): not reproducible.  Here all rows are sampled by one
kernel launch, and the uniform number of a row is a pure function of (seed, request, index of the
generated token), so a request's tokens do not depend on what else is in the batch or on how often
it was preempted.
"""
from __future__ import annotations

import operator
from array import array
from typing import List, Sequence, Tuple

import numpy as np
import torch

from .. import kernels
from .params import SamplingParams

_MASK = (1 << 64) - 1


def _mix(x: int) -> int:
    """splitmix64 finaliser."""
    x = (x + 0x9E3779B97F4A7C15) & _MASK
    x = ((x ^ (x >> 30)) * 0xBF58476D1CE4E5B9) & _MASK
    x = ((x ^ (x >> 27)) * 0x94D2049BB133111B) & _MASK
    return x ^ (x >> 31)


def uniform_for(seed: int, request_key: int, index: int) -> float:
    """u in [0, 1) with 24 bits, a pure function of its arguments."""
    x = _mix(_mix(_mix(seed & _MASK) ^ (request_key & _MASK)) ^ (index & _MASK))
    return (x >> 40) / float(1 << 24)


def _words(values: Sequence[int]) -> array:
    try:
        return array("Q", values)
    except OverflowError:     # negative ones wrap, and of numbers of more than 64 bits the lowest count
        return array("Q", [operator.index(v) & _MASK for v in values])


def _int32s(values: Sequence[int]) -> array:
    """The rows' top-k as the kernels take them: numbers with a fraction lose it, those beyond 32 bits keep the whole
    vocabulary as the largest of them does."""
    try:
        return array("i", values)
    except (TypeError, OverflowError):
        return array("i", [int(min(v, 0x7fffffff)) for v in values])


def _uniforms_into(out: int, seeds: Sequence[int], request_keys: Sequence[int], indices: Sequence[int]) -> None:
    """`uniform_for` of every row, float32 at the host address `out`, in native code (0.1 us a row against 1.4, or 23 us for 64 rows
    at once in numpy).  The arrays live until the call returns."""
    n, first = len(seeds), seeds[0]
    one = seeds.count(first) == n      # the engine's own seed, as a rule
    s, k, i = None if one else _words(seeds), _words(request_keys), _words(indices)
    if not len(k) == len(i) == n:
        raise ValueError("a seed, a key and an index a row")
    kernels.uniforms(out, None if one else s.buffer_info()[0], _words((first,))[0], k.buffer_info()[0], i.buffer_info()[0], n)


def uniforms_for(seeds: Sequence[int], request_keys: Sequence[int], indices: Sequence[int]) -> np.ndarray:
    """`uniform_for` of every row; one by one where there is no native library (they are numbers of the host, and need no GPU)."""
    out = np.empty((len(seeds),), dtype=np.float32)
    if len(seeds):
        try:
            _uniforms_into(out.ctypes.data, list(seeds), request_keys, indices)
        except (OSError, RuntimeError):
            out[:] = [uniform_for(*map(operator.index, row)) for row in zip(seeds, request_keys, indices)]
    return out


class Sampler:
    def __init__(self, seed: int = 0):
        self.seed = int(seed)
        # pinned host memory for the rows' parameters: two buffers in turn, each waited for only when
        # its own last copy may still be reading it (a step may be launched before the one before it
        # has run)
        self._staging = [None, None]
        self._copied = [None, None]
        self._copied_on = [-1, -1]
        self._turn = 0

    def _event(self, t: int, device: int):
        """The event of buffer t's copy.  It belongs to the device that it was first recorded on, and the next logits may lie on another."""
        if self._copied_on[t] != device:
            self._copied[t], self._copied_on[t] = torch.cuda.Event(), device
        return self._copied[t]

    def sample(self, logits: torch.Tensor, rows: Sequence[Tuple[SamplingParams, int, int]]) -> List[int]:
        """`rows[i]` = (params, request key, index of the token being generated) for logits[i]."""
        if logits.shape[0] == 0 and not rows:
            return []
        return self.sample_device(logits, rows).tolist()

    def sample_device(self, logits: torch.Tensor, rows: Sequence[Tuple[SamplingParams, int, int]]) -> torch.Tensor:
        """The same, the tokens left on the device (int32 [rows]); nothing waits for the stream."""
        n = logits.shape[0]
        if n != len(rows):
            raise ValueError(f"{n} rows of logits for {len(rows)} requests")
        if n == 0:
            raise ValueError("no rows to sample")
        if all(p.greedy for p, _, _ in rows):
            return kernels.argmax(logits)
        params, keys, indices = zip(*rows)
        top_k = [p.top_k for p in params]
        few = 0 < min(top_k) and kernels.sample_one_reading(n, logits.shape[1], max(top_k))
        temperature, top_p = array("f", [p.temperature for p in params]), array("f", [p.top_p for p in params])
        seeds = [self.seed if p.seed is None else p.seed for p in params]
        if n <= kernels.SAMPLE_HOST_ROWS:      # they travel with the launch
            one = seeds.count(seeds[0]) == n
            return kernels.sample_host(logits, temperature, _int32s(top_k), top_p, None if one else _words(seeds), _words(seeds[:1])[0], _words(keys),
                                       _words(indices), few)
        # temperature, top_k, top_p and the uniform numbers in one pinned buffer and one copy that
        # queues behind the step (a copy from pageable memory would make the host wait for the step
        # and the device wait for four copies)
        dev = logits.device
        t = self._turn = self._turn ^ 1
        if self._copied[t] is not None:
            self._copied[t].synchronize()
        if self._staging[t] is None or self._staging[t][0].numel() < 4 * n:
            buf = torch.empty((4 * max(n, 64),), dtype=torch.float32, pin_memory=dev.type == "cuda")
            self._staging[t] = (buf, memoryview(buf.numpy()).cast("B"), buf.data_ptr())
        buf, raw, at = self._staging[t]
        raw[0:4 * n] = memoryview(temperature).cast("B")
        raw[4 * n:8 * n] = memoryview(_int32s(top_k)).cast("B")
        raw[8 * n:12 * n] = memoryview(top_p).cast("B")
        _uniforms_into(at + 12 * n, seeds, keys, indices)
        d = torch.empty((4 * n,), dtype=torch.float32, device=dev)
        d.copy_(buf[:4 * n], non_blocking=True)
        if dev.type == "cuda":
            self._event(t, dev.index).record()
        return kernels.sample_packed(logits, d, few=few)
