"""Sampling parameters, the counter-based random stream, and the device sampler,
named from Python (sampling/sampler.cpp has them, and what the reference does:
src/main.cpp:23-84).
"""
from __future__ import annotations

import ctypes
import struct
from dataclasses import dataclass
from typing import List, Sequence

from .. import native

_RECORD = struct.Struct("@fif4xQ")      # a SamplingParams of the library's
DEFAULT_TOP_K = 512          # the reference's cut when --top-k is 0: src/main.cpp:47-48


class _Recorded:
    """Where a SamplingParams keeps its record: beside its attributes, which are what it is given."""
    __slots__ = ("_record",)


@dataclass(frozen=True)
class SamplingParams(_Recorded):
    temperature: float = 0.0     # <= 0: greedy (src/main.cpp:24,31-38)
    top_k: int = 0               # 0: the reference's default of 512
    top_p: float = 1.0
    seed: int = 42               # src/main.cpp:27

    def __post_init__(self):
        if type(self) is SamplingParams:      # (a class derived from it may not have its numbers yet, or change them)
            _pack(self)

    def __getstate__(self):
        return self.__dict__

    def effective_top_k(self) -> int:
        return self.top_k if self.top_k > 0 else DEFAULT_TOP_K


_keep = _Recorded._record.__set__


def _pack(p):
    """What the library reads of a request, once: four lists of a number a request each took longer at every call than its kernels' launches.  None for
    numbers of other types or out of their type's range, which are converted at every call."""
    t, k, q, s = p.temperature, p.top_k, p.top_p, p.seed
    try:
        plain = type(k) is type(s) is int and (type(t) is float or type(t) is int) and (type(q) is float or type(q) is int)
        _keep(p, _RECORD.pack(t, k, q, s & ((1 << 64) - 1)) if plain else None)
    except (struct.error, OverflowError):
        _keep(p, None)


def uniform(seed: int, request: int, n_generated: int) -> float:
    """A number in [0, 1) with 24 random bits (exact in float32), a pure function of its three keys."""
    mask = (1 << 64) - 1
    return float(native.lib().ti_uniform(seed & mask, request & mask, n_generated & mask))


class Sampler:
    """Draws one token per row of logits on the device."""

    def __init__(self, ops, device=None):
        self.ops = ops
        self._ptr = native.pointer("ti_sampler_create", ops._ptr)

    def __del__(self):
        try:
            if native._lib is not None:
                native._lib.ti_sampler_release(self._ptr)
        except Exception:  # noqa: BLE001
            pass

    @staticmethod
    def _arguments(n, params, requests, counters):
        mask = (1 << 64) - 1
        requests, counters = tuple(requests), tuple(counters)     # (any iterable)
        try:
            # packed at once: an element of a ctypes array at a time takes longer than the kernels (70 us for 64 rows, this 15)
            if not len(params) == len(requests) == len(counters) == n:
                raise ValueError
            floats, ints, words = f"{n}f", f"{n}i", f"{n}q"
            return (struct.pack(floats, *[p.temperature for p in params]), struct.pack(ints, *[p.top_k for p in params]),
                    struct.pack(floats, *[p.top_p for p in params]), struct.pack(f"{n}Q", *[p.seed & mask for p in params]),
                    struct.pack(words, *requests), struct.pack(words, *counters))
        except (struct.error, OverflowError, ValueError, TypeError):     # numbers out of their type's range, which ctypes cuts to it, or too few of them
            return ((ctypes.c_float * n)(*[p.temperature for p in params]), (ctypes.c_int * n)(*[p.top_k for p in params]),
                    (ctypes.c_float * n)(*[p.top_p for p in params]), (ctypes.c_uint64 * n)(*[p.seed & mask for p in params]),
                    (ctypes.c_int64 * n)(*requests), (ctypes.c_int64 * n)(*counters))

    @staticmethod
    def _records(n, params, requests, counters):
        """The same from the parameters' own records, or None where one of them can have none or a number does not fit (64 rows: 5 us, 17 above; a whole
        call of 64 rows of 151,936 61.6 -> 55.3)."""
        try:
            if not len(params) == len(requests) == len(counters) == n:
                return None
            words = f"{n}q"
            try:
                records = b"".join([p._record for p in params])
            except AttributeError:
                if {*map(type, params)} != {SamplingParams}:
                    return None
                for p in params:              # (of a pickle or a copy)
                    _pack(p)
                records = b"".join([p._record for p in params])
            if len(records) != n * _RECORD.size:      # (somebody else's attribute)
                return None
            return records, struct.pack(words, *requests), struct.pack(words, *counters)
        except (AttributeError, TypeError, struct.error, OverflowError):
            return None

    def sample(self, logits, params: Sequence[SamplingParams], requests: Sequence[int], counters: Sequence[int]) -> List[int]:
        """logits f32 [n, V]; row i belongs to request number `requests[i]`, which has generated
        `counters[i]` tokens so far."""
        n = logits.shape[0]
        native.ensure_kernels(["sampling"])
        out = (ctypes.c_int * n)()
        requests, counters = tuple(requests), tuple(counters)     # (any iterable)
        records = self._records(n, params, requests, counters)
        if records:
            native.call("ti_sampler_sample_records", self._ptr, native.describe_many([logits]), n, *records, out)
        else:
            native.call("ti_sampler_sample", self._ptr, native.describe_many([logits]), n,
                        *self._arguments(n, params, requests, counters), out)
        return out[:]

    def sample_async(self, logits, params: Sequence[SamplingParams], requests: Sequence[int], counters: Sequence[int],
                     feed=None):
        """The same without waiting: returns a ticket for `collect`.  `feed`: an engine whose token
        feedback receives the ids too, so that its next step can name them with
        `token_from_feedback(row)` before they are read.  At most two calls may be under way."""
        n = logits.shape[0]
        native.ensure_kernels(["sampling"])
        ticket = ctypes.c_uint64()
        requests, counters = tuple(requests), tuple(counters)
        records = self._records(n, params, requests, counters)
        feeds = feed._ptr if feed is not None else None
        if records:
            native.call("ti_sampler_sample_records_async", self._ptr, native.describe_many([logits]), n, *records, feeds, ctypes.byref(ticket))
        else:
            native.call("ti_sampler_sample_async", self._ptr, native.describe_many([logits]), n,
                        *self._arguments(n, params, requests, counters), feeds, ctypes.byref(ticket))
        return (ticket.value, n)

    def collect(self, ticket) -> List[int]:
        """Wait for the ids of a `sample_async` call."""
        number, n = ticket
        out = (ctypes.c_int * n)()
        native.call("ti_sampler_collect", self._ptr, number, n, out)
        return out[:]
