"""Token sampling on the gfx950 sampling kernel.

Mirrors ``src/engine/sampling.rs``:

* ``SamplingParams`` with ``normalized()`` (``:8-47``);
* ``Sampler.sample_batch(logits, params)`` -> list of ids, raising
  ``SamplingError`` for an invalid distribution (``:281-372``, ``sampled_ids``);
* ``Sampler.defer_batch(logits, params)`` -> ``PendingSample`` whose ids are
  copied into pinned host memory behind an event (the reference's ``Readback``,
  ``:193-237``); ``relay()`` gives the device ids clamped at 0 for the next
  step's embedding, ``finish()`` waits and validates.

Unlike the reference, which groups rows by identical parameters and launches
one FlashInfer call per group (``:343-371``), one library call serves the
whole heterogeneous batch: the parameters travel as per-row device arrays.
The call is one launch, or two to six where rows are spread over several
workgroups. The random stream is (seed, offset): ``manual_seed`` resets both
and every sampling call advances the offset by one.
"""
from __future__ import annotations

import math
from collections import Counter
from dataclasses import dataclass, replace

import torch

from ._native import NativeError, check, lib, stream_of


class SamplingError(RuntimeError):
    """Invalid logits shape, parameter count mismatch or invalid distribution."""


@dataclass(frozen=True)
class SamplingParams:
    temperature: float = 0.0
    top_k: int = -1
    top_p: float = 1.0
    ignore_eos: bool = False
    max_tokens: int = 1024

    def normalized(self) -> "SamplingParams":
        top_p = self.top_p if (math.isfinite(self.top_p) and 0.0 <= self.top_p <= 1.0) else 1.0
        return replace(self, max_tokens=max(self.max_tokens, 1), top_p=top_p)


# The split sampler cuts rows with a top_k up to this among their listed largest logits. A
# larger one below the vocabulary takes one workgroup per row from the start (k 200, 64 rows of
# 151,936: 61 us; as a fallback within the split call 92).
LISTED_TOP_K = 128
# From this many rows on an all-greedy batch takes one workgroup per row and one launch: what the
# split call still gives there is small below 100,000 columns (127 fp32 rows of 80,000: 3%) and gone
# in a full round (151,936 columns, one workgroup per row against split: one row 28.6 us and 11.5,
# 128 rows 32.2 and 23.9, 256 rows 33.0 and 34.9).
GREEDY_ROWS = 128
# Rows that one workgroup each runs side by side, one on a CU; more take another round.
ROUND_ROWS = 256


def _split_pays(rows: int, vocab: int, greedy: int, race: int, listed: int, widest_k: int,
                top_p: int, fp32: bool, vec: bool) -> bool:
    """Whether rows spread over several workgroups beat one workgroup per row, for a batch of so
    many greedy, unfiltered, listed top-k (the largest ``widest_k``) and top-p rows; ``vec``: every
    row starts on 16 bytes.

    The vocabulary from which it does, measured at 13 vocabularies from 16,385 to 128,256, 14 row
    counts up to 1,024, bf16 and fp32. The split call has a launch more and a pass that grows with
    the rows; one workgroup per row costs the same up to 256 rows and again for each further 256,
    so that a full round needs the longest rows. Listed rows gain at every size. us, one workgroup
    per row against split: greedy, 16 rows of 32,000 12.8 and 13.7, of 100,000 23.1 and 14.2;
    unfiltered, 64 of 32,000 22.5 and 17.4, 256 24.1 and 28.8, 256 of 50,257, which one workgroup
    reads token by token, 58 and 43; top-p, 256 of 32,000 78 and 104, of 80,000 144 and 122, 320 of
    32,000 141 and 128; top-k 50 and top-p 0.9, 256 of 20,000 27.5 and 22.3. In a batch of several
    kinds one workgroup per row waits for the slowest row and the split call for their mean (a
    fifth top-p, 256 rows of 32,000: 82 and 58)."""
    if greedy == rows:
        return rows < GREEDY_ROWS and vocab >= 40_000 + 200 * rows
    # Nine to twelve segments bound a large k loosely (k 128 of 16,385 at 256 rows: 26 and 72).
    if widest_k > 96 and vocab < 49_152:
        return False
    rounds = -(-rows // ROUND_ROWS)
    fill = (rows / (rounds * ROUND_ROWS)) ** 2
    if top_p:
        share = top_p / rows
        if rounds == 1:
            need = (97_000 if fp32 else 65_000) * share * fill
        else:
            need = (70_000 if fp32 else 36_000) * math.sqrt(share) * fill
    else:
        need = (12_000 + (60_000 if rounds == 1 else 32_000) * fill) * race / rows if vec else 0
    return vocab >= need


_DTYPES = {torch.bfloat16: 0, torch.float16: 1, torch.float32: 2}


def _validate_logits(logits: torch.Tensor) -> None:
    if logits.dim() != 2 or logits.size(1) <= 0:
        raise SamplingError(f"logits must be 2-D (num_reqs, vocab_size), got {list(logits.shape)}")
    if not logits.is_cuda:
        raise NativeError("sampling requires GPU logits")
    if logits.dtype not in _DTYPES:
        raise NativeError(f"unsupported logits dtype {logits.dtype}")
    if logits.stride(1) != 1:
        raise NativeError("logits rows must be contiguous")


class PendingSample:
    """One in-flight sampling launch; ids land in pinned host memory behind an event."""

    def __init__(self, ids: torch.Tensor, logits: torch.Tensor):
        self.ids = ids
        self._logits = logits  # keeps the input alive until the copy has run
        self._host = torch.empty(ids.shape, dtype=ids.dtype, pin_memory=True)
        self._host.copy_(ids, non_blocking=True)
        self._event = torch.cuda.Event()
        self._event.record(torch.cuda.current_stream(ids.device))

    def relay(self) -> torch.Tensor:
        """Device ids with the -1 sentinel clamped to 0, safe to feed an embedding."""
        return self.ids.clamp_min(0)

    def ready(self) -> bool:
        return self._event.query()

    def finish(self) -> list[int]:
        self._event.synchronize()
        ids = self._host.tolist()
        if any(i < 0 for i in ids):
            raise SamplingError("invalid probability distribution")
        return ids


class Sampler:
    """Samples one next-token id per logits row, the whole heterogeneous batch in one call."""

    def __init__(self, seed: int = 0):
        self.manual_seed(seed)
        self._param_key: tuple | None = None
        self._param_objs: tuple | None = None
        self._params: tuple[torch.Tensor, torch.Tensor, torch.Tensor] | None = None
        self._top_p_rows = False  # some row of _params may be cut by top_p alone
        self._kinds = (0, 0, 0, 0, 0)  # _split_pays' greedy, race, listed, widest_k and top_p
        self._large_k: int | None = None  # smallest top_k of _params beyond LISTED_TOP_K

    def manual_seed(self, seed: int) -> None:
        self.seed = int(seed) & (2 ** 64 - 1)
        self.offset = 0

    def _device_params(self, params_list, device: torch.device):
        # A decode step usually passes the very objects of the previous step (each running
        # request keeps its SamplingParams, which are frozen): reuse the device arrays after
        # an identity check instead of normalising every row again on the host.
        objs = self._param_objs
        if (objs is not None and self._param_key is not None and self._param_key[0] == device
                and len(objs) == len(params_list)
                and all(a is b for a, b in zip(params_list, objs))):
            return self._params
        # Plain walks over the fields (``normalized`` would copy every object): a batch whose
        # members changed comes here on each step that a request joins or leaves.
        temps = [p.temperature for p in params_list]
        ks = [p.top_k for p in params_list]
        ps = [p.top_p if 0.0 <= p.top_p <= 1.0 else 1.0 for p in params_list]
        key = (device, temps, ks, ps)
        if key != self._param_key:
            n = len(temps)
            host = torch.empty(3 * n, dtype=torch.float32, pin_memory=True)
            k = torch.tensor(ks, dtype=torch.int32)
            torch.cat((torch.tensor(temps, dtype=torch.float32), k.view(torch.float32),
                       torch.tensor(ps, dtype=torch.float32)), out=host)  # top-k bit for bit
            dev = host.to(device, non_blocking=True)
            self._params = (dev[:n], dev[n:2 * n].view(torch.int32), dev[2 * n:])
            greedy = race = listed = widest = top_p = 0
            self._large_k = None
            for (t, k, p), rows in Counter(zip(temps, ks, ps)).items():
                if t <= 0 or p == 0:
                    greedy += rows
                elif 0 < k <= LISTED_TOP_K:
                    listed += rows
                    widest = max(widest, k)
                else:
                    if k > LISTED_TOP_K:
                        self._large_k = k if self._large_k is None else min(self._large_k, k)
                    top_p += rows if p < 1 else 0
                    race += rows if p >= 1 else 0
            self._top_p_rows = top_p > 0
            self._kinds = (greedy, race, listed, widest, top_p)
            self._param_key = key
        self._param_objs = tuple(params_list)  # last: a build that raised is not taken for built
        return self._params

    def sample_batch_device(self, logits: torch.Tensor, params_list, *,
                            out: torch.Tensor | None = None) -> torch.Tensor:
        """Device int64 ids [rows]; an invalid distribution yields -1 in its row."""
        _validate_logits(logits)
        rows = logits.size(0)
        if rows != len(params_list):
            raise SamplingError(
                f"SamplingParams count ({len(params_list)}) must equal logits rows ({rows})")
        if out is None:
            out = torch.empty(rows, dtype=torch.int64, device=logits.device)
        if rows == 0:
            return out
        temperature, top_k, top_p = self._device_params(params_list, logits.device)
        args = (logits.data_ptr(), rows, logits.size(1), logits.stride(0),
                _DTYPES[logits.dtype], temperature.data_ptr(), top_k.data_ptr(),
                top_p.data_ptr(), self.seed, self.offset, out.data_ptr())
        need = 0
        if ((self._large_k is None or self._large_k >= logits.size(1))
                and _split_pays(rows, logits.size(1), *self._kinds,
                                logits.dtype == torch.float32, logits.stride(0) % 8 == 0)):
            need = lib().mi355x_sample_workspace_bytes(rows, logits.size(1), self._top_p_rows)
        ws = None
        if need:
            try:
                ws = torch.empty(need, dtype=torch.uint8, device=logits.device)
            except torch.OutOfMemoryError:
                pass  # one workgroup per row needs no workspace
        if ws is not None:
            check(lib().mi355x_sample_split(*args, self._top_p_rows, ws.data_ptr(), need,
                                            stream_of(logits)), "sample")
        else:
            check(lib().mi355x_sample(*args, stream_of(logits)), "sample")
        self.offset += 1
        return out

    def sample_batch(self, logits: torch.Tensor, params_list) -> list[int]:
        return self.defer_batch(logits, params_list).finish()

    def defer_batch(self, logits: torch.Tensor, params_list) -> PendingSample:
        return PendingSample(self.sample_batch_device(logits, params_list), logits)


__all__ = ["SamplingParams", "Sampler", "PendingSample", "SamplingError"]
