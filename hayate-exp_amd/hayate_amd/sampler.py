"""Token sampling on the GPU for a whole batch at once.

Semantics of the reference's hayate/engine/sampler.py:
* ``validate_parameters`` (:15-37): same checks and messages;
* per row (``_sample_row``, :39-65): temperature 0 is argmax; otherwise the
  scores are logits / temperature, top-k keeps every score >= the k-th
  largest, top-p keeps the shortest prefix of the descending-sorted
  distribution whose mass exceeds p together with the token that crosses
  it, and one token is drawn from the softmax of what is left;
* ``finalize`` (:87-93): append, stop on a stop token or the length limit.

The reference loops over rows in Python, one small kernel chain per row
(:67-85). Here every row of the batch goes through one sort and a handful of
batched ops, with per-row temperature / k / p as tensors, so a tick costs
the same few launches whatever the batch size. 16-bit logits on a HIP device
(the engine's) take hy_sample instead: no sort, the same draws
from the same generator.
"""

from __future__ import annotations

import math
from typing import Optional, Sequence

import numpy as np
import torch

from . import _native, linear


def validate_parameters(temperature, top_k, top_p) -> None:
    """Reject invalid temperature, top-k or nucleus settings (sampler.py:15-37)."""
    if (
        isinstance(temperature, bool)
        or not isinstance(temperature, (int, float))
        or not math.isfinite(temperature)
        or temperature < 0
    ):
        raise ValueError("temperature must be a finite number greater than or equal to 0")
    if top_k is not None and (isinstance(top_k, bool) or not isinstance(top_k, int) or top_k < 1):
        raise ValueError("top_k must be a positive integer or None")
    if top_p is not None and (
        isinstance(top_p, bool)
        or not isinstance(top_p, (int, float))
        or not math.isfinite(top_p)
        or not 0 < top_p <= 1
    ):
        raise ValueError("top_p must be greater than 0 and at most 1, or None")


def sample_batch(logits: torch.Tensor, temperature: Sequence[float],
                 top_k: Sequence[Optional[int]], top_p: Sequence[Optional[float]],
                 generator: Optional[torch.Generator] = None) -> torch.Tensor:
    """One token id per row of logits (n, vocab) -> int64 (n, 1)."""
    if _native_rows(logits, temperature, top_k, top_p):
        return _sample_native(logits, temperature, top_k, top_p, generator)
    n, vocab = logits.shape
    dev = logits.device
    greedy_rows = [i for i, t in enumerate(temperature) if t == 0]
    out = torch.argmax(logits, dim=-1, keepdim=True)
    if len(greedy_rows) == n:
        return out
    rows = [i for i in range(n) if temperature[i] != 0]
    idx = torch.tensor(rows, device=dev, dtype=torch.long)
    temp = torch.tensor([float(temperature[i]) for i in rows], device=dev).unsqueeze(1)
    scores = logits.index_select(0, idx).float() / temp
    sorted_scores, sorted_idx = torch.sort(scores, dim=-1, descending=True)
    # top-k: keep scores >= the k-th largest (ties kept, as masked_fill(< threshold))
    ks = [min(top_k[i], vocab) if top_k[i] is not None else vocab for i in rows]
    kth = sorted_scores.gather(1, torch.tensor(ks, device=dev).unsqueeze(1) - 1)
    keep = scores >= kth
    sorted_scores = sorted_scores.masked_fill(sorted_scores < kth, -torch.inf)
    # top-p over the top-k survivors: remove a token once the mass before it
    # exceeds p (the crossing token stays, so the set is never empty)
    ps = torch.tensor([float(top_p[i]) if top_p[i] is not None else 1.0 for i in rows],
                      device=dev).unsqueeze(1)
    use_p = ps < 1
    probs = torch.softmax(sorted_scores, dim=-1)
    remove_sorted = torch.cumsum(probs, dim=-1) > ps
    remove_sorted = torch.cat(
        [torch.zeros_like(remove_sorted[:, :1]), remove_sorted[:, :-1]], dim=1) & use_p
    remove = torch.zeros_like(remove_sorted).scatter(1, sorted_idx, remove_sorted)
    scores = scores.masked_fill(~keep | remove, -torch.inf)
    drawn = torch.multinomial(torch.softmax(scores, dim=-1), 1, generator=generator)
    out.index_copy_(0, idx, drawn)
    return out


_DTYPES = {torch.bfloat16: 0, torch.float16: 1}
MAX_VOCAB = 4_194_304
_TINY = float(np.finfo(np.float32).tiny)


def _greedy_pays(rows: int, vocab: int) -> bool:
    """Whether hy_sample beats torch.argmax where every row is greedy: one
    workgroup a row against a reduction that is slow on a few long rows only, and
    splits a single row past 131,072 values. Measured on MI355X (us, hy_sample /
    argmax): 20 rows of 151,936 17 / 38, 128 of them 32 / 48, 256 53 / 49; 20 of
    65,536 16 / 19, 64 of them 22 / 20; 20 of 32,000 17 / 12; one of 151,936 14 / 12,
    of 100,352 14 / 26."""
    return vocab >= 65_536 and rows * 1400 <= vocab and (rows > 1 or vocab <= 131_072)


def _native_rows(logits: torch.Tensor, temperature, top_k, top_p) -> bool:
    """True when hy_sample takes these rows: 16-bit logits on the current HIP
    device, contiguous along the vocabulary, whole numbers as top_k (the path
    below refuses others), temperatures whose scores keep the logits' order
    (outside [1e-30, 1e30] they vanish or overflow and become equal), nothing
    watching the ops, and not only greedy rows that argmax is faster for."""
    return (type(logits) is torch.Tensor and logits.dtype in _DTYPES and logits.is_cuda
            and logits.dim() == 2 and logits.shape[0] > 0 and 0 < logits.shape[1] <= MAX_VOCAB
            and logits.stride(1) == 1
            and len(temperature) == len(top_k) == len(top_p) == logits.shape[0]
            and all(t == 0 or 1e-30 <= t <= 1e30 for t in temperature)
            and all(k is None or (type(k) is int or isinstance(k, np.integer)) and k >= 1
                    for k in top_k)
            and all(p is None or p > 0 for p in top_p)
            and (any(temperature) or _greedy_pays(*logits.shape))
            and linear.unwatched() and logits.device.index == torch.cuda.current_device())


def _sample_native(logits, temperature, top_k, top_p, generator):
    n, vocab = logits.shape
    dev = logits.device
    temp = np.asarray(list(map(float, temperature)), dtype=np.float32)
    k = np.asarray([vocab if v is None else min(v, vocab) for v in top_k], dtype=np.int32)
    # a top_p that fp32 rounds to 0 keeps what the smallest number does: the
    # logits with no mass before them
    p = np.asarray([1.0 if v is None else max(float(v), _TINY) for v in top_p], dtype=np.float32)
    drawn = int(np.count_nonzero(temp))
    noise = valid = None
    if drawn:
        # the noise torch.multinomial draws for these rows' probabilities
        noise = torch.empty((drawn, vocab), device=dev).exponential_(1, generator=generator)
        valid = torch.empty((), dtype=torch.bool, device=dev)
    out = torch.empty((n, 1), dtype=torch.long, device=dev)
    lib = _native.lib()
    work = torch.empty(lib.hy_sample_workspace_bytes(n, vocab), dtype=torch.uint8, device=dev)
    rc = lib.hy_sample(
        logits.data_ptr(), logits.stride(0), _DTYPES[logits.dtype], n, vocab, temp.ctypes.data,
        k.ctypes.data, p.ctypes.data, noise.data_ptr() if drawn else None, out.data_ptr(),
        valid.data_ptr() if drawn else None, work.data_ptr(), work.numel(),
        _native.stream_of(logits.get_device()))
    if rc:
        _native.check(rc, "hy_sample")
    if drawn:
        torch._assert_async(valid, "logits hold NaN or have no finite maximum")
    return out


class Sampler:
    """Samples the next token of each request (sampler.py:8-93)."""

    def __init__(self, tokenizer=None, stop_token_ids: Optional[set[int]] = None,
                 generator: Optional[torch.Generator] = None):
        self.tokenizer = tokenizer
        self.stop_token_ids = set(stop_token_ids or ())
        self.generator = generator

    validate_parameters = staticmethod(validate_parameters)

    def sample(self, logits: torch.Tensor, requests=None) -> torch.Tensor:
        if requests is None:
            return torch.argmax(logits, dim=-1, keepdim=True)
        if logits.ndim != 2 or logits.shape[0] != len(requests):
            raise ValueError("sampling logits must have one vocabulary row per request")
        for r in requests:
            validate_parameters(r.temperature, r.top_k, r.top_p)
        return sample_batch(logits, [r.temperature for r in requests],
                            [r.top_k for r in requests], [r.top_p for r in requests],
                            self.generator)

    def finalize(self, request, tok: int) -> None:
        request.tokens.append(tok)
        if tok in self.stop_token_ids or len(request.tokens) >= request.max_tokens:
            request.is_completed = True
            if self.tokenizer is not None:
                request.response = self.tokenizer.decode(request.tokens,
                                                         skip_special_tokens=True)
