"""ctypes binding of libhayate_attn.so (the C ABI in include/hayate_attn.h).

The shared library is the only compute path: if it is missing this module
raises instead of substituting anything else. Host-only entry points
(hy_plan_tick, hy_decode_workspace_bytes, hy_version) work without a GPU.
"""

from __future__ import annotations

import ctypes
import os
from typing import Optional

import numpy as np
import torch

LIB_NAME = "libhayate_attn.so"
# HAYATE_ATTN_LIB may point at another build of the same library.
LIB_PATH = os.environ.get(
    "HAYATE_ATTN_LIB", os.path.join(os.path.dirname(os.path.abspath(__file__)), LIB_NAME)
)

HY_OK = 0
HY_EINVAL = -1
HY_ELAUNCH = -2
HY_EUNSUPPORTED = -3
HY_ENOSPACE = -4
# Static device scratch of hy_paged_decode_append_noalloc (bytes per GPU).
NOALLOC_SCRATCH_BYTES = 8 * 1024 * 1024

_P = ctypes.c_void_p
_I64 = ctypes.c_int64
_I32 = ctypes.c_int32
_F32 = ctypes.c_float

# Argument signatures, in header order.
_SIGNATURES = {
    "hy_version": ([], ctypes.c_int),
    "hy_last_error": ([], ctypes.c_char_p),
    "hy_kv_append": (
        [_P, _P, _I64, _P, _I64, _I64, _I64, _P, _I64, _I64, _I64, _P, _P, _P,
         _I64, _I32, _I32, _I32, _I32, _I32, _P],
        ctypes.c_int,
    ),
    "hy_qknorm_rope_append": (
        [_P, _I64, _I64, _I64, _P, _I64, _I64, _I64, _P, _I64, _I64, _I64, _P,
         _I64, _I64, _I64, _P, _P, _F32, _F32, _P, _P, _I32, _P, _P, _I64, _P, _P,
         _P, _I64, _I32, _I32, _I32, _I32, _I32, _I32, _P],
        ctypes.c_int,
    ),
    "hy_page_gather": (
        [_P, _I64, _I64, _P, _I32, _P, _I32, _I32, _I32, _I32, _P],
        ctypes.c_int,
    ),
    "hy_page_scatter": (
        [_P, _I64, _I64, _P, _I32, _P, _I64, _I64, _I64, _I32, _I32, _I32,
         _I32, _P],
        ctypes.c_int,
    ),
    "hy_plan_tick": (
        [_P, _P, _I32, _I32, _I32, _I32, _I32, _I32, _P, _I32, _P, _I32, _P, _I32, _P,
         _I32, _P],
        ctypes.c_int,
    ),
    "hy_decode_workspace_bytes": ([_I32, _I32, _I32], ctypes.c_int64),
    "hy_paged_decode": (
        [_P, _I64, _I64, _I64, _P, _I64, _I64, _I64, _P, _P, _I64, _P, _I64,
         _P, _P, _I32, _I32, _P, _I64, _I32, _I32, _I32, _I32, _I32, _F32, _P],
        ctypes.c_int,
    ),
    "hy_paged_decode_append": (
        [_P, _I64, _I64, _I64, _P, _I64, _I64, _I64, _P, _I64, _I64, _I64, _P, _I64, _I64,
         _I64, _P, _P, _F32, _F32, _P, _P, _I32, _P, _P, _P, _I64, _P, _I64, _P, _P, _P, _I32,
         _I32, _P, _I64, _I32, _I32, _I32, _I32, _I32, _F32, _P],
        ctypes.c_int,
    ),
    "hy_paged_decode_merge": (
        [_P, _I64, _I64, _I64, _P, _P, _I32, _I32, _P, _I64, _I32, _I32, _P],
        ctypes.c_int,
    ),
    "hy_paged_decode_append_noalloc": (
        [_P, _I64, _I64, _I64, _P, _I64, _I64, _I64, _P, _I64, _I64, _I64, _P, _I64, _I64,
         _I64, _P, _P, _F32, _F32, _P, _P, _I32, _P, _I64, _I64, _I64, _P, _P, _I64, _P, _I64, _P,
         _P, _P, _I32, _P, _I32, _I32, _I32, _I32, _I32, _I32, _I32, _F32, _P],
        ctypes.c_int,
    ),
    "hy_prefill_tile_rows": ([], ctypes.c_int32),
    "hy_prefill_workspace_bytes": ([_I32, _I32, _I32], ctypes.c_int64),
    "hy_paged_prefill": (
        [_P, _I64, _I64, _I64, _P, _I64, _I64, _I64, _P, _P, _I64, _P, _I64,
         _P, _P, _P, _I32, _I32, _P, _I64, _I32, _I32, _I32, _I32, _I32, _F32, _P],
        ctypes.c_int,
    ),
    "hy_paged_prefill_merge": (
        [_P, _I64, _I64, _I64, _P, _P, _I32, _I32, _P, _I64, _I32, _I32, _I32, _P],
        ctypes.c_int,
    ),
    "hy_norm_linear": (
        [_P, _I64, _I32, _I32, _P, _F32, _P, _P, _I64, _I32, _P, _I64, _P],
        ctypes.c_int,
    ),
    "hy_sample": (
        [_P, _I64, _I32, _I32, _I32, _P, _P, _P, _P, _P, _P, _P, _I64, _P],
        ctypes.c_int,
    ),
    "hy_sample_workspace_bytes": ([_I32, _I32], ctypes.c_int64),
    "hy_linear_tiles": (
        [_P, _I64, _I32, _I32, _P, _P, _I64, _I32, _P, _I64, _P, _I64, _P, _I64, _P],
        ctypes.c_int,
    ),
    "hy_linear_tiles_workspace_bytes": ([_I32, _I32, _I32, _I32], ctypes.c_int64),
    "hy_row_norm": ([_P, _I64, _I32, _I32, _P, _F32, _P, _P], ctypes.c_int),
    "hy_linear_add": (
        [_P, _I64, _I32, _I32, _P, _I64, _I32, _P, _I64, _P, _I64, _P],
        ctypes.c_int,
    ),
}

EXPORTED_SYMBOLS = tuple(_SIGNATURES)

_lib: Optional[ctypes.CDLL] = None


class NativeLibraryMissing(RuntimeError):
    """The HIP library has not been built; there is no other compute path."""


def lib() -> ctypes.CDLL:
    """Load (once) and return the native library, or raise loudly."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise NativeLibraryMissing(
            f"{LIB_PATH} is not built; run `make -C hayate-exp_amd/csrc` "
            "(or __graft_entry__.build()) first"
        )
    handle = ctypes.CDLL(LIB_PATH, mode=ctypes.RTLD_LOCAL)
    for name, (argtypes, restype) in _SIGNATURES.items():
        fn = getattr(handle, name)
        fn.argtypes = argtypes
        fn.restype = restype
    _lib = handle
    return handle


def stream_of(device_index: int) -> int:
    """Handle of the device's current stream, without building a Stream object
    (0.1 us against 1.8, and every call into the library asks for it)."""
    return torch._C._cuda_getCurrentRawStream(device_index)


def last_error() -> str:
    msg = lib().hy_last_error()
    return msg.decode() if msg else ""


def check(rc: int, what: str) -> None:
    """Map a C return code onto the exception types the reference raises."""
    if rc == HY_OK:
        return
    msg = f"{what}: {last_error()}"
    if rc == HY_EINVAL:
        raise ValueError(msg)
    if rc == HY_EUNSUPPORTED:
        raise NotImplementedError(msg)
    if rc == HY_ENOSPACE:
        raise MemoryError(msg)
    raise RuntimeError(msg)


class TickPlan:
    """Host copy of one tick's work lists (hy_plan_tick)."""

    __slots__ = ("decode", "n_chunks", "merge", "n_slots", "prefill", "prefill_merge",
                 "n_prefill_slots")

    def __init__(self, decode, n_chunks, merge, n_slots, prefill, prefill_merge,
                 n_prefill_slots):
        # int32 (n_chunks + n_pieces, 8): chunk records {piece_begin,
        # piece_end, n_slices, 0..} then piece records {seq, tok_begin,
        # tok_end, slot_base, slice_begin, q_row, 0, 0}
        self.decode = decode
        self.n_chunks = n_chunks
        self.merge = merge                  # int32 (n, 4) {seq, first_slot, num_partials, q_row}
        self.n_slots = n_slots
        self.prefill = prefill              # int32 (n, 8) {seq, q0, q1, kv0, kv1, slot, q_row, cache}
        self.prefill_merge = prefill_merge  # int32 (n, 8) {seq, q0, q1, first_slot, splits, q_row, ..}
        self.n_prefill_slots = n_prefill_slots


def plan_tick(
    q_lens: np.ndarray,
    kv_lens: np.ndarray,
    num_q_heads: int,
    num_kv_heads: int,
    page_size: int,
    num_cus: int,
    tokens_per_split: int = 0,
) -> TickPlan:
    """Run the native tick planner."""
    q_lens = np.ascontiguousarray(q_lens, dtype=np.int32)
    kv_lens = np.ascontiguousarray(kv_lens, dtype=np.int32)
    n = int(q_lens.shape[0])
    group = max(1, num_q_heads // max(1, num_kv_heads))
    tile = max(1, int(lib().hy_prefill_tile_rows()) // group)
    dec_mask = q_lens == 1
    pre_mask = q_lens > 1
    dec_tokens = int(kv_lens[dec_mask].astype(np.int64).sum())
    # the planner takes num_cus <= 0 as 256 CUs
    cus = num_cus if num_cus > 0 else 256
    max_chunks = 2 * cus + 1
    if tokens_per_split > 0:
        max_chunks = max(max_chunks, dec_tokens // tokens_per_split + 1)
    # chunk records + piece records: a piece starts at every chunk boundary
    # and every sequence; chunks also close at the kernel's piece limit
    n_dec = int(dec_mask.sum())
    dec_cap = 2 * (max_chunks + n_dec) + 2
    n_tiles = int(((q_lens[pre_mask].astype(np.int64) + tile - 1) // tile).sum())
    max_steps = int((kv_lens.max() + 63) // 64) if n else 1
    # the planner splits a tile into ranges of at least two 64-key steps
    pre_cap = n_tiles * max(1, max_steps // 2 + 1) + 1
    dec = np.zeros((dec_cap, 8), dtype=np.int32)
    mrg = np.zeros((n + 1, 4), dtype=np.int32)
    pre = np.zeros((pre_cap, 8), dtype=np.int32)
    pmrg = np.zeros((n_tiles + 1, 8), dtype=np.int32)
    counts = np.zeros(7, dtype=np.int32)
    rc = lib().hy_plan_tick(
        q_lens.ctypes.data, kv_lens.ctypes.data, n, num_q_heads, num_kv_heads,
        page_size, num_cus, tokens_per_split, dec.ctypes.data, dec_cap,
        mrg.ctypes.data, n + 1, pre.ctypes.data, pre_cap, pmrg.ctypes.data, n_tiles + 1,
        counts.ctypes.data,
    )
    check(rc, "hy_plan_tick")
    nd, nm, ns, npf, npm, nps, npc = (int(x) for x in counts)
    return TickPlan(dec[: nd + npc].copy(), nd, mrg[:nm].copy(), ns, pre[:npf].copy(),
                    pmrg[:npm].copy(), nps)


def decode_workspace_bytes(n_slots: int, num_q_heads: int, head_dim: int) -> int:
    return int(lib().hy_decode_workspace_bytes(n_slots, num_q_heads, head_dim))


def prefill_workspace_bytes(n_slots: int, num_kv_heads: int, head_dim: int) -> int:
    return int(lib().hy_prefill_workspace_bytes(n_slots, num_kv_heads, head_dim))
