"""Cumulative left-ordered Hamilton product along the sequence axis.

Mirrors parallel_scan_quaternion, mambaqc/kernels/parallel_scan.py:171-264,
with the semantics of its sequential reference (:267-295):
    cumulative[:, t] = q[:, t] (x) q[:, t-1] (x) ... (x) q[:, 0]
The HIP kernel scans the true time axis for every (b, d, k) lane; it does not
reproduce the reference GPU path's reshape of a [B,T,D,S,4] tensor to
[B*D, T, S, 4], which mixes the time and d_model axes whenever D > 1.
"""
from __future__ import annotations

import torch

from .. import _native as nat


# The time-chunked product (mqc_cumprod_scan_chunked) reads q twice, so it pays where the whole
# walk is bound by its serial chain (us, whole / chunked): fp32 T 4096 1024 lanes 182 / 55, 4096
# 188 / 146, but 8192 263 / 318; bf16 1024 433 / 44, 24576 (T 2000) 379 / 218, 16000 (T 256)
# 30 / 25, 49152 (T 2000) 463 / 430. Short sequences leave little to save, the more the fewer the
# lanes (with the Cayley map that wrote q, bf16): T 128 1024 lanes 18.5 / 22.5, 2048 20 / 22.6, 6144
# 27 / 22, 24576 36 / 31; T 160 256 lanes 23.3 / 22.8, 2048 26 / 23; T 234 16384 lanes 56 / 37.
CHUNK_MAX_LANES = {4: 4096, 2: 24576}   # batch x lanes, by element size
CHUNK_MIN_SEQ = {4: 512, 2: 128}
CHUNK_FEW_LANES = 4096                  # below this many:
CHUNK_FEW_MIN_SEQ = {4: 512, 2: 160}


def _chunk_len(B: int, T: int, lanes: int, el: int) -> int:
    """Steps per chunk, 0 for the whole walk."""
    if B < 1 or lanes < 1 or B * lanes > CHUNK_MAX_LANES[el]:
        return 0
    if T < (CHUNK_FEW_MIN_SEQ if B * lanes < CHUNK_FEW_LANES else CHUNK_MIN_SEQ)[el]:
        return 0
    L = nat.q_chunk_len(B, T, lanes, el)
    return L if L < T and B * -(-T // L) <= 65535 else 0


def parallel_scan_quaternion(q_sequence: torch.Tensor) -> torch.Tensor:
    """q_sequence: [batch, seq_len, d_model, d_state, 4] -> cumulative products (new tensor)."""
    assert q_sequence.shape[-1] == 4
    assert q_sequence.ndim == 5
    nat.require_device("parallel_scan_quaternion", q_sequence)
    code = nat.dtype_code(q_sequence)
    q = nat.aligned16(q_sequence)
    B, T, D, S, _ = q.shape
    out = torch.empty_like(q)
    L = _chunk_len(B, T, D * S, q.element_size())
    if L:
        nbytes = int(nat.load().mqc_q_chunked_workspace_bytes(B, T, D * S, L, 0))
        ws = torch.empty(nbytes, device=q.device, dtype=torch.uint8)
        nat.call("mqc_cumprod_scan_chunked", q, q.data_ptr(), out.data_ptr(), B, T, D * S, L,
                 code, ws.data_ptr(), nbytes, nat.stream_of(q))
        return out
    nat.call("mqc_cumprod_scan_fwd", q, q.data_ptr(), out.data_ptr(), B, T, D * S,
             code, nat.stream_of(q))
    return out
