"""One query per sequence against explicit key windows, on the paged kernel.

The reference's contiguous decode entry points (``simplicial_decode_attention``,
``packed_simplicial_decode``, ``tilelang_decode``) take, per batch row, the
short-axis rows (k1, v1) [B, N1, HK, D] and the long-axis rows (k2, v2)
[B, N2, HK, D] that the single query attends to: every (j, k) pair of those
rows is valid.  This module expresses that as a paged call: the rows become
caches with a block size of one row, the query sits at position P, the long
rows occupy positions P-L+1 .. P and the short rows P-N1+1 .. P.  Where the
lengths are known on the host the rows are consecutive blocks of the caches and
the call carries no tables (SA_FLAG_CONSECUTIVE_ROWS); the bounded form maps
each position to its row in two block tables.  Nothing is copied: K and V stay
separate tensors and the cache's K-to-V stride is the distance between them.
"""

from __future__ import annotations

import torch

from .simplicial_paged import _paged_launch, _rows_launch


class _KVPair:
    """K and V rows [B, N, HK, D] described as one paged cache
    [2 (K, V), B * N blocks, block_size 1, HK, D] without a copy: the dim-0
    stride is the element distance from K's first element to V's (it may be
    negative), a block is one row."""

    def __init__(self, k, v, first=0):
        # ``first``: rows before it are left out of every batch element
        b, n, hk, d = k.shape
        es = k.element_size()

        def fits(k, v):
            return (v.stride() == k.stride() and k.stride(-1) == 1 and k.stride(1) > 0
                    and k.stride(0) % k.stride(1) == 0 and k.stride(0) // k.stride(1) >= n
                    and (v.data_ptr() - k.data_ptr()) % es == 0)
        if not fits(k, v):
            k, v = k.contiguous(), v.contiguous()
        # block of row (batch i, row r) = i * rows_per_batch + r (a sliced view
        # of a longer cache keeps its own row stride, no copy)
        self.rows_per_batch = k.stride(0) // k.stride(1) if b > 1 else n
        self._k, self._v = k, v  # keep both alive for the launch
        self.shape = (2, b * self.rows_per_batch - first, 1, hk, d)
        self._offset = first * k.stride(1) * es
        self.dtype = k.dtype
        self._strides = ((v.data_ptr() - k.data_ptr()) // es, k.stride(1), k.stride(1), k.stride(2), 1)

    def data_ptr(self):
        return self._k.data_ptr() + self._offset

    def stride(self, dim=None):
        return self._strides if dim is None else self._strides[dim]


def window_decode(q, k1, k2, v1, v2, scale, key_lower=0, kernel="auto"):
    """q [B, HQ, D]; k1/v1 [B, N1, HK, D]; k2/v2 [B, N2, HK, D].

    Returns the fp32 output [B, HQ, D] of one joint softmax over all pairs
    (j < N1, key_lower <= k < N2).  Requires N1 <= N2 - key_lower.
    """
    b, hq, d = q.shape
    n1, n2 = k1.shape[1], k2.shape[1]
    length = n2 - key_lower
    if not 1 <= n1 <= length:
        raise ValueError("the short axis must not be longer than the long axis")
    if q.stride(-1) != 1:
        q = q.contiguous()
    return _rows_launch(q, _KVPair(k1, v1), _KVPair(k2, v2, first=key_lower), n1, length, scale, kernel)


def window_decode_bounded(q, k1, k2, v1, v2, scale, lengths, max_short, kernel="auto"):
    """The bounded form: ``lengths`` is a device int32 tensor
    [long length, short length, start]; the query attends to every pair of
    the last min(short length, max_short, N1) short rows and the long rows
    [start, start + long length) (clipped to the cache).  Nothing is read
    back to the host: the block tables, the query position and per-token
    window limits are computed on the device, so the call can be captured
    into a graph.  Lengths below 1 act as 1.

    Layout: with P = max(long, short) - 1 the query sits at position P; long
    position p holds long row start + p - (P - long + 1), short position p
    holds short row N1 - 1 - (P - p); the windows N1 (short) and max(N2, N1)
    (long) are capped per token at (short, long).
    """
    b, hq, d = q.shape
    n1, n2 = k1.shape[1], k2.shape[1]
    dev = q.device
    long_cache = _KVPair(k2, v2)
    short_cache = _KVPair(k1, v1)
    lens = lengths.to(device=dev, dtype=torch.int64)
    start = lens[2].clamp(0, n2 - 1)
    long_len = torch.minimum(lens[0], n2 - start).clamp_min(1)
    short_len = lens[1].clamp(1, min(max_short, n1))
    top = torch.maximum(long_len, short_len) - 1  # query position P
    width = max(n2, n1)
    p = torch.arange(width, device=dev, dtype=torch.int64)
    rows = torch.arange(b, device=dev, dtype=torch.int64)[:, None]
    long_row = (start + p - (top - long_len + 1)).clamp(0, n2 - 1)
    short_row = (n1 - 1 - (top - p)).clamp(0, n1 - 1)
    long_table = (rows * long_cache.rows_per_batch + long_row[None, :]).to(torch.int32)
    short_table = (rows * short_cache.rows_per_batch + short_row[None, :]).to(torch.int32)
    token_seq = torch.arange(b, device=dev, dtype=torch.int32)
    token_pos = top.to(torch.int32).expand(b).contiguous()
    caps = torch.stack((short_len, long_len)).to(torch.int32)[None, :].expand(b, 2).contiguous()
    if q.stride(-1) != 1:
        q = q.contiguous()
    return _paged_launch(q, short_cache, long_cache, short_table, long_table, token_seq, token_pos,
                         n1, width, scale, None, False, kernel, window_caps=caps)
