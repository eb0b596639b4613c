"""The fp32 paged kernel (fp32 query, caches not both bf16) at the edges of its
tasks (1, 16, 17 and 32 short keys, odd groups), chunks and splits, against the
fp64 oracle; and the table-free row form against the same call with tables.

Tolerance: a score sums D products of fp32 values, each rounded to 2^-24; with
|q k1 k2| summing to at most ~16 here its error is below D/2 2^-24 16 < 1.3e-4 in
the worst order, ~1e-6 typically, and P carries it as a relative error.  Outputs
are averages of v1 v2 below ~10: 2e-5 is 20 typical errors and below the bound.
"""

import ctypes

import pytest
import torch

from helpers import assert_lse_close, assert_out_close, paged_batch
from oracle import simplicial_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,heads,kv_heads,ws,wl,short_t,long_t", [
    (64, 6, 2, 16, 33, torch.float32, torch.float32),
    (64, 8, 1, 17, 64, torch.float32, torch.float16),
    (128, 8, 2, 1, 31, torch.float32, torch.float32),
    (128, 5, 1, 33, 100, torch.bfloat16, torch.float32),
    (128, 2, 2, 32, 1000, torch.float16, torch.float16),
    (256, 3, 1, 16, 65, torch.float32, torch.bfloat16),
    (256, 4, 2, 40, 97, torch.float32, torch.float32),
])
def test_matches_oracle_at_tile_edges(cuda, dim, heads, kv_heads, ws, wl, short_t, long_t):
    from archlab_amd.architectures.simplicial_paged import paged_plan, simplicial_paged_attention
    lengths = [1, 16, 34, 150]
    (short, long), table, dense = paged_batch(lengths, kv_heads, dim, 16, torch.bfloat16, seed=3, device=cuda)
    short, long = short.to(short_t), long.to(long_t)
    g = torch.Generator().manual_seed(4)
    q = torch.randn(len(lengths), 1, heads, dim, generator=g) * dim ** -0.5
    seq = torch.arange(len(lengths), dtype=torch.int32, device=cuda)
    pos = torch.tensor(lengths, dtype=torch.int32, device=cuda) - 1
    expect, lse_ref = [], []
    for i, (n, (k1, k2, v1, v2)) in enumerate(zip(lengths, dense)):
        qs = torch.zeros(1, n, heads, dim)
        qs[0, -1] = q[i, 0]
        o, l = O.reference_simplicial(*(x.double() for x in (qs, k1, k2, v1, v2)), ws, wl, scale=1.0,
                                      return_lse=True)
        expect.append(o[0, -1])
        lse_ref.append(l[0, -1])
    args = (q[:, 0].to(cuda), short, long, table, seq, pos)
    kw = dict(short_window=ws, long_window=wl, scale=1.0)
    assert paged_plan(*args, **kw)[0] == "generic"
    for splits in (None, 1, 2, 7):
        out, lse = simplicial_paged_attention(*args, **kw, splits=splits, return_lse=True)
        assert_out_close(out, torch.stack(expect), torch.float32, atol=2e-5)
        assert_lse_close(lse, torch.stack(lse_ref), torch.float32, rtol=2e-5)


def test_runs_without_a_workspace(cuda):
    """A caller that brings no workspace (none was needed on the portable kernel) is served."""
    from archlab_amd import _native
    from archlab_amd.architectures.simplicial_paged import _paged_args, simplicial_paged_attention
    lib, stream = _native.load(), _native.stream_handle(cuda)
    (short, long), table, _ = paged_batch([300, 90], 2, 128, 16, torch.float32, seed=5, device=cuda)
    q = torch.randn(2, 8, 128, device=cuda, generator=torch.Generator(cuda).manual_seed(6)) / 128 ** 0.5
    seq = torch.arange(2, dtype=torch.int32, device=cuda)
    pos = torch.tensor([299, 89], dtype=torch.int32, device=cuda)
    for ws in (16, 40):
        want = simplicial_paged_attention(q, short, long, table, seq, pos, short_window=ws, long_window=256, scale=1.0)
        for entry in ("ws", "noalloc"):
            out = torch.full_like(q, float("nan"))
            args = _paged_args(q, short, long, table, table, seq, pos, ws, 256, 1.0, None, out, None, 0)
            if entry == "ws":
                _native.check(lib.sa_paged_fwd(ctypes.byref(args), None, 0, stream))
            else:
                _native.check(lib.sa_paged_fwd_noalloc(ctypes.byref(args), stream))
            torch.testing.assert_close(out, want, rtol=2e-5, atol=2e-5)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("kernel", ["auto", "generic"])
@pytest.mark.parametrize("dim,n1,n2,lower", [(64, 1, 40, 0), (128, 16, 130, 5), (128, 33, 1000, 0), (64, 20, 20, 0)])
def test_rows_without_tables_match_tables(cuda, dtype, kernel, dim, n1, n2, lower):
    """Consecutive rows read the same rows as a call with explicit tables: bit-equal."""
    from archlab_amd.architectures.simplicial_paged import _paged_launch
    from archlab_amd.architectures.window_decode import _KVPair, window_decode
    b, hq, hk = 3, 4, 2
    g = torch.Generator().manual_seed(7)
    q = (torch.randn(b, hq, dim, generator=g) / dim ** 0.5).to(dtype).to(cuda)
    k1, v1 = (torch.randn(b, n1 + 3, hk, dim, generator=g).to(dtype).to(cuda)[:, 3:] for _ in range(2))
    k2, v2 = (torch.randn(b, n2, hk, dim, generator=g).to(dtype).to(cuda) for _ in range(2))
    out = window_decode(q, k1, k2, v1, v2, 1.0, key_lower=lower, kernel=kernel)
    long, short, n = _KVPair(k2, v2), _KVPair(k1, v1), n2 - lower
    p, rows = torch.arange(n, device=cuda), torch.arange(b, device=cuda)[:, None]
    table2 = (rows * long.rows_per_batch + lower + p).to(torch.int32)
    table1 = (rows * short.rows_per_batch + (p - (n - n1)).clamp_min(0)).to(torch.int32)
    want = _paged_launch(q, short, long, table1, table2, torch.arange(b, device=cuda, dtype=torch.int32),
                         torch.full((b,), n - 1, device=cuda, dtype=torch.int32), n1, n, 1.0, None, False, kernel)
    assert torch.equal(out, want)


@pytest.mark.parametrize("ws,wl", [(16, 200), (16, 40), (32, 200)])
def test_scores_of_minus_infinity(cuda, ws, wl):
    """A short key whose scores overflow to -inf over the first chunks of the
    window, and one over all of it, weigh nothing there, as on the portable
    kernel (whose running maximum is one for all rows); the other rows, and the
    first one's later keys, decide the output."""
    from archlab_amd.architectures.simplicial_paged import simplicial_paged_attention
    n, hk, hq, dim = 230, 2, 4, 64
    (short, long), table, _ = paged_batch([n], hk, dim, n + 2, torch.float32, seed=9, device=cuda)
    block = table[0, 0].item()
    q = torch.ones(1, hq, dim, device=cuda) / dim
    seq, pos = torch.zeros(1, dtype=torch.int32, device=cuda), torch.full((1,), n - 1, dtype=torch.int32, device=cuda)
    short[0, block, :n] = 1.0
    short[0, block, n - 3] = 1e30    # -inf over keys of -1e30, 0 over keys of 0
    short[0, block, n - 5] = 3e38    # -inf over every negative key
    long[0, block, :n - 20] = -1e30
    long[0, block, n - 20:n] = -2.0
    long[0, block, n - 10] = 0.0
    kw = dict(short_window=ws, long_window=wl, scale=1.0, return_lse=True)
    for splits in (None, 1, 2):
        out, lse = simplicial_paged_attention(q, short, long, table, seq, pos, splits=splits, **kw)
        want, lse_ref = simplicial_paged_attention(q, short, long, table, seq, pos, kernel="generic", **kw)
        assert torch.isfinite(want).all() and torch.isfinite(lse_ref).all()
        torch.testing.assert_close(out, want, rtol=2e-5, atol=2e-5)
        torch.testing.assert_close(lse, lse_ref, rtol=2e-5, atol=2e-5)
