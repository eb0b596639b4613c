"""dk2 / dv2 pass at the edges of its steps and walks: short windows at and
around the 8- and 16-key steps (two or four units per 32-row step), groups that
leave the last step partly filled, key blocks of 256 and 128 with a remainder,
row groups past the first, and sequences that end inside a key block.  Checked
with all five gradients against the portable kernels and for repeatability.

Same rounding points, another order of the fp32 sums: in bf16 the forward's O and
a few P and dS round the other way (2^-8 of a term), and the results once more, so
that a gradient moves by about 2e-3 of its norm and at most some 2^-7 of its
largest value; a dropped unit, row group or piece of one of these shapes is a
percent or more.  fp32: hi/lo terms, 2^-16."""

import pytest
import torch

from helpers import assert_grads_close, rand_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,hq,hk,d,ws,wl,dtype", [
    (300, 2, 2, 128, 16, 40, "bf16"),    # two units per step, one head: query pairs
    (259, 3, 1, 128, 9, 300, "bf16"),    # ... three heads: steps straddle queries, odd unit count
    (131, 6, 3, 64, 8, 20, "bf16"),      # four units: pairs of heads of two queries
    (97, 8, 2, 128, 1, 1, "bf16"),       # one pair per query
    (70, 5, 1, 64, 7, 33, "bf16"),       # 8 keys or fewer, odd group: two units
    (513, 1, 1, 128, 17, 64, "bf16"),    # one unit per step again, a key past two blocks
    (140, 4, 2, 256, 16, 50, "bf16"),    # width 256
    (200, 4, 1, 256, 64, 100, "bf16"),   # ... two row groups in one walk
    (150, 2, 1, 64, 128, 140, "bf16"),   # four row groups
    (257, 6, 2, 128, 8, 30, "f32"),
    (129, 3, 3, 64, 16, 129, "f32"),     # width 64: 128-key blocks where they all run at once
    (200, 4, 2, 64, 32, 70, "f32"),
    (131, 4, 2, 64, 8, 40, "f32"),
    (257, 129, 129, 64, 32, 40, "f32"),  # ... 256-key blocks past that
    # bf16 as well: the shapes above take 128-key blocks, grids that fill the CUs 256-key ones
    (257, 100, 100, 128, 16, 40, "bf16"),
    (257, 200, 100, 64, 8, 40, "bf16"),
    (259, 100, 100, 128, 32, 300, "bf16"),
    (300, 128, 128, 64, 100, 120, "bf16"),
    (513, 80, 80, 128, 40, 60, "bf16"),
])
def test_dkv2_step_edges(cuda, n, hq, hk, d, ws, wl, dtype):
    from archlab_amd import simplicial_varlen_attention
    dt = torch.bfloat16 if dtype == "bf16" else torch.float32
    x = [t[0].to(cuda) for t in rand_inputs(1, n, hq, hk, d, seed=n + ws, dtype=dt)]
    cu = torch.tensor([0, 1, n // 3, n // 3 + 5, n], dtype=torch.int32, device=cuda)
    dout = torch.randn(n, hq, d, generator=torch.Generator().manual_seed(n)).to(dt).to(cuda)
    runs = []
    for kernel in ("auto", "auto", "generic"):
        xd = [t.clone().requires_grad_(True) for t in x]
        simplicial_varlen_attention(*xd, cu, ws, wl, scale=1.0, kernel=kernel).backward(dout)
        runs.append([t.grad.float() for t in xd])
    assert all(torch.equal(a, a2) for a, a2 in zip(*runs[:2]))
    assert_grads_close(runs[0], runs[2], *((2e-2, 5e-3) if dtype == "bf16" else (1e-4, 1e-4)))


@pytest.mark.parametrize("hq,hk,d,dv,ws,dtype", [
    (2, 2, 128, 128, 16, "bf16"), (6, 3, 64, 64, 8, "bf16"), (4, 2, 128, 64, 32, "bf16"), (2, 1, 64, 64, 100, "bf16"),
    (3, 1, 256, 256, 64, "bf16"), (4, 1, 512, 256, 32, "bf16"), (4, 1, 512, 256, 5, "bf16"),
    (4, 2, 128, 128, 32, "f32"), (2, 1, 64, 64, 7, "f32")])
def test_short_rows_of_the_sequence_before(cuda, hq, hk, d, dv, ws, dtype):
    """k1 and v1 rows that stand before a sequence's first token, infinite here,
    bring nothing into its dk2 and dv2 (a key block starts at the boundary)."""
    from helpers import backward_grads
    dt = torch.bfloat16 if dtype == "bf16" else torch.float32
    lo, n = 256, 330
    x = [t[0] for t in rand_inputs(1, n, hq, hk, d, dv, seed=ws, dtype=dt, device=cuda)]
    dout = torch.randn(n, hq, dv, generator=torch.Generator().manual_seed(n)).to(dt).to(cuda)
    cu = torch.tensor([0, lo, n], dtype=torch.int32, device=cuda)
    want = backward_grads(x, dout, cu, ws, 300)
    q, k1, k2, v1, v2 = (t.clone() for t in x)
    k1[lo - 5:lo] = float("inf")
    v1[lo - 9:lo] = float("inf")
    got = backward_grads((q, k1, k2, v1, v2), dout, cu, ws, 300)
    for name, i in (("dk2", 2), ("dv2", 4)):
        assert torch.isfinite(want[i]).all() and torch.equal(got[i][lo:], want[i][lo:]), name


@pytest.mark.parametrize("hq,hk,d,dv,ws,dtype", [
    (2, 1, 128, 128, 16, "bf16"), (4, 1, 64, 64, 8, "bf16"), (2, 2, 128, 128, 32, "bf16"), (2, 1, 256, 256, 40, "bf16"),
    (4, 1, 512, 256, 32, "bf16"), (4, 2, 128, 128, 32, "f32"), (8, 2, 64, 64, 5, "f32")])
def test_queries_that_do_not_reach_a_wave(cuda, hq, hk, d, dv, ws, dtype):
    """Non-finite queries reach the 32-key groups that their long windows overlap,
    not the rest of a workgroup's keys: a sequence before (k1 infinite) and later
    tokens (q NaN) in the same key blocks."""
    from helpers import backward_grads
    dt = torch.bfloat16 if dtype == "bf16" else torch.float32
    lo, hi, n, wl = 96, 300, 420, 44
    x = [t[0] for t in rand_inputs(1, n, hq, hk, d, dv, seed=ws, dtype=dt, device=cuda)]
    dout = torch.randn(n, hq, dv, generator=torch.Generator().manual_seed(n)).to(dt).to(cuda)
    cu = torch.tensor([0, lo, n], dtype=torch.int32, device=cuda)
    want = backward_grads(x, dout, cu, ws, wl)
    q, k1, k2, v1, v2 = (t.clone() for t in x)
    k1[lo - 40:lo] = float("inf")
    q[hi:] = float("nan")
    got = backward_grads((q, k1, k2, v1, v2), dout, cu, ws, wl)
    end = (hi - wl + 1) // 32 * 32
    for name, i in (("dk2", 2), ("dv2", 4)):
        assert torch.isfinite(want[i]).all() and torch.equal(got[i][lo:end], want[i][lo:end]), name
