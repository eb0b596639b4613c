"""dq / dk1 / dv1 pass at the edges of its workgroups: groups that divide a
workgroup's units, are divided by them or neither, last units past the tokens,
short windows at the 16-key units, and sequences that end inside a workgroup.
All five gradients against the portable kernels and for repeatability (same
rounding points, another order of the fp32 sums: some terms and the results round
the other way, about 2e-3 of a gradient's norm and at most some 2^-7 of its
largest value)."""

import pytest
import torch

from helpers import assert_grads_close, rand_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,hq,hk,d,dv,ws,wl", [
    (131, 4, 1, 512, 256, 32, 40),
    (67, 3, 1, 512, 256, 17, 300),
    (90, 2, 2, 512, 256, 16, 33),
    (53, 8, 1, 512, 256, 1, 7),
    (131, 16, 4, 128, 128, 16, 40),
    (67, 3, 1, 128, 128, 7, 300),
    (90, 2, 2, 128, 128, 16, 33),
    (53, 24, 1, 128, 128, 1, 7),
    (131, 4, 4, 64, 64, 16, 70),
    (75, 12, 2, 64, 64, 13, 90),
])
def test_dq_block_edges(cuda, n, hq, hk, d, dv, ws, wl):
    from archlab_amd import simplicial_varlen_attention
    x = [t[0].to(cuda) for t in rand_inputs(1, n, hq, hk, d, dv, seed=n + ws)]
    cu = torch.tensor([0, 1, n // 3, n // 3 + 5, n], dtype=torch.int32, device=cuda)
    dout = torch.randn(n, hq, dv, generator=torch.Generator().manual_seed(n)).to(x[0].dtype).to(cuda)
    runs = []
    for kernel in ("auto", "auto", "generic"):
        xd = [t.clone().requires_grad_(True) for t in x]
        simplicial_varlen_attention(*xd, cu, ws, wl, scale=1.0, kernel=kernel).backward(dout)
        runs.append([t.grad.float() for t in xd])
    assert all(torch.equal(a, a2) for a, a2 in zip(*runs[:2]))
    assert_grads_close(runs[0], runs[2], 2e-2, 5e-3)


@pytest.mark.parametrize("hq,hk,d,dv,ws", [(4, 1, 512, 256, 32), (8, 1, 512, 256, 16), (16, 1, 128, 128, 16),
                                           (32, 2, 64, 64, 9)])
def test_values_that_no_query_of_the_block_sees(cuda, hq, hk, d, dv, ws):
    """Short rows of the sequence before (k1, v1 infinite) and keys of later
    tokens (k2 NaN): the other queries' gradients are those of finite tensors,
    bit for bit.  One query per workgroup here; dk1 / dv1 also gather the 31
    queries after a key."""
    from helpers import backward_grads
    n, lo, hi = 140, 40, 120
    x = [t[0] for t in rand_inputs(1, n, hq, hk, d, dv, seed=ws, device=cuda)]
    dout = torch.randn(n, hq, dv, generator=torch.Generator().manual_seed(n)).to(x[0].dtype).to(cuda)
    cu = torch.tensor([0, lo, n], dtype=torch.int32, device=cuda)
    want = backward_grads(x, dout, cu, ws, 300)
    q, k1, k2, v1, v2 = (t.clone() for t in x)
    k1[lo - 10:lo] = float("inf")
    v1[lo - 10:lo] = float("inf")
    k2[hi:] = float("nan")
    got = backward_grads((q, k1, k2, v1, v2), dout, cu, ws, 300)
    for name, i, end in (("dq", 0, hi), ("dk1", 1, hi - 31), ("dv1", 3, hi - 31)):
        assert torch.isfinite(want[i]).all() and torch.equal(got[i][lo:end], want[i][lo:end]), name
