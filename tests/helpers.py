"""Shared builders and tolerance checks for the parity tests."""

from __future__ import annotations

import math

import torch

# Tolerances stated by the benchmark contract: bf16 output max-abs <= 2e-2,
# LSE relative <= 1e-3; fp32 <= 1e-4.
#  - The LSE "relative" error is taken against max(|lse|, 1): the LSE is a log,
#    an absolute error e in it is a relative error ~e in the partition sum,
#    and |lse| -> 0 (one or two pairs) would make a pure ratio meaningless.
#  - bf16 outputs additionally get half a bf16 ulp of the reference value
#    (2^-8 |ref|): a bf16 result cannot be closer than its own rounding, which
#    matters only where |O| > 1 (windows of one or two pairs).
BF16_OUT_ATOL = 2e-2
BF16_OUT_RTOL = 2.0 ** -8
BF16_LSE_RTOL = 1e-3
FP32_TOL = 1e-4


def rand_inputs(b, n, hq, hk, d, dv=None, seed=0, dtype=torch.bfloat16, sigma=1.0, device="cpu"):
    """(q, k1, k2, v1, v2): fp32 N(0, sigma^2) draws, q scaled by 1/sqrt(d), cast to dtype."""
    dv = d if dv is None else dv
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(b, n, hq, d, generator=g) * sigma / math.sqrt(d)
    k1, k2 = (torch.randn(b, n, hk, d, generator=g) * sigma for _ in range(2))
    v1, v2 = (torch.randn(b, n, hk, dv, generator=g) * sigma for _ in range(2))
    return [x.to(dtype).to(device) for x in (q, k1, k2, v1, v2)]


def assert_out_close(actual, expected, dtype, atol=None, rtol=None):
    """max |a - e| - rtol*|e| <= atol; returns the plain max-abs error."""
    actual = actual.float().cpu()
    expected = expected.float().cpu()
    assert torch.isfinite(actual).all(), "non-finite output"
    if atol is None:
        atol = BF16_OUT_ATOL if dtype == torch.bfloat16 else FP32_TOL
    if rtol is None:
        rtol = BF16_OUT_RTOL if dtype == torch.bfloat16 else 0.0
    diff = (actual - expected).abs()
    excess = (diff - rtol * expected.abs()).max().item()
    err = diff.max().item()
    where = divmod(int(diff.argmax()), expected.shape[-1]) if expected.ndim else 0
    assert excess <= atol, f"max-abs error {err:.3e} (excess {excess:.3e} > {atol:.1e}) at {where}"
    return err


def assert_lse_close(actual, expected, dtype, rtol=None):
    """max |a - e| / max(|e|, 1) <= rtol; returns that relative error."""
    actual = actual.float().cpu()
    expected = expected.float().cpu()
    assert torch.isfinite(actual).all(), "non-finite lse"
    if rtol is None:
        rtol = BF16_LSE_RTOL if dtype == torch.bfloat16 else FP32_TOL
    rel = ((actual - expected).abs() / expected.abs().clamp_min(1.0)).max().item()
    assert rel <= rtol, f"lse relative error {rel:.3e} > {rtol:.1e}"
    return rel


def assert_grads_close(actual, expected, rel_max, rel_norm):
    """dq, dk1, dk2, dv1, dv2 each within rel_max of its own largest value and
    rel_norm of its norm (no absolute floor: dk1 and dk2 are small)."""
    for name, a, e in zip(("dq", "dk1", "dk2", "dv1", "dv2"), actual, expected):
        a, e = a.float(), e.float()
        assert torch.isfinite(a).all(), f"{name}: non-finite"
        diff, norm = (a - e).abs().max().item(), (a - e).norm().item()
        print(f"{name}: max {diff / max(e.abs().max().item(), 1e-30):.1e}, "
              f"norm {norm / max(e.norm().item(), 1e-30):.1e}", flush=True)
        assert diff <= rel_max * e.abs().max().item(), f"{name}: {diff:.2e}"
        assert norm <= rel_norm * e.norm().item(), f"{name}: {norm:.2e} of {e.norm().item():.2e}"


def paged_batch(lengths, kv_heads, dim, block_size, dtype, hnd=False, seed=0, device="cuda"):
    """Contiguous per-sequence K/V plus the same rows scattered into shuffled pages.

    Block 0 is the null block.  Returns ([short, long] caches, int32 table,
    list of per-sequence (k1, k2, v1, v2) [1, n, HK, D]).
    """
    g = torch.Generator().manual_seed(seed)
    per = [math.ceil(n / block_size) for n in lengths]
    total = 1 + sum(per)
    perm = (torch.randperm(total - 1, generator=g) + 1).tolist()
    table = torch.zeros(len(lengths), max(per), dtype=torch.int32)
    shape = (2, total, kv_heads, block_size, dim) if hnd else (2, total, block_size, kv_heads, dim)
    caches = [torch.zeros(shape, dtype=dtype) for _ in range(2)]
    dense = []
    for s, n in enumerate(lengths):
        table[s, :per[s]] = torch.tensor(perm[:per[s]], dtype=torch.int32)
        perm = perm[per[s]:]
        k1, k2, v1, v2 = (torch.randn(1, n, kv_heads, dim, generator=g).to(dtype) for _ in range(4))
        dense.append((k1, k2, v1, v2))
        idx = torch.arange(n)
        blocks = table[s].long()[idx // block_size]
        offs = idx % block_size
        for cache, (k, v) in zip(caches, ((k1, v1), (k2, v2))):
            view = cache.transpose(2, 3) if hnd else cache
            view[0, blocks, offs] = k[0]
            view[1, blocks, offs] = v[0]
    if hnd:
        caches = [c.transpose(2, 3) for c in caches]
    return [c.to(device) for c in caches], table.to(device), dense


def backward_grads(x, dout, cu, ws, wl, flags=0, scratch=None):
    """dq, dk1, dk2, dv1, dv2 of [T, H, *] tensors of any layout through the C ABI.
    ``scratch`` (a list): receives the workspace bytes past the delta and dlse rows."""
    import ctypes

    from archlab_amd import _native
    from archlab_amd.architectures.simplicial_attention import _prefill
    lib, dev = _native.load(), x[0].device
    dense = [t.contiguous() for t in x]
    out, lse = _prefill(*dense, ws, wl, 0.3, cu, cu.numel() - 1, 0, True, 
                        "generic" if flags & _native.SA_FLAG_FORCE_GENERIC else "auto")
    grads = [torch.empty_like(t) for t in dense]
    q, k1, k2, v1, v2 = x
    dq, dk1, dk2, dv1, dv2 = grads
    fwd = _native.PrefillArgs(
        q=q.data_ptr(), k1=k1.data_ptr(), k2=k2.data_ptr(), v1=v1.data_ptr(), v2=v2.data_ptr(), out=out.data_ptr(),
        lse=lse.data_ptr(), cu_seqlens=cu.data_ptr(), q_stride_t=q.stride(0), q_stride_h=q.stride(1),
        k_stride_t=k1.stride(0), k_stride_h=k1.stride(1), v_stride_t=v1.stride(0), v_stride_h=v1.stride(1),
        o_stride_t=out.stride(0), o_stride_h=out.stride(1), lse_stride_t=lse.stride(0), num_seqs=cu.numel() - 1,
        total_tokens=q.shape[0], heads_q=q.shape[1], heads_kv=k1.shape[1], head_dim=q.shape[2],
        value_dim=v1.shape[2], short_window=ws, long_window=wl, scale=0.3, dtype=_native.dtype_code(q.dtype),
        flags=flags)
    args = _native.PrefillBwdArgs(
        fwd=fwd, dout=dout.data_ptr(), do_stride_t=dout.stride(0), do_stride_h=dout.stride(1), dq=dq.data_ptr(),
        dq_stride_t=dq.stride(0), dq_stride_h=dq.stride(1), dk1=dk1.data_ptr(), dk2=dk2.data_ptr(),
        dk_stride_t=dk1.stride(0), dk_stride_h=dk1.stride(1), dv1=dv1.data_ptr(), dv2=dv2.data_ptr(),
        dv_stride_t=dv1.stride(0), dv_stride_h=dv1.stride(1))
    nbytes = lib.sa_prefill_bwd_workspace_bytes(ctypes.byref(args))
    if scratch is not None:
        scratch.append(nbytes - 2 * ((q.shape[0] * q.shape[1] * 4 + 255) // 256 * 256))
    work = torch.empty(nbytes + 256, device=dev, dtype=torch.uint8)
    _native.check(lib.sa_prefill_bwd(ctypes.byref(args), (work.data_ptr() + 255) & ~255, nbytes,
                                     _native.stream_handle(dev)))
    torch.cuda.synchronize()
    return grads
