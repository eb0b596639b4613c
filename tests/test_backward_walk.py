"""The dk2 / dv2 pass's walk over its units, as the kernel steps it
(csrc/sa_bwd_walk.h, compiled here for the host): the row that the staging
pointer holds is the unit's own within the walk, and never leaves the walk's
rows for the units that pad the last step."""

import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "next-gen-arch_amd", "csrc")

_PROGRAM = r"""
#include <cstdio>
#include <initializer_list>
#include "sa_bwd_walk.h"
using namespace sa;
int main() {
  long bad = 0, units = 0;
  for (int group = 1; group <= 14; ++group)
    for (int nr = 1; nr <= 4; ++nr)
      for (int pk : {1, 2, 4}) {
        if (pk > 1 && nr > 1) continue;  // several units per step: one row group
        for (int tfirst : {0, 3})
          for (int queries = 1; queries <= 9; ++queries) {
            const int tlast = tfirst + queries - 1, n = queries * group * nr;
            WalkUnit u{tfirst, 0, 0};
            int t = tfirst, h = 0;  // the staged row
            for (int i = 0; i < (n + pk - 1) / pk * pk; ++i, ++units) {
              const int wt = i < n ? tfirst + i / (nr * group) : tlast, wh = i < n ? i / nr % group : group - 1;
              if (i < n && (u.t != wt || u.h != wh || u.r != i % nr)) ++bad;
              if (t != wt || h != wh) {
                if (bad++ == 0)
                  printf("group %d nr %d pk %d queries %d unit %d: row (%d, %d)\n", group, nr, pk, queries, i, t, h);
              }
              const WalkUnit y = walk_next(u, group, nr);
              if (walk_moves(u, y, i, n, pk)) {
                if (y.t == u.t) ++h;
                else ++t, h = 0;
              }
              u = y;
            }
          }
      }
  printf("%ld units, %ld off\n", units, bad);
  return bad != 0;
}
"""


def test_staged_rows_stay_inside_the_walk(tmp_path):
    src, exe = tmp_path / "walk.cpp", tmp_path / "walk"
    src.write_text(_PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout


def _grads(x, dout, cu, ws, wl):
    """dq, dk1, dk2, dv1, dv2 of tensors of any layout through the C ABI."""
    import ctypes

    import torch
    from archlab_amd import _native
    from archlab_amd.architectures.simplicial_attention import _prefill
    lib, dev = _native.load(), x[0].device
    dense = [t.contiguous() for t in x]
    out, lse = _prefill(*dense, ws, wl, 0.3, cu, cu.numel() - 1, 0, True, "auto")
    grads = [torch.empty_like(t) for t in dense]
    q, k1, k2, v1, v2 = x
    dq, dk1, dk2, dv1, dv2 = grads
    fwd = _native.PrefillArgs(
        q=q.data_ptr(), k1=k1.data_ptr(), k2=k2.data_ptr(), v1=v1.data_ptr(), v2=v2.data_ptr(), out=out.data_ptr(),
        lse=lse.data_ptr(), cu_seqlens=cu.data_ptr(), q_stride_t=q.stride(0), q_stride_h=q.stride(1),
        k_stride_t=k1.stride(0), k_stride_h=k1.stride(1), v_stride_t=v1.stride(0), v_stride_h=v1.stride(1),
        o_stride_t=out.stride(0), o_stride_h=out.stride(1), lse_stride_t=lse.stride(0), num_seqs=cu.numel() - 1,
        total_tokens=q.shape[0], heads_q=q.shape[1], heads_kv=k1.shape[1], head_dim=q.shape[2],
        value_dim=v1.shape[2], short_window=ws, long_window=wl, scale=0.3, dtype=_native.dtype_code(q.dtype))
    args = _native.PrefillBwdArgs(
        fwd=fwd, dout=dout.data_ptr(), do_stride_t=dout.stride(0), do_stride_h=dout.stride(1), dq=dq.data_ptr(),
        dq_stride_t=dq.stride(0), dq_stride_h=dq.stride(1), dk1=dk1.data_ptr(), dk2=dk2.data_ptr(),
        dk_stride_t=dk1.stride(0), dk_stride_h=dk1.stride(1), dv1=dv1.data_ptr(), dv2=dv2.data_ptr(),
        dv_stride_t=dv1.stride(0), dv_stride_h=dv1.stride(1))
    nbytes = lib.sa_prefill_bwd_workspace_bytes(ctypes.byref(args))
    work = torch.empty(nbytes + 256, device=dev, dtype=torch.uint8)
    _native.check(lib.sa_prefill_bwd(ctypes.byref(args), (work.data_ptr() + 255) & ~255, nbytes,
                                     _native.stream_handle(dev)))
    torch.cuda.synchronize()
    return grads


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("layout", ["token", "head"])
@pytest.mark.parametrize("n,hq,hk,ws", [(131, 6, 3, 8), (33, 2, 1, 1), (5, 6, 1, 7), (259, 12, 2, 8), (33, 2, 1, 16)])
def test_rows_past_the_tensors_are_not_used(cuda, n, hq, hk, ws, layout, dtype):
    """Every tensor is the front of a larger one whose rest is NaN, with the
    heads of a token or the tokens of a head adjacent: the gradients are
    those of separate tensors, bit for bit."""
    import torch
    from helpers import rand_inputs
    dt = torch.bfloat16 if dtype == "bf16" else torch.float32
    x = [t[0] for t in rand_inputs(1, n, hq, hk, 64, seed=n, dtype=dt, device=cuda)]
    x.append(torch.randn(n, hq, 64, generator=torch.Generator().manual_seed(n)).to(dt).to(cuda))  # dout
    cu = torch.tensor([0, n // 3, n], dtype=torch.int32, device=cuda)

    def front(t):
        if layout == "token":
            big = torch.full((n + 2, t.shape[1], 64), float("nan"), dtype=dt, device=cuda)
            view = big[:n]
        else:
            big = torch.full((t.shape[1] + 2, n, 64), float("nan"), dtype=dt, device=cuda)
            view = big[:t.shape[1]].transpose(0, 1)
        view.copy_(t)
        return view

    want = _grads(x[:5], x[5], cu, ws, 20)
    y = [front(t) for t in x]
    got = _grads(y[:5], y[5], cu, ws, 20)
    for name, a, b in zip(("dq", "dk1", "dk2", "dv1", "dv2"), got, want):
        assert torch.isfinite(b).all() and torch.equal(a, b), name
