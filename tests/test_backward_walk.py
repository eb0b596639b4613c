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
  // pointer steps: head-major strides of large tensors pass 32 bits
  for (long long tokens : {1000LL, 1LL << 20, 1LL << 24})
    for (int group : {1, 2, 64, 128})
      for (long long row : {8LL, 32LL})  // 16-byte units of a row
        for (int major : {0, 1, -1}) {
          const long long st_t = major ? row : group * row, st_h = major ? major * tokens * row : row;
          const long long q = st_t - (group - 1) * st_h;
          const bool fit = (int)st_h == st_h && (int)q == q;
          if (walk_steps_fit(st_t, st_h, group) != fit || walk_query_step(st_t, st_h, group) != q) ++bad;
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


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("layout", ["token", "head"])
@pytest.mark.parametrize("n,hq,hk,ws", [(131, 6, 3, 8), (33, 2, 1, 1), (5, 6, 1, 7), (259, 12, 2, 8), (33, 2, 1, 16)])
def test_rows_past_the_tensors_are_not_used(cuda, n, hq, hk, ws, layout, dtype):
    """Every tensor is the front of a larger one whose rest is NaN, with the
    heads of a token or the tokens of a head adjacent: the gradients are
    those of separate tensors, bit for bit."""
    import torch
    from helpers import backward_grads, rand_inputs
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

    want = backward_grads(x[:5], x[5], cu, ws, 20)
    y = [front(t) for t in x]
    got = backward_grads(y[:5], y[5], cu, ws, 20)
    for name, a, b in zip(("dq", "dk1", "dk2", "dv1", "dv2"), got, want):
        assert torch.isfinite(b).all() and torch.equal(a, b), name
