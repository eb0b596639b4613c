"""Phases of the dq / dk1 / dv1 pass (csrc/sa_bwd_walk.h), taken where its
partials pass the space there is: the blocks and keys of every phase on the
host, and on the GPU calls that need several against the portable kernels."""

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
  long bad = 0, runs = 0, most = 0;
  for (int U : {4, 8, 16})
    for (int R : {16, 32})
      for (int group : {1, 2, 3, 5, 8, 16, 24, 128})
        for (int tokens : {1, 31, 200, 1024, 2048, 5001})
          for (long long cap = 1; cap < 2000; cap += 1 + cap / 7)
            for (int least : {1, 129}) {
              const int reach = R - 1;
              if (!dq_phases_pay(tokens, group, U, reach, cap, least)) continue;
              const long long blocks = ((long long)tokens * group + U - 1) / U;
              long long phases = 0, next = 0, taken = 0;
              for (int j0 = 0; j0 < tokens; ++phases) {
                const DqPhase p = dq_phase(j0, tokens, group, U, reach, cap);
                // no block left out, no more than there is room for, forward
                if (p.j0 != j0 || p.j1 <= j0 || p.j1 > tokens || p.nb < 1 || p.nb > cap || p.b0 > next ||
                    p.b0 + p.nb > blocks) {
                  ++bad;
                  break;
                }
                for (int j = j0; j < p.j1; ++j) {  // the blocks whose partials key j sums
                  const int thi = j + reach < tokens - 1 ? j + reach : tokens - 1;
                  const long long blo = (long long)j * group / U, bhi = ((long long)thi * group + group - 1) / U;
                  if (blo < p.b0 || bhi >= p.b0 + p.nb) ++bad;
                }
                next = p.b0 + p.nb;
                taken += p.nb;
                j0 = p.j1;
              }
              if (next != blocks || 2 * taken > 3 * blocks || (phases > 1 && cap < least)) ++bad;
              if (phases > most) most = phases;
              ++runs;
            }
  printf("%ld runs, at most %ld phases, %ld wrong\n", runs, most, bad);
  return bad != 0 || most < 4;
}
"""


def test_phases_cover_every_block_and_key(tmp_path):
    src, exe = tmp_path / "phases.cpp", tmp_path / "phases"
    src.write_text(_PROGRAM)
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout


def _against_portable(cuda, n, hq, hk, d, dv, ws, wl, flags):
    import torch
    from archlab_amd import _native
    from helpers import assert_grads_close, backward_grads, rand_inputs
    x = [t[0] for t in rand_inputs(1, n, hq, hk, d, dv, seed=n + ws, device=cuda)]
    dout = torch.randn(n, hq, dv, generator=torch.Generator().manual_seed(n)).to(x[0].dtype).to(cuda)
    cu = torch.tensor([0, n // 3, n], dtype=torch.int32, device=cuda)
    scratch = []
    got = backward_grads(x, dout, cu, ws, wl, flags, scratch)
    again = backward_grads(x, dout, cu, ws, wl, flags)
    want = backward_grads(x, dout, cu, ws, wl, _native.SA_FLAG_FORCE_GENERIC)
    assert all(torch.equal(a, b) for a, b in zip(got, again))
    # the same rounding points in another order of the fp32 sums: some P and dS
    # round the other way (2^-8 of a term), and the results once more
    assert_grads_close(got, want, 2e-2, 5e-3)
    return scratch[0]


@pytest.mark.gpu
@pytest.mark.parametrize("hq,hk,d,ws,wl,phases", [
    (8, 1, 128, 16, 1000, True), (12, 1, 64, 13, 1000, True), (12, 1, 128, 1, 1000, True), (24, 2, 64, 16, 300, True),
    (64, 1, 64, 16, 1000, True), (3, 1, 128, 16, 1000, False), (16, 1, 128, 13, 200, False)])
def test_small_workspace(cuda, hq, hk, d, ws, wl, phases):
    """SA_FLAG_SEPARATE_DK1 at no more than 16 short keys leaves the space of the
    dk2 / dv2 pieces: phases where one of them takes more than half of the CUs,
    else one phase that fits, or the dk1 / dv1 pass."""
    import torch
    from archlab_amd import _native
    n, group = 1024, hq // hk
    room = _against_portable(cuda, n, hq, hk, d, d, ws, wl, _native.SA_FLAG_SEPARATE_DK1)
    queries = 16 // group if 16 % group == 0 else 1 if group % 16 == 0 else (14 + group) // group + 1
    cap = room // (hk * (15 + queries) * 2 * d * 4)
    cus = torch.cuda.get_device_properties(cuda).multi_processor_count
    assert phases == (cap < n * group // 16 and cap >= 4 * (-(-15 * group // 16) + 1) and cap * hk > cus // 2)


@pytest.mark.gpu
def test_wide_partials_past_their_limit(cuda):
    """Score width 512 past 2 GiB of partials: two phases."""
    n = 11100
    room = _against_portable(cuda, n, 8, 2, 512, 256, 20, 40, 0)
    assert room // (2 * 32 * 768 * 4) < n
