// Index walks of the backward passes, constexpr so that the kernels, their
// launches and host checks run the same steps.
#pragma once

namespace sa {

// dk2 / dv2 pass: units in ascending (query t, head h of the KV group, 32-row
// group r of t's short keys).
struct WalkUnit {
  int t, h, r;  // h: head within the group
};

constexpr WalkUnit walk_next(WalkUnit u, int group, int nr) {
  if (++u.r == nr) {
    u.r = 0;
    if (++u.h == group) u.h = 0, ++u.t;
  }
  return u;
}

// Whether the staged rows change after unit u, unit i of the walk's n, with the
// successor y: to the next head's (same t) or the next query's first head's.
// Row groups of a head share its rows, and units past the walk, which pad the
// last step of pk units, keep its last unit's: no row outside the walk is read.
// (One unit per step: nothing is staged after the last.)
constexpr bool walk_moves(WalkUnit u, WalkUnit y, int i, int n, int pk) {
  return (y.h != u.h || y.t != u.t) && (pk == 1 || i + 1 < n);
}


// Pointer steps between staged rows, in 16-byte units (strides in the same): the
// next head's row, and from the last head of a query to the first of the next.
// The kernel holds them in 32 bits.
constexpr long long walk_query_step(long long stride_t, long long stride_h, int group) {
  return stride_t - (group - 1) * stride_h;
}
constexpr bool walk_steps_fit(long long stride_t, long long stride_h, int group) {
  const long long q = walk_query_step(stride_t, stride_h, group), lim = 0x7fffffffLL;
  return stride_h >= -lim && stride_h <= lim && q >= -lim && q <= lim;
}

// dq / dk1 / dv1 pass: blocks of U consecutive units (t, h), whose partials may
// take more space than there is (room for `cap` blocks).  It then runs in
// phases, blocks [b0, b0 + nb) each, followed by the sums of the keys [j0, j1)
// that the phase completes: a key waits for the queries up to `reach` after its
// own, so the next phase starts with the blocks of the last `reach` queries.
struct DqPhase {
  int b0, nb, j0, j1;
};

constexpr DqPhase dq_phase(int j0, int tokens, int group, int U, int reach, long long cap) {
  const long long blocks = ((long long)tokens * group + U - 1) / U;
  const long long b0 = (long long)j0 * group / U;
  const long long nb = cap < blocks - b0 ? cap : blocks - b0;
  const int tend = (int)((b0 + nb) * U / group);  // queries before it are complete
  return {(int)b0, (int)nb, j0, b0 + nb == blocks ? tokens : tend - reach};
}

// Whether the pass runs, in one phase or in phases of at least `least` blocks of
// which about a quarter at most is repeated by the next one.
constexpr bool dq_phases_pay(int tokens, int group, int U, int reach, long long cap, long long least) {
  const long long blocks = ((long long)tokens * group + U - 1) / U;
  const long long repeated = ((long long)reach * group + U - 1) / U + 1;
  return cap >= blocks || (cap >= 4 * repeated && cap >= least);
}

}  // namespace sa
