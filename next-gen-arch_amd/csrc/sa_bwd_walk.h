// Walk of the dk2 / dv2 pass over its units: query t, head h of the KV group,
// 32-row group r of t's short keys, in ascending (t, h, r).  constexpr, so that
// the kernel and host checks run the same steps.
#pragma once

namespace sa {

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

}  // namespace sa
