// dk2 / dv2 pass (sa_bwd_dkv2.h): launch, and the bf16 kernels of widths 64 and 128.
#include "sa_bwd_dkv2.h"

namespace sa {

namespace {

// Widths of 64 and 128: two sets per wave, or one where blocks of 128 keys take
// fewer steps in turn (dkv2_plan; kOneSet: a step of one set against one of two --
// its chain, not its products, takes the time): grids that are small for the pieces
// that the scratch holds.  Whole backward with one set against two, 160 shapes: 0.59
// to 0.98 of the time where the plan's steps are at most 1.05 times the two-set
// ones, 0.88 to 1.17 above.  1000 tokens, 8 / 2 heads, width 128: windows 128 x 128
// (no room for pieces: one launch per gradient and half of the short window had
// taken 8.64 ms) 10.4 -> 6.2 ms, 64 x 256 0.88 -> 0.60, with SA_FLAG_SEPARATE_DK1
// 7.6 -> 4.6 (3.5 by one launch per gradient, whose pieces were half as large).
template <int DK, int DV>
hipError_t launch_dkv2_sets(const BwdParams& p, size_t scratch_bytes, hipStream_t stream) {
  constexpr double kOneSet = 0.95;
  const int pk = dkv2_units(p);
  if (kOneSet * dkv2_plan(p, scratch_bytes, 128, pk).time < dkv2_plan(p, scratch_bytes, 256, pk).time)
    return launch_dkv2_pk<DK, DV, 1>(p, scratch_bytes, stream);
  return launch_dkv2_pk<DK, DV, 2>(p, scratch_bytes, stream);
}

}  // namespace

int64_t dkv2_piece_bytes(int tokens, int hk, int d, int dv) { return (int64_t)tokens * hk * (d + dv) * sizeof(float); }

// Short windows: up to 128 keys at widths <= 128, 64 at score width 256 (the
// k1 / v1 ring's LDS); fp32 inputs 32 (the other fp32 passes' bound).
hipError_t launch_bwd_dkv2_mfma(const BwdParams& p, size_t scratch_bytes, hipStream_t stream) {
  if (!bwd_mfma_ok(p)) return hipErrorNotSupported;
  const int per16 = p.f32 ? 4 : 8;  // elements per 16 bytes
  if (!walk_steps_fit(p.q_st / per16, p.q_sh / per16, p.group) || !walk_steps_fit(p.do_st / per16, p.do_sh / per16, p.group) ||
      !walk_steps_fit(p.k_st / per16, 0, 1) || !walk_steps_fit(p.v_st / per16, 0, 1))
    return hipErrorNotSupported;
  if (p.f32 ? p.ws > 32 : p.ws > (p.d > 256 ? 32 : p.d > 128 ? 64 : 128)) return hipErrorNotSupported;
  if (p.f32 || p.d > 128) return launch_bwd_dkv2_wide(p, scratch_bytes, stream);
  if (p.d == 128)
    return p.dv == 128 ? launch_dkv2_sets<128, 128>(p, scratch_bytes, stream)
                       : launch_dkv2_sets<128, 64>(p, scratch_bytes, stream);
  return p.dv == 128 ? launch_dkv2_sets<64, 128>(p, scratch_bytes, stream)
                     : launch_dkv2_sets<64, 64>(p, scratch_bytes, stream);
}

}  // namespace sa
