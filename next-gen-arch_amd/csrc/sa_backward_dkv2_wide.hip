// dk2 / dv2 pass (sa_bwd_dkv2.h): the fp32 kernels, and the bf16 ones of score
// widths 256 and 512 (a translation unit of their own: compile time).
#include "sa_bwd_dkv2.h"

namespace sa {

hipError_t launch_bwd_dkv2_wide(const BwdParams& p, size_t scratch_bytes, hipStream_t stream) {
  if (p.f32) {
    if (p.d == 128) return launch_dkv2_pk<128, 128, 1, true>(p, scratch_bytes, stream);
    // fp32 walks are not cut into pieces: where blocks of 128 keys all run at
    // once, two sets per wave only lengthen the walks (2048 tokens, 8 / 8 heads,
    // windows 32 x 256, forward + backward: 1.63 ms with two, 1.13 with one; 6000
    // tokens, 376 such blocks: 2.47 ms with two)
    const int64_t blocks = ((int64_t)p.tokens + 127) / 128 * p.hk;
    return blocks <= device_cu_count() ? launch_dkv2_pk<64, 64, 1, true>(p, scratch_bytes, stream)
                                       : launch_dkv2_pk<64, 64, 2, true>(p, scratch_bytes, stream);
  }
  if (p.d == 512) {
    if (p.ws <= 16) return launch_dkv2_t<512, 256, 1, 2, false>(p, scratch_bytes, stream);
    return launch_dkv2_t<512, 256, 1, 1, false>(p, scratch_bytes, stream);
  }
  return p.dv == 256 ? launch_dkv2_pk<256, 256, 1>(p, scratch_bytes, stream)
                     : launch_dkv2_pk<256, 128, 1>(p, scratch_bytes, stream);
}

}  // namespace sa
