// Which heads of a float32 call run on the split fp16 products
// (bsa_fwd_f32s.hip), and at which scales; shared with the fp32 kernel
// (bsa_fwd_f32.hip), which takes the others.
#pragma once

#include "dsa_common.h"

namespace bsa {

constexpr int kMaxParts = 64;                      // magnitude maxima per (tensor, head)

// The scales of one (batch, head).
struct SplitScales {
  bool ok;           // the head runs here; else on the fp32 kernel
  float q, k, v;     // powers of two that Q, K and V are multiplied by
  float score_log2;  // log2 units per unit of the scaled S accumulator
  float out;         // 1 / v
};

// `parts`: [3][pairs][kMaxParts] magnitude maxima (fp32 bits) of Q, K and V;
// every lane of a full wave calls it.  A head runs here when its largest
// magnitudes are 0 or within 2^+-40 (NaN and infinities exceed that as bits),
// no token range's is below 2^-14 of the head's (beside an outlier that far
// up, the other tokens' split would be coarser than fp32's rounding) and the
// combined score scale is a normal number.
__device__ __forceinline__ SplitScales split_scales(const uint32_t* parts, int pairs, int bh,
                                                    float scale_log2) {
  const int lane = threadIdx.x & 63;
  SplitScales s;
  s.ok = true;
  float scale[3];
#pragma unroll
  for (int t = 0; t < 3; ++t) {
    uint32_t m = parts[((int64_t)t * pairs + bh) * kMaxParts + lane];
    uint32_t low = m == 0u ? 0xffffffffu : m;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      m = max(m, (uint32_t)__shfl_xor((int)m, d));
      low = min(low, (uint32_t)__shfl_xor((int)low, d));
    }
    const int e = (int)(m >> 23) - 127;  // floor(log2), or -127 for 0 and denormals
    s.ok = s.ok && (m == 0u || (e >= -40 && e <= 40 && e + 127 - (int)(low >> 23) <= 14));
    scale[t] = m == 0u || !s.ok ? 1.f : __uint_as_float((uint32_t)(127 + 14 - e) << 23);
  }
  s.q = scale[0];
  s.k = scale[1];
  s.v = scale[2];
  s.score_log2 = scale_log2 / s.q / s.k;
  s.ok = s.ok && s.score_log2 >= 1.2e-38f && s.score_log2 <= 3e38f;
  s.out = 1.f / s.v;
  return s;
}

}  // namespace bsa
