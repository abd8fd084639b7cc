// Which heads of a float32 call run on the split fp16 products
// (bsa_fwd_f32s.hip), and at which scales; shared with the fp32 kernel
// (bsa_fwd_f32.hip), which takes the others.
#pragma once

#include "dsa_common.h"

namespace bsa {

constexpr int kMaxParts = 64;  // token ranges whose magnitudes are measured, per (tensor, head)
// Arrays [pairs][kMaxParts] of f32_range_kernel: the largest magnitude (fp32
// bits) of each range of Q, K and V; the smallest magnitude of V's range that
// has to survive the split; and which of V's 4-dim groups the range uses.
enum { kQMax, kKMax, kVMax, kVLow, kVUsed, kRangeKinds };

// Ranges of a tensor: at least 8 tokens each (or one), so that the largest of
// a dim's values over a range tells the dim's size.
__host__ __device__ constexpr int range_count(int tokens) {
  return tokens < 16 ? 1 : tokens / 8 < kMaxParts ? tokens / 8 : kMaxParts;
}

constexpr int kVSpread = 12;

// The scales of one (batch, head).
struct SplitScales {
  bool ok;           // the head runs here; else on the fp32 kernel
  float q, k, v;     // powers of two that Q, K and V are multiplied by
  float score_log2;  // log2 units per unit of the scaled S accumulator
  float out;         // 1 / v
};

// Every lane of a full wave calls it.  One scale per head and tensor leaves an
// element an absolute error of 2^-40 of the head's largest beside the relative
// 2^-23 of the split, and the probabilities one of 2^-36 of the row's largest.
// A head runs here only where neither can show:
//  * its largest magnitudes are 0 or within 2^+-40 (NaN and infinities exceed
//    that as bits) and the combined score scale is a normal number;
//  * Q and K: the absolute parts move a score (log2 units) by at most
//    D scale 2^(e_q + e_k - 37), and that is at most 2^-22, what the exp's own
//    argument is rounded to (with e_q + e_k 13, N(0,1) x 2^9 against N(0,1),
//    the error passes that of the fp32 products; 10, the most that D = 128
//    lets through, is half of it);
//  * V: every used group of 8 dims of every token, and every dim over every
//    token range, reaches 2^-kVSpread of the head's largest; N(0,1) takes 4
//    or 5 of those powers.  A group that no token uses is exact zeros.  (N(0,1)
//    with a dim 2^18 above the others, 256 tokens: theirs come out at 1.35
//    times the error of the fp32 products, 2^14 at 0.67.  With a token that
//    takes nearly all of every row's attention and is 2^-14 of the rest, 3.7
//    times, from the split of the small probabilities; 2^-10: 0.55.  So the
//    zeros of a used group count.)
__device__ __forceinline__ SplitScales split_scales(const uint32_t* ranges, int pairs, int bh,
                                                    float scale_log2, int head_dim,
                                                    int kv_tokens) {
  const int lane = threadIdx.x & 63;
  auto load = [&](int kind) -> uint32_t {
    return ranges[((int64_t)kind * pairs + bh) * kMaxParts + lane];
  };
  SplitScales s;
  s.ok = true;
  float scale[3];
  int e[3];
#pragma unroll
  for (int t = 0; t < 3; ++t) {
    uint32_t m = load(t);
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) m = max(m, (uint32_t)__shfl_xor((int)m, d));
    e[t] = (int)(m >> 23) - 127;  // floor(log2), or -127 for 0 and denormals
    s.ok = s.ok && (m == 0u || (e[t] >= -40 && e[t] <= 40));
    scale[t] = m == 0u || !s.ok ? 1.f : __uint_as_float((uint32_t)(127 + 14 - e[t]) << 23);
  }
  const bool in = lane < range_count(kv_tokens);
  uint32_t low = in ? load(kVLow) : 0xffffffffu;
  uint32_t any = in ? load(kVUsed) : 0u, all = in ? any : 0xffffffffu;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    low = min(low, (uint32_t)__shfl_xor((int)low, d));
    any |= (uint32_t)__shfl_xor((int)any, d);
    all &= (uint32_t)__shfl_xor((int)all, d);
  }
  s.ok = s.ok && any == all && e[kVMax] + 127 - (int)(low >> 23) <= kVSpread;
  const int e_s = e[kQMax] + e[kKMax];
  s.ok = s.ok && (e_s < -100 || scale_log2 * (float)head_dim *
                                        __uint_as_float((uint32_t)(127 + min(e_s, 127)) << 23) <=
                                    32768.f);
  s.q = scale[kQMax];
  s.k = scale[kKMax];
  s.v = scale[kVMax];
  s.score_log2 = scale_log2 / s.q / s.k;
  s.ok = s.ok && s.score_log2 >= 1.2e-38f && s.score_log2 <= 3e38f;
  s.out = 1.f / s.v;
  return s;
}

}  // namespace bsa
