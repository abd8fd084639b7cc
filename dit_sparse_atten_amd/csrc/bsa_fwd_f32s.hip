// Float32 attention on the fp16 matrix cores (gfx950): every fp32 operand as
// the sum of two fp16 numbers.  Replaces, like bsa_fwd_f32.hip, the float32
// SDPA of the reference's DenseBackend (attention_backends/dense.py:34-47) and
// the float32 `sparse_chunk` / `_dense_route` of MatrixSparseBackend
// (attention_backends/sparse.py:184-233, 670-751), for head dims up to 128 and
// without dropout.
//
// x = hi + lo with hi = fp16(x), lo = fp16(x - hi) holds 22 bits and a sign of
// x, and x y is hi hi + hi lo + lo hi up to 2^-24 |x y| (Ootomo and Yokota,
// "Recovering single precision accuracy from Tensor Cores while surpassing the
// FP32 theoretical peak performance", IJHPCA 2022): three products at the
// 16-bit rate, 16 times that of v_mfma_f32_32x32x2_f32.  Each MFMA adds 16
// products to the fp32 accumulator where the fp32 instruction adds 2, so there
// are fewer roundings than in the fp32 products it stands for, and on ordinary
// inputs the result is closer to 64 bits than theirs (N(0,1), 3,600 tokens x 2
// heads, relative error of O: 4.4e-7, fp32 kernel 1.17e-6).
//
// fp16's range: each head of Q, K and V is scaled by the power of two that
// takes its largest magnitude into [2^14, 2^15) (f32_range_kernel finds it),
// so the split of an element is exact to 2^-23 of it, or to 2^-40 of the
// head's largest; the scales leave the fp32 accumulators exactly.  The
// probabilities are computed 2^11 times larger, with the row's reference kept
// within 2^4 of its largest score, for the same reason: to 2^-23, or to 2^-36
// of the row's largest.  A head with a non-finite or extreme element, or whose
// dims or tokens differ so much that these absolute parts would show
// (split_scales), is left to the fp32 kernel, launched over the same grid,
// whose workgroups return at once for the others.
//
// Error of O against float64 over that of the fp32 kernel, N(0,1): 0.87 to 0.38
// at 128 dims from 33 to 3,600 tokens, 0.99 to 0.38 at 64.  Fewer dims and few
// keys have few roundings in fp32 (8 dims: 1.7 at 16 tokens, 1.03 at 128, 0.94
// at 256), and run here only from 256 keys for every row (split_takes).
//
// Work per 32-key sub-tile and 32 query rows: 48 MFMAs (24 for S^T, 24 for
// O^T) beside 16 exps and 16 two-way splits per lane; matrix-core bound.  K
// and V are split once per call (f32_split_kernel) into rows of 128 hi and 128
// lo values, so a sub-tile is 16 KB of each, staged and read exactly as the
// 16-bit kernel's 64-key half-tile (bsa_kernel.h): buffer -> LDS loads one
// sub-tile ahead, K chunks XOR-swizzled, V^T through the transposing read.
// Measured against the fp32 kernel, same box: dense 14,400 tokens x 12 heads
// 11.59 -> 3.35 ms (380 TFLOP/s), 3,600 tokens 1.00 -> 0.28 ms; 12,288 tokens in
// 8 x 8 tiles with statistics, routed (keep 0.625) 10.2 -> 2.1 ms, dense 16.2 ->
// 3.0 ms.
#include "bsa_kernel.h"
#include "bsa_split.h"

namespace bsa {

constexpr int kSplitKeys = 32;                     // keys per staged sub-tile
constexpr int kSplitRow = 4 * kHeadDim;            // bytes of a split row: 128 hi, 128 lo
constexpr float kPScaleLog2 = 11.0f;               // P is computed 2^11 times larger
constexpr float kPUnscale = 1.0f / 2048.0f;
constexpr float kSplitMoveLog2 = 4.0f;             // the reference moves past 2^4

// hi and lo fp16 parts of eight scaled values.
__device__ __forceinline__ void split8(const dsa_f32x4& a, const dsa_f32x4& b, float scale,
                                       dsa_f16x8& hi, dsa_f16x8& lo) {
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float x = (e < 4 ? a[e & 3] : b[e & 3]) * scale;
    hi[e] = (_Float16)x;
    lo[e] = (_Float16)(x - (float)hi[e]);
  }
}

// Magnitudes of the token ranges of every head of Q, K and V (split_scales):
// workgroup (range, bh, tensor), 32 lanes per token (4 dims each).
__global__ void __launch_bounds__(256) f32_range_kernel(BsaParams p, uint32_t* ranges) {
  const int part = blockIdx.x, bh = blockIdx.y, t = blockIdx.z, pairs = gridDim.y;
  const int h = bh % p.heads, b = bh / p.heads;
  const int tokens = t == kQMax ? p.q_tokens : p.kv_tokens;
  const int64_t st = t == kQMax ? p.q_st : t == kKMax ? p.k_st : p.v_st;
  const float* base = t == kQMax   ? static_cast<const float*>(p.q) + b * p.q_sb + h * p.q_sh
                      : t == kKMax ? static_cast<const float*>(p.k) + b * p.k_sb + h * p.k_sh
                                   : static_cast<const float*>(p.v) + b * p.v_sb + h * p.v_sh;
  const int count = range_count(tokens);
  const int t0 = part < count ? (int)((int64_t)tokens * part / count) : 0;
  const int t1 = part < count ? (int)((int64_t)tokens * (part + 1) / count) : 0;
  const int c = threadIdx.x & 31;
  // Per lane: the largest of each of its dims, and the smallest over the tokens
  // of its 8-dim group's largest (lanes c and c ^ 1 share a group).
  uint32_t dim[4] = {0u, 0u, 0u, 0u}, group = 0xffffffffu;
  if (c * 4 < p.head_dim) {
    for (int i = t0 + (threadIdx.x >> 5); i < t1; i += 8) {
      const dsa_u32x4 x = *reinterpret_cast<const dsa_u32x4*>(base + (int64_t)i * st + c * 4);
      uint32_t top = 0u;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t m = x[e] & 0x7fffffffu;
        dim[e] = max(dim[e], m);
        top = max(top, m);
      }
      group = min(group, max(top, (uint32_t)__shfl_xor((int)top, 1)));
    }
  }
  __shared__ uint32_t part_of[4][32][5];
#pragma unroll
  for (int e = 0; e < 4; ++e) dim[e] = max(dim[e], (uint32_t)__shfl_xor((int)dim[e], 32));
  group = min(group, (uint32_t)__shfl_xor((int)group, 32));
  if ((threadIdx.x & 32) == 0) {
    uint32_t* to = part_of[threadIdx.x >> 6][c];
#pragma unroll
    for (int e = 0; e < 4; ++e) to[e] = dim[e];
    to[4] = group;
  }
  dsa::lds_barrier();
  if (threadIdx.x >= 32) return;
  uint32_t best = 0u, low = 0xffffffffu;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    uint32_t m = 0u;
#pragma unroll
    for (int w = 0; w < 4; ++w) m = max(m, part_of[w][c][e]);
    best = max(best, m);
    if (m != 0u) low = min(low, m);
  }
  const bool used = max(best, (uint32_t)__shfl_xor((int)best, 1)) != 0u;
  if (used)
#pragma unroll
    for (int w = 0; w < 4; ++w) low = min(low, part_of[w][c][4]);
  const uint32_t lanes_used = (uint32_t)__ballot(used);
#pragma unroll
  for (int d = 1; d < 32; d <<= 1) {
    best = max(best, (uint32_t)__shfl_xor((int)best, d));
    low = min(low, (uint32_t)__shfl_xor((int)low, d));
  }
  if (c == 0) {
    const int64_t at = (int64_t)bh * kMaxParts + part, kind = (int64_t)pairs * kMaxParts;
    ranges[t * kind + at] = best;
    if (t == kVMax) {
      ranges[kVLow * kind + at] = low;
      ranges[kVUsed * kind + at] = lanes_used;
    }
  }
}

// Scaled split rows of K (z = 0) and V (z = 1): workgroup (64 tokens, bh), 16
// lanes per token (8 dims each; dims past head_dim are zeros).
constexpr int kSplitTokens = 64;
__global__ void __launch_bounds__(256) f32_split_kernel(BsaParams p, const uint32_t* ranges,
                                                       unsigned char* planes) {
  const int bh = blockIdx.y, pairs = gridDim.y;
  const bool is_v = blockIdx.z != 0;
  const SplitScales sc = split_scales(ranges, pairs, bh, p.scale_log2, p.head_dim, p.kv_tokens);
  if (!sc.ok) return;
  const int h = bh % p.heads, b = bh / p.heads;
  const float scale = is_v ? sc.v : sc.k;
  const int64_t st = is_v ? p.v_st : p.k_st;
  const float* base = is_v ? static_cast<const float*>(p.v) + b * p.v_sb + h * p.v_sh
                           : static_cast<const float*>(p.k) + b * p.k_sb + h * p.k_sh;
  unsigned char* out =
      planes + ((int64_t)(is_v ? pairs : 0) + bh) * p.kv_tokens * kSplitRow;
  const int c = threadIdx.x & 15;
#pragma unroll
  for (int u = 0; u < kSplitTokens / 16; ++u) {
    const int i = blockIdx.x * kSplitTokens + u * 16 + (threadIdx.x >> 4);
    if (i >= p.kv_tokens) break;
    dsa_f32x4 a = {0.f, 0.f, 0.f, 0.f}, d = a;
    if (c * 8 < p.head_dim) {
      const float* src = base + (int64_t)i * st + c * 8;
      a = *reinterpret_cast<const dsa_f32x4*>(src);
      d = *reinterpret_cast<const dsa_f32x4*>(src + 4);
    }
    dsa_f16x8 hi, lo;
    split8(a, d, scale, hi, lo);
    unsigned char* row = out + (int64_t)i * kSplitRow + c * 16;
    *reinterpret_cast<dsa_f16x8*>(row) = hi;
    *reinterpret_cast<dsa_f16x8*>(row + 2 * kHeadDim) = lo;
  }
}

// kWaves: 32 query rows each (4, or 2 for blocks of at most 64 tokens).
// kSingle: one LDS stage pair, filled after every wave is done with it: half
// the LDS, so that twice as many 2-wave workgroups share a CU and cover each
// other's waits; calls too small to give a CU that many keep two.
template <bool kRouted, bool kStats, int kWaves, bool kSingle>
__global__ void __launch_bounds__(kWaves * 64, 2) bsa_fwd_split_kernel(
    BsaParams p, const uint32_t* ranges, const unsigned char* planes) {
  typedef dsa::Elem<_Float16> E;
  __shared__ __attribute__((aligned(1024))) unsigned char lds_k0[kKStage];
  __shared__ __attribute__((aligned(1024))) unsigned char lds_k1[kSingle ? 16 : kKStage];
  __shared__ __attribute__((aligned(1024))) unsigned char lds_v0[kKStage];
  __shared__ __attribute__((aligned(1024))) unsigned char lds_v1[kSingle ? 16 : kKStage];
  __shared__ dsa_f32x2 offs[kStats ? 128 : 1];
  static_assert(kSplitKeys * kSplitRow == kKStage, "a split sub-tile fills a stage");

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5;
  const int qi = lane & 31;
  // Split last round, as in bsa_fwd_kernel (bsa_merge_kernel combines the parts).
  const int wg = (int)blockIdx.x;
  const bool split = wg >= p.split_from;
  int work = wg, part = 0;
  if (split) {
    const int t = wg - p.split_from;
    work = p.split_from + t / p.parts;
    part = t % p.parts;
  } else if (!kRouted) {
    work = dsa::xcd_remap(wg, p.split_from);
  }
  const int qb = work % p.q_blocks;
  const int bh = work / p.q_blocks;
  const int h = bh % p.heads;
  const int b = bh / p.heads;
  const int pairs = p.batch * p.heads;
  const SplitScales sc = split_scales(ranges, pairs, bh, p.scale_log2, p.head_dim, p.kv_tokens);
  if (!sc.ok) return;  // every wave alike: the fp32 kernel takes this head

  int start = 0, end = p.kv_blocks;
  if (!kRouted && p.causal) {
    const int last_row = min(qb * p.block + p.block, p.q_tokens) - 1;
    end = min(p.kv_blocks, last_row / p.block + 1);
  }
  if (kRouted) {
    const dsa_const_i32 rp = (dsa_const_i32)p.row_ptr;
    const int rb = p.route_batches == 1 ? 0 : b;
    const int64_t row = ((int64_t)rb * p.heads + h) * p.q_blocks + qb;
    start = rp[row];
    end = rp[row + 1];
  }
  if (split) {
    const int n = end - start;
    end = start + (int)((int64_t)n * (part + 1) / p.parts);
    start = start + (int)((int64_t)n * part / p.parts);
  }
  const dsa_const_i32 cidx = (dsa_const_i32)p.col_idx;
  const int nblk = end - start;

  const int local_row = wave * 32 + qi;
  const int tq = qb * p.block + local_row;
  const bool row_ok = local_row < p.block && tq < p.q_tokens;
  const bool wave_active = wave * 32 < p.block;
  const int tq_c = tq < p.q_tokens ? tq : p.q_tokens - 1;

  // Split Q fragments: dims 16 dc + 8 g .. + 7 of the lane's query row.
  dsa_f16x8 qh[8], ql[8];
  {
    const float* qrow = static_cast<const float*>(p.q) + b * p.q_sb + h * p.q_sh +
                        (int64_t)tq_c * p.q_st;
#pragma unroll
    for (int dc = 0; dc < 8; ++dc) {
      dsa_f32x4 a = {0.f, 0.f, 0.f, 0.f}, c = a;
      if (dc * 16 + g * 8 < p.head_dim) {
        a = *reinterpret_cast<const dsa_f32x4*>(qrow + dc * 16 + g * 8);
        c = *reinterpret_cast<const dsa_f32x4*>(qrow + dc * 16 + g * 8 + 4);
      }
      split8(a, c, sc.q, qh[dc], ql[dc]);
    }
  }
  if constexpr (kStats) {
    // Tile-local (y, x) of each key offset in a block (zeros past it: masked
    // keys read them with p = 0).
    for (int i = tid; i < 128; i += kWaves * 64) {
      const bool in = i < p.stat_tile;
      offs[i] = dsa_f32x2{in ? dsa::tile_axis(i / p.tile_w, p.tile_h) : 0.f,
                          in ? dsa::tile_axis(i % p.tile_w, p.tile_w) : 0.f};
    }
    dsa::lds_barrier();
  }

  const unsigned char* kplane = planes + (int64_t)bh * p.kv_tokens * kSplitRow;
  const unsigned char* vplane = planes + ((int64_t)pairs + bh) * p.kv_tokens * kSplitRow;
  auto block_of = [&](int j) -> int {
    const int kb = kRouted ? cidx[start + j] : start + j;
    return (unsigned)kb < (unsigned)p.kv_blocks ? kb : -1;
  };
  // The first walk index at or past j whose key block is in range.
  auto next_valid = [&](int j) -> int {
    while (j < nblk && block_of(j) < 0) ++j;
    return j;
  };

  // Staging: slice i of a stage's 16 1-KB slices holds 4 rows of the hi (i < 8)
  // or lo part; each wave loads kSlices of K and of V.
  constexpr int kSlices = 16 / kWaves;
  uint32_t koff[kSlices], voff[kSlices];
#pragma unroll
  for (int u = 0; u < kSlices; ++u) {
    const int idx = (wave * kSlices + u) * 64 + lane;
    const int row = (idx >> 4) & (kSplitKeys - 1), part = idx >> 9;
    const int at = row * kSplitRow + part * 2 * kHeadDim;
    koff[u] = (uint32_t)(at + k2_swz(row, idx & 15) * 16);
    voff[u] = (uint32_t)(at + v_swz(row, idx & 15) * 16);
  }
  auto issue = [&](int kb, int st, unsigned char* kdst, unsigned char* vdst)
      __attribute__((always_inline)) {
    const int key0 = kb * p.block + st * kSplitKeys;
    const int rows = min(kSplitKeys, p.kv_tokens - key0);
    const uint32_t bytes = rows > 0 ? (uint32_t)(rows * kSplitRow) : 0u;
    const __amdgpu_buffer_rsrc_t k_rsrc = make_rsrc(kplane + (int64_t)key0 * kSplitRow, bytes);
    const __amdgpu_buffer_rsrc_t v_rsrc = make_rsrc(vplane + (int64_t)key0 * kSplitRow, bytes);
#pragma unroll
    for (int u = 0; u < kSlices; ++u)
      lds_load16(k_rsrc, kdst + (wave * kSlices + u) * 1024, koff[u], 0);
#pragma unroll
    for (int u = 0; u < kSlices; ++u)
      lds_load16(v_rsrc, vdst + (wave * kSlices + u) * 1024, voff[u], 0);
  };

  // V^T fragment reads, as in bsa_fwd_kernel.
  int vfrag[4];
  {
    const int lam = lane & 15, r = lam >> 2, c = lam & 3;
    const int row = 4 * g + r;
    const int sub = 2 * ((lane >> 4) & 1) + (c >> 1);
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
      vfrag[dt] = row * kRowBytes + v_swz(row, 4 * dt + sub) * 16 + (c & 1) * 8;
  }

  float m_run = -INFINITY;  // log2 units of the scaled scores
  float l_run = 0.f;
  dsa_f32x16 oacc[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) oacc[dt][r] = 0.f;
  float cm = 0.f, cy = 0.f, cx = 0.f;  // statistics of the open key tile

  constexpr int kLo = kSplitKeys * kRowBytes;  // the lo part of a stage
  auto compute = [&](const unsigned char* k_lds, const unsigned char* v_lds, int kb, int st)
      __attribute__((always_inline)) {
    const int key0 = kb * p.block + st * kSplitKeys;
    const int valid = min(kSplitKeys, min(p.block - st * kSplitKeys, p.kv_tokens - key0));
    const int lim = !kRouted && p.causal ? tq - key0 + 1 : kSplitKeys;
    // hi hi and the two cross products in accumulators of their own: the
    // small terms are summed before they meet the large ones.
    dsa_f32x16 s, x;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = x[r] = 0.f;
#pragma unroll
    for (int dc = 0; dc < 8; ++dc) {
      const unsigned char* at = k_lds + qi * kRowBytes + k2_swz(qi, dc * 2 + g) * 16;
      const dsa_f16x8 kh = *reinterpret_cast<const dsa_f16x8*>(at);
      const dsa_f16x8 kl = *reinterpret_cast<const dsa_f16x8*>(at + kLo);
      s = E::mfma32(kh, qh[dc], s);
      x = E::mfma32(kh, ql[dc], x);
      x = E::mfma32(kl, qh[dc], x);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] += x[r];
    const int bound = min(valid, lim);
    if (bound < kSplitKeys) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (8 * (r >> 2) + 4 * g + (r & 3) >= bound) s[r] = -INFINITY;
    }
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[r]);
    mx = dsa::pair32_max(mx) * sc.score_log2;
    const bool up = mx > m_run + kSplitMoveLog2;
    if (__any(up)) {
      // A whole number: the rescale is a power of two, and the reference
      // leaves no rounding in the exponents, the LSE or the log-masses.
      const float m_new = floorf(mx);
      const float alpha = up ? __builtin_amdgcn_exp2f(m_run - m_new) : 1.f;
      if (up) m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[dt][r] *= alpha;
      if constexpr (kStats) {
        cm *= alpha;
        cy *= alpha;
        cx *= alpha;
      }
    }
    const float m_use = m_run == -INFINITY ? 0.f : m_run - kPScaleLog2;
    dsa_f16x8 ph[2], pl[2];
    float sum0 = 0.f, sum1 = 0.f;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        const float pr = __builtin_amdgcn_exp2f(fmaf(s[8 * j + t], sc.score_log2, -m_use));
        if (t & 1) sum1 += pr;
        else sum0 += pr;
        ph[j][t] = (_Float16)pr;
        pl[j][t] = (_Float16)(pr - (float)ph[j][t]);
        if constexpr (kStats) {
          const int r = 8 * j + t;
          const dsa_f32x2 o = offs[st * kSplitKeys + 8 * (r >> 2) + 4 * g + (r & 3)];
          cy = fmaf(pr, o[0], cy);
          cx = fmaf(pr, o[1], cx);
        }
      }
    }
    l_run += sum0 + sum1;
    if constexpr (kStats) cm += sum0 + sum1;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
      for (int d2 = 0; d2 < 4; d2 += 2) {
        dsa_f16x8 a[2][2];
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int part = 0; part < 2; ++part) {
            const unsigned char* at = v_lds + vfrag[d2 + u] + j * 16 * kRowBytes + part * kLo;
            const dsa_f16x4 lo = lds_read_tr<_Float16>(at);
            const dsa_f16x4 hi = lds_read_tr<_Float16>(at + 8 * kRowBytes);
            a[u][part] = dsa_f16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
          }
        // Two output tiles in turn, so that no product waits for the one before.
#pragma unroll
        for (int u = 0; u < 2; ++u) oacc[d2 + u] = E::mfma32(a[u][1], ph[j], oacc[d2 + u]);
#pragma unroll
        for (int u = 0; u < 2; ++u) oacc[d2 + u] = E::mfma32(a[u][0], pl[j], oacc[d2 + u]);
#pragma unroll
        for (int u = 0; u < 2; ++u) oacc[d2 + u] = E::mfma32(a[u][0], ph[j], oacc[d2 + u]);
      }
    }
  };

  // The statistics of walk index j (key block kb), after its last sub-tile.
  auto close_tile = [&](int j, int kb) {
    const float tm = dsa::pair32_sum(cm), ty = dsa::pair32_sum(cy), tx = dsa::pair32_sum(cx);
    if (g == 0 && row_ok) {
      int64_t at;
      bool ok = true;
      if (kRouted) {
        const int64_t e = start + j;
        at = e * p.block + local_row;
        ok = e < p.rs_entries;
      } else {
        at = ((int64_t)h * p.kv_blocks + kb) * p.q_tokens + tq;
      }
      if (ok) {
        p.rs_logm[at] = tm > 0.f ? log2f(tm * kPUnscale) + m_run : -INFINITY;
        if (p.rs_mean != nullptr) {
          const float inv = tm > 0.f ? 1.f / tm : 0.f;
          const dsa_f16x2 mean =
              __builtin_convertvector(dsa_f32x2{ty * inv, tx * inv}, dsa_f16x2);
          p.rs_mean[at] = __builtin_bit_cast(uint32_t, mean);
        }
      }
    }
    cm = cy = cx = 0.f;
  };

  int j = next_valid(0), st = 0;
  int kb = j < nblk ? block_of(j) : -1;
  if (j < nblk) issue(kb, 0, lds_k0, lds_v0);
  // One sub-tile: wait for its stage, load the next one, compute.
  auto step = [&](const unsigned char* kc, const unsigned char* vc, unsigned char* kn,
                  unsigned char* vn) __attribute__((always_inline)) {
    int nj = j, nst = st + 1, nkb = kb;
    if (nst * kSplitKeys >= min(p.block, p.kv_tokens - kb * p.block)) {
      nst = 0;
      nj = next_valid(j + 1);
      nkb = nj < nblk ? block_of(nj) : -1;
    }
    const bool more = nj < nblk;
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    __syncthreads();
    if (!kSingle && more) issue(nkb, nst, kn, vn);
    if (wave_active) {
      compute(kc, vc, kb, st);
      if constexpr (kStats) {
        if (nst == 0) close_tile(j, kb);
      }
    }
    if constexpr (kSingle) {
      __syncthreads();  // every wave is done with the stage
      if (more) issue(nkb, nst, kn, vn);
    }
    j = nj;
    st = nst;
    kb = nkb;
  };
  while (j < nblk) {
    step(lds_k0, lds_v0, kSingle ? lds_k0 : lds_k1, kSingle ? lds_v0 : lds_v1);
    if (kSingle) continue;
    if (j >= nblk) break;
    step(lds_k1, lds_v1, lds_k0, lds_v0);
  }

  const float l_tot = dsa::pair32_sum(l_run);
  if (split) {
    if (row_ok) {
      float* po = p.part + (int64_t)(wg - p.split_from) * kPartFloats;
      const float unscale = sc.out * kPUnscale;  // powers of two
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr)
          *reinterpret_cast<dsa_f32x4*>(po + local_row * kHeadDim + dt * 32 + rr * 8 + g * 4) =
              dsa_f32x4{oacc[dt][rr * 4 + 0] * unscale, oacc[dt][rr * 4 + 1] * unscale,
                        oacc[dt][rr * 4 + 2] * unscale, oacc[dt][rr * 4 + 3] * unscale};
      if (g == 0) {
        po[128 * 128 + local_row] = m_run;
        po[128 * 128 + 128 + local_row] = l_tot * kPUnscale;
      }
    }
    return;
  }
  const float inv = (l_tot > 0.f ? 1.f / l_tot : 0.f) * sc.out;
  if (row_ok) {
    float* orow = static_cast<float*>(p.o) + b * p.o_sb + h * p.o_sh + (int64_t)tq * p.o_st;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        const int dim = dt * 32 + rr * 8 + g * 4;
        if (dim < p.head_dim)
          *reinterpret_cast<dsa_f32x4*>(orow + dim) =
              dsa_f32x4{oacc[dt][rr * 4 + 0] * inv, oacc[dt][rr * 4 + 1] * inv,
                        oacc[dt][rr * 4 + 2] * inv, oacc[dt][rr * 4 + 3] * inv};
      }
    if (p.lse && g == 0)
      p.lse[((int64_t)b * p.heads + h) * p.q_tokens + tq] =
          l_tot > 0.f ? m_run * 0.6931471805599453f + logf(l_tot * kPUnscale) : -INFINITY;
  }
}

// Bytes of the range magnitudes and the split K and V of `pairs` (batch, head)
// pairs, rounded up to 256.
size_t split_workspace_bytes(int64_t pairs, int64_t kv_tokens) {
  return round256((size_t)(kRangeKinds * pairs * kMaxParts * (int64_t)sizeof(uint32_t) +
                           2 * pairs * kv_tokens * kSplitRow));
}

// Whether a float32 call runs here: at head dims below 64 only where every row
// attends 256 keys (see the errors above), and only with enough keys for four
// launches, each waiting for the one before, to beat one launch of the fp32
// kernel, whose workgroups take 0.15 us per key.  us here / there, same box:
// 3,600 queries x 12 heads on 32 keys 32 / 23, 2,400 x 40 on 64 keys 55 / 52; 96
// keys: 96 tokens x 12 heads 24 / 20 (1,024 queries on 77 keys 28 / 23), but
// 3,600 queries x 12 heads 37 / 43 and 14,400 x 40 on 77 keys 275 / 319, as the
// fp32 kernel runs out of CUs; 97 tokens x 12 heads 25 / 25, 256 tokens 32 / 45.
bool split_takes(const BsaParams& p) {
  if (p.kv_tokens <= kSplitFewKeys) return false;
  if (p.kv_tokens <= 96 && (int64_t)p.batch * p.heads * p.q_blocks <= 256) return false;
  return p.head_dim >= 64 || (p.row_ptr == nullptr && p.causal == 0 && p.kv_tokens >= 256);
}

}  // namespace bsa

// Launches a prepared float32 call (head dim up to 128, no dropout) on at least
// split_workspace_bytes of 16-byte aligned workspace (what follows them holds
// split partials): the heads that run here, then the fp32 kernel over the rest.
int bsa_launch_f32_split(bsa::BsaParams p, void* workspace, size_t workspace_bytes,
                         hipStream_t stream, const char* who) {
  using namespace bsa;
  const unsigned pairs = (unsigned)(p.batch * p.heads);
  uint32_t* ranges = static_cast<uint32_t*>(workspace);
  unsigned char* planes = static_cast<unsigned char*>(workspace) +
                          (size_t)kRangeKinds * pairs * kMaxParts * sizeof(uint32_t);
  hipLaunchKernelGGL(f32_range_kernel, dim3(kMaxParts, pairs, 3), dim3(256), 0, stream, p, ranges);
  hipLaunchKernelGGL(f32_split_kernel,
                     dim3((unsigned)((p.kv_tokens + kSplitTokens - 1) / kSplitTokens), pairs, 2),
                     dim3(256), 0, stream, p, ranges, planes);
  const int64_t grid = (int64_t)pairs * p.q_blocks;
  // 2-wave workgroups with two stages put two on a CU, with one stage four:
  // the latter where the call has more than two per CU.
  const int slots = device_slots(stream);
  const bool two = p.block <= 64, single = grid > slots;
  // Split last round: a 4-wave workgroup alone on a CU runs nearly twice as fast
  // as one of two, so a round is one per CU (2-wave ones: two).  Whole calls,
  // dense, us without and with it: 144 workgroups (1,536 tokens x 12 heads) 93 ->
  // 81, 160 (4,096 x 5) 204 -> 157, 192 (8,192 x 3) 405 -> 317, 192 of 16 key
  // blocks 121 -> 119, 348 (3,600 x 12) 299 -> 270, 564 (6,000 x 12) 782 -> 628;
  // 400 of 10 key blocks, 456 and 480 are not split.
  const size_t lead = split_workspace_bytes(pairs, p.kv_tokens);
  p.part = reinterpret_cast<float*>(static_cast<unsigned char*>(workspace) + lead);
  p.parts = 1;
  const int split = choose_split(
      grid, two ? slots : slots / 2, split_max_parts(p.kv_blocks),
      std::min<int64_t>((int64_t)((workspace_bytes - lead) / kPartBytes), kMaxPartGroups), &p.parts);
  p.split_from = (int32_t)(grid - split);
  const dim3 blocks((unsigned)(grid - split + (int64_t)split * p.parts));
  auto run = [&](auto kernel, int waves) {
    hipLaunchKernelGGL(kernel, blocks, dim3((unsigned)waves * 64), 0, stream, p, ranges, planes);
  };
  if (p.row_ptr) {
    if (p.rs_logm) {
      if (!two) run(bsa_fwd_split_kernel<true, true, 4, false>, 4);
      else if (single) run(bsa_fwd_split_kernel<true, true, 2, true>, 2);
      else run(bsa_fwd_split_kernel<true, true, 2, false>, 2);
    } else {
      if (!two) run(bsa_fwd_split_kernel<true, false, 4, false>, 4);
      else if (single) run(bsa_fwd_split_kernel<true, false, 2, true>, 2);
      else run(bsa_fwd_split_kernel<true, false, 2, false>, 2);
    }
  } else {
    if (p.rs_logm) {
      if (!two) run(bsa_fwd_split_kernel<false, true, 4, false>, 4);
      else if (single) run(bsa_fwd_split_kernel<false, true, 2, true>, 2);
      else run(bsa_fwd_split_kernel<false, true, 2, false>, 2);
    } else {
      if (!two) run(bsa_fwd_split_kernel<false, false, 4, false>, 4);
      else if (single) run(bsa_fwd_split_kernel<false, false, 2, true>, 2);
      else run(bsa_fwd_split_kernel<false, false, 2, false>, 2);
    }
  }
  if (split > 0) launch_merge<float>(p, split, stream);
  p.split_ranges = ranges;
  return bsa_launch_f32(p, DSA_F32, stream, who);
}
