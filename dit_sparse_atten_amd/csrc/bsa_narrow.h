// Attention on tile blocks of 65..96 tokens (gfx950), bf16 or fp16: the gathered
// key stream of bsa_fwd_kernel with query rows in groups of 16.  Routed calls,
// and dense ones (kRouted = false: every block listed) that take statistics of
// such tiles.  Included by bsa_kernel.h, whose definitions it uses.
//
// On the 32-row MFMAs of bsa_fwd_kernel a 72-row query tile fills three waves'
// 96 rows and leaves the fourth wave of a workgroup idle, so a CU's two
// workgroups advance 144 rows in the time eight full waves advance 256.  Here
// v_mfma_f32_16x16x32 takes the rows in groups of 16 (72 -> 80 rows), three
// groups to a wave: two waves cover a tile, a workgroup needs one 32 KB stage
// pair (K and V of a 64-key chunk), and four workgroups share a CU.  Each
// fragment read from LDS feeds up to three products.  720p (9 x 8 tiles, keep
// 0.65, 57,600 tokens x 40 heads), same box: 57.9 -> 50.0 ms, with statistics
// and their reduction 71.7 -> 61.5 ms.  What bounds it: streaming each kept
// chunk from L2 for 72 rows (607 GB per call; without the loads, timing only,
// 39 ms) and the wave that holds three of the five groups (two each: 42 ms).
// Longer prefetch (32-key double-buffered stages) and three waves of two groups
// measured no faster; blocks of 57..64 tokens (two groups per wave) ran equal to
// the 32-row 2-wave kernel.  Dense statistics, 240 tiles x 40 heads: 5 x 13
// tokens 14.3 -> 9.4 ms, 9 x 10 tokens 15.0 -> 13.2 ms.
//
// Layouts (lane = 16 q4 + c16): S^T = K Q^T leaves lane (q4, c16) the keys
// 16 kg + 4 q4 + r of query row c16 (r = 0..3), and two 16-key groups' values
// are the eight k slots of P^T in O^T = V^T P^T, whose V^T fragments come out
// of the stage through the transposing LDS read with the keys in that order.
// O^T leaves lane (q4, c16) the dims 16 dt + 4 q4 + r of row c16.
//
// kStats: the key-side sums of a tile (rs_logm, rs_mean) accumulate over its
// chunks in one 16x16 accumulator per row group: C += W^T P^T, where W^T holds
// for the stream's even tiles the rows 0..2 = 1, Y, X and for the odd ones
// rows 4..6, so lanes q4 = 0 hold the even tile's three sums and q4 = 1 the
// odd one's.  Y and X are the offsets 2 i - (n - 1) on a tile side of n
// tokens, whole numbers and so exact in the input type; the mean is divided
// by n - 1 when the tile closes.
#pragma once

namespace bsa {

constexpr int kNarrowGroups = 3;   // 16-row groups per wave
constexpr int kNarrowCols = 264;   // >= 2 * 96 + 64 stream positions, = 8 mod 64
constexpr int kNarrowWRows = 7;    // 2 parities x 3 kinds, then a zero row

// V chunk c of key row r sits at chunk position c ^ 2 (r & 7): a transposed
// read touches 16 key rows x 32 bytes, eight rows (256 bytes) at a time.
__device__ __forceinline__ int v8_swz(int r, int c) { return c ^ (2 * (r & 7)); }

template <typename T, bool kRouted, bool kStats>
__global__ void __launch_bounds__(128, 2) bsa_fwd_narrow_kernel(BsaParams p) {
  typedef dsa::Elem<T> E;
  typedef typename E::x8 x8;
  typedef typename E::x4 x4;
  __shared__ __attribute__((aligned(1024))) unsigned char lds_k[kKStage];
  __shared__ __attribute__((aligned(1024))) unsigned char lds_v[kKStage];
  __shared__ __attribute__((aligned(16))) T wtab[kStats ? kNarrowWRows * kNarrowCols : 8];
  __shared__ int wg_lds, rot_lds;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q4 = lane >> 4;
  const int c16 = lane & 15;

  // Launch slot, split range and aligned walk as in bsa_fwd_kernel.
  int wg = (int)blockIdx.x;
  if (p.queue != nullptr) {
    if (tid == 0)
      wg_lds = __hip_atomic_fetch_add(p.queue, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    dsa::lds_barrier();
    wg = __builtin_amdgcn_readfirstlane(wg_lds);
  }
  const bool split = wg >= p.split_from;
  int slot = wg, part = 0;
  if (split) {
    const int t = wg - p.split_from;
    slot = p.split_from + t / p.parts;
    part = t % p.parts;
  }
  int work = slot;
  if (kRouted && p.order) work = ((dsa_const_i32)p.order)[slot];
  const int qb = work % p.q_blocks;
  const int bh = work / p.q_blocks;
  const int h = bh % p.heads;
  const int b = bh / p.heads;
  int start = 0, end = p.kv_blocks;
  if (kRouted) {
    const dsa_const_i32 rp = (dsa_const_i32)p.row_ptr;
    const int rb = p.route_batches == 1 ? 0 : b;
    const int64_t csr_row = ((int64_t)rb * p.heads + h) * p.q_blocks + qb;
    start = rp[csr_row];
    end = rp[csr_row + 1];
  }
  if (split) {
    const int n = end - start;
    end = start + (int)((int64_t)n * (part + 1) / p.parts);
    start = start + (int)((int64_t)n * part / p.parts);
  }
  const dsa_const_i32 cidx = (dsa_const_i32)p.col_idx;
  const int nblk = end - start;
  int rot = 0;
  uint64_t* walk_at = nullptr;
  if (kRouted && !split && p.walk != nullptr) {
    uint64_t* const tab = p.walk + xcc_id() * kWalkSlots;
    if (nblk > 1) {
      if (wave == 0) {
        const int r = walk_start(tab, lane, bh, p.kv_blocks, cidx, start, nblk);
        if (lane == 0) rot_lds = r;
      }
      dsa::lds_barrier();
      rot = __builtin_amdgcn_readfirstlane(rot_lds);
    }
    if (tid == 0) walk_at = tab + (wg / dsa::kNumXcd) % kWalkSlots;
  }
  auto walked = [&](int j) -> int { return start + (j + rot < nblk ? j + rot : j + rot - nblk); };

  if constexpr (kStats) {
    // Weight of stream position pos (mod two tiles) for kind r.
    const int bp = p.block_pad;
    for (int i = tid; i < kNarrowWRows * kNarrowCols; i += 128) {
      const int r = i / kNarrowCols, q2 = (i % kNarrowCols) % (2 * bp);
      const int par = q2 / bp, off = q2 % bp;
      float w = 0.f;
      if (r < 6 && r / 3 == par && off < p.stat_tile) {
        const int y = 2 * (off / p.tile_w) - (p.tile_h - 1);
        const int x = 2 * (off % p.tile_w) - (p.tile_w - 1);
        w = r % 3 == 0 ? 1.f : (float)(r % 3 == 1 ? y : x);
      }
      wtab[i] = (T)w;
    }
    dsa::lds_barrier();
  }
  const T* const wrow =
      wtab + (kStats ? (c16 < 3 ? c16 : c16 >= 4 && c16 < 7 ? c16 - 1 : 6) * kNarrowCols + 4 * q4
                     : 0);

  // Staging (issue_gather of bsa_fwd_kernel for two waves): lane (wave, q4, c16)
  // moves chunk c16 of stream rows r0 + 4 j, j = 0..7; rows j and j + 4 (V: j + 2)
  // share a swizzle, so four (two) offsets serve.
  const T* kbase = static_cast<const T*>(p.k) + b * p.k_sb + h * p.k_sh;
  const T* vbase = static_cast<const T*>(p.v) + b * p.v_sb + h * p.v_sh;
  const __amdgpu_buffer_rsrc_t k_rsrc = make_rsrc(
      kbase, (uint32_t)((int64_t)(p.kv_tokens - 1) * p.k_st * 2 + p.head_dim * 2));
  const __amdgpu_buffer_rsrc_t v_rsrc = make_rsrc(
      vbase, (uint32_t)((int64_t)(p.kv_tokens - 1) * p.v_st * 2 + p.head_dim * 2));
  const uint32_t ks = (uint32_t)(p.k_st * 2), vs = (uint32_t)(p.v_st * 2);
  // (V's dims past head_dim may hold anything: they only reach O dims that are
  // not stored.)
  const int r0 = wave * 32 + q4;
  uint32_t gk[4], gv[2];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int row = r0 + 4 * j;
    const int kc = k2_swz(row, c16);
    gk[j] = (uint32_t)row * ks + (uint32_t)(kc * 16) + dsa::dead_bits(kc, p.head_dim);
  }
#pragma unroll
  for (int j = 0; j < 2; ++j)
    gv[j] = (uint32_t)(r0 + 4 * j) * vs + (uint32_t)(v8_swz(r0 + 4 * j, c16) * 16);
  // Stages K or V of the 64-key chunk that starts o0 slots into stream block
  // kb0 and runs on into kb1.
  auto issue = [&](auto is_v, int kb0, int kb1, int o0) __attribute__((always_inline)) {
    constexpr bool kV = decltype(is_v)::value;
    const int base0 = max(kb0, 0) * p.block + o0;
    const int base1 = max(kb1, 0) * p.block + o0 - p.block_pad;
    const uint32_t st = kV ? vs : ks;
    const uint32_t at = (uint32_t)base0 * st, step = (uint32_t)(base1 - base0) * st;
    // Load j moves the four rows from wave 32 + 4 j, all in one block (blocks
    // take multiples of 8 rows), so everything but the lane's offset is uniform.
    const int first_rows = p.block_pad - o0 - wave * 32;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t row = at + (4 * j < first_rows ? 0u : step);
      if constexpr (kV)
        lds_load16(v_rsrc, lds_v + (wave * 8 + j) * 1024, gv[j & 1] + (row + (j >> 1) * (8 * vs)),
                   0);
      else
        lds_load16(k_rsrc, lds_k + (wave * 8 + j) * 1024, gk[j & 3] + (row + (j >> 2) * (16 * ks)),
                   0);
    }
  };
  const std::bool_constant<false> of_k;
  const std::bool_constant<true> of_v;
  auto gblock = [&](int j) -> int {
    const int at = walked(j < nblk ? j : nblk - 1);
    const int kb = kRouted ? cidx[at] : at;
    return (unsigned)kb < (unsigned)p.kv_blocks ? kb : -1;
  };

  // The walk of one wave over its kGroups row groups from row group grp0.
  auto run = [&](auto groups_c, int grp0) __attribute__((always_inline)) {
    constexpr int kGroups = decltype(groups_c)::value;
    x8 qf[kGroups][4];
    float thr[kGroups], m_run[kGroups], l_run[kGroups];
    bool row_ok[kGroups];
    dsa_f32x4 oacc[kGroups][8];
    dsa_f32x4 carry[kGroups];
    float kmax = 0.f;
    if (p.kv_norm != nullptr) {
      kmax = p.kv_norm[(int64_t)bh * kNormParts + lane];
#pragma unroll
      for (int m = 1; m < 64; m <<= 1) kmax = fmaxf(kmax, __shfl_xor(kmax, m));
    }
#pragma unroll
    for (int n = 0; n < kGroups; ++n) {
      const int local = 16 * (grp0 + n) + c16;
      const int tq = qb * p.block + local;
      row_ok[n] = local < p.block && tq < p.q_tokens;
      const T* qrow = static_cast<const T*>(p.q) + b * p.q_sb + h * p.q_sh +
                      (int64_t)min(tq, p.q_tokens - 1) * p.q_st;
      float qq = 0.f;
#pragma unroll
      for (int dc = 0; dc < 4; ++dc) {
#pragma unroll
        for (int e = 0; e < 8; ++e) qf[n][dc][e] = (T)0.0f;
        if (dc * 32 + q4 * 8 < p.head_dim)
          qf[n][dc] = *reinterpret_cast<const x8*>(qrow + dc * 32 + q4 * 8);
#pragma unroll
        for (int e = 0; e < 8; ++e) qq = fmaf((float)qf[n][dc][e], (float)qf[n][dc][e], qq);
      }
      // Key-norm bound of the row, as in bsa_fwd_kernel.
      qq += __shfl_xor(qq, 16);
      qq += __shfl_xor(qq, 32);
      thr[n] = p.kv_norm == nullptr
                   ? INFINITY
                   : fmaf(sqrtf(qq) * fabsf(p.scale_log2) * 1.0001f, kmax, -bound_log2<T>());
      m_run[n] = -INFINITY;
      l_run[n] = 0.f;
      carry[n] = dsa_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) oacc[n][dt] = dsa_f32x4{0.f, 0.f, 0.f, 0.f};
    }
    // Fragment addresses: K row 16 kg + c16, chunk 4 dc + q4; V rows 4 q4 + r
    // (+ 16, + 32 u), dims 16 dt + 4 c .. + 3, for lane c16 = 4 r + c.
    const int kfrag = c16 * kRowBytes + ((q4 ^ (c16 & 3)) << 4);
    const int vr = 4 * q4 + (c16 >> 2);
    const int vfrag = vr * kRowBytes + ((((c16 & 3) >> 1) ^ ((2 * (vr & 7)) & 1)) << 4) +
                      (c16 & 1) * 8;

    // While some row's reference is below its bound (thr), the row max is taken
    // and the accumulators may be rescaled.
    auto bounded = [&]() __attribute__((always_inline)) {
      bool under = false;
#pragma unroll
      for (int n = 0; n < kGroups; ++n) under = under || !(m_run[n] >= thr[n]);
      return !__any(under);
    };
    // One 32-key half (u) of the staged chunk: its scores, its probabilities, its
    // products with V.  The XORed fragment offsets are rebuilt each time (the
    // empty asm keeps the compiler from holding all twelve).
    dsa_f32x4 s[kGroups][2];
    x8 pf[kGroups];
    auto scores = [&](int u) __attribute__((always_inline)) {
      int kf = kfrag, ck = c16 >> 2;
      asm volatile("" : "+v"(kf), "+v"(ck));
#pragma unroll
      for (int n = 0; n < kGroups; ++n)
#pragma unroll
        for (int kg = 0; kg < 2; ++kg) s[n][kg] = dsa_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int dc = 0; dc < 4; ++dc)
#pragma unroll
        for (int kg = 0; kg < 2; ++kg) {
          // Chunk (4 dc + q4) ^ c16 of the row: 4 (dc ^ (c16 >> 2)) + (q4 ^ (c16 & 3)).
          const x8 a = *reinterpret_cast<const x8*>(
              lds_k + (2 * u + kg) * 16 * kRowBytes + kf + ((dc ^ ck) << 6));
#pragma unroll
          for (int n = 0; n < kGroups; ++n) s[n][kg] = E::mfma16(a, qf[n][dc], s[n][kg]);
        }
    };
    auto softmax = [&](int u, uint64_t invalid, auto move_c) __attribute__((always_inline)) {
      if (invalid != 0) {
        const uint32_t mine = (uint32_t)(invalid >> (32 * u)) >> (4 * q4);
#pragma unroll
        for (int kg = 0; kg < 2; ++kg)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (mine & (1u << (16 * kg + r)))
#pragma unroll
              for (int n = 0; n < kGroups; ++n) s[n][kg][r] = -INFINITY;
      }
      if constexpr (decltype(move_c)::value) {
#pragma unroll
        for (int n = 0; n < kGroups; ++n) {
          float mx = -INFINITY;
#pragma unroll
          for (int kg = 0; kg < 2; ++kg)
#pragma unroll
            for (int r = 0; r < 4; ++r) mx = fmaxf(mx, s[n][kg][r]);
          mx = fmaxf(mx, __shfl_xor(mx, 16));
          mx = dsa::pair32_max(mx);
          const float mx2 = mx * p.scale_log2;
          float m_new = mx2 > m_run[n] + kRescaleLog2 ? mx2 : m_run[n];
          if (thr[n] > m_new && thr[n] <= mx2 + raise_log2<T>()) m_new = thr[n];
          const bool up = m_new != m_run[n];
          if (__any(up)) {
            const float alpha = up ? __builtin_amdgcn_exp2f(m_run[n] - m_new) : 1.0f;
            m_run[n] = m_new;
            l_run[n] *= alpha;
#pragma unroll
            for (int dt = 0; dt < 8; ++dt) oacc[n][dt] *= alpha;
            if constexpr (kStats) carry[n] *= alpha;
          }
        }
      }
#pragma unroll
      for (int n = 0; n < kGroups; ++n) {
        const float m_use = m_run[n] == -INFINITY ? 0.f : m_run[n];
        float sum0 = 0.f, sum1 = 0.f;
#pragma unroll
        for (int kg = 0; kg < 2; ++kg)
#pragma unroll
          for (int r = 0; r < 4; r += 2) {
            const float p0 =
                __builtin_amdgcn_exp2f(fmaf(s[n][kg][r], p.scale_log2, -m_use));
            const float p1 =
                __builtin_amdgcn_exp2f(fmaf(s[n][kg][r + 1], p.scale_log2, -m_use));
            const dsa_f32x2 two = {p0, p1};
            const typename E::x2 pb = __builtin_convertvector(two, typename E::x2);
            sum0 += p0;
            sum1 += p1;
            pf[n][4 * kg + r] = pb[0];
            pf[n][4 * kg + r + 1] = pb[1];
          }
        l_run[n] += sum0 + sum1;
      }
    };
    auto products = [&](int u, int wbase) __attribute__((always_inline)) {
      int vf = vfrag, cv = vr & 7;
      asm volatile("" : "+v"(vf), "+v"(cv));
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) {
        // Chunk 2 dt + (c >> 1), XORed with 2 (row & 7).
        const unsigned char* at =
            lds_v + u * 32 * kRowBytes + vf + ((dt ^ cv) << 5);
        const x4 lo = lds_read_tr<T>(at);
        const x4 hi = lds_read_tr<T>(at + 16 * kRowBytes);
        const x8 a = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
        for (int n = 0; n < kGroups; ++n) oacc[n][dt] = E::mfma16(a, pf[n], oacc[n][dt]);
      }
      if constexpr (kStats) {
        const x4 lo = *reinterpret_cast<const x4*>(wrow + wbase + 32 * u);
        const x4 hi = *reinterpret_cast<const x4*>(wrow + wbase + 32 * u + 16);
        const x8 a = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
        for (int n = 0; n < kGroups; ++n) carry[n] = E::mfma16(a, pf[n], carry[n]);
      }
    };
    // Stream tile j has ended: its parity's lanes write their rows' entries.
    auto close = [&](int j) __attribute__((always_inline)) {
      if (q4 != (j & 1)) return;
      // Routed: CSR entry e at e block + row; dense: key tile e of head h at
      // (h tiles + e) q_tokens + token.
      const int64_t e = walked(j);
      const bool in = !kRouted || e < p.rs_entries;
      const int64_t at0 = kRouted ? e * p.block
                                  : ((int64_t)h * p.kv_blocks + e) * p.q_tokens + qb * p.block;
#pragma unroll
      for (int n = 0; n < kGroups; ++n) {
        const float mass = carry[n][0];
        if (row_ok[n] && in) {
          const int64_t at = at0 + 16 * (grp0 + n) + c16;
          p.rs_logm[at] = mass > 0.f ? __log2f(mass) + m_run[n] : -INFINITY;
          if (p.rs_mean != nullptr) {
            const float inv = mass > 0.f ? __builtin_amdgcn_rcpf(mass) : 0.f;
            const dsa_f32x2 mean = {carry[n][1] * inv * (1.f / (float)max(p.tile_h - 1, 1)),
                                    carry[n][2] * inv * (1.f / (float)max(p.tile_w - 1, 1))};
            const dsa_f16x2 hm = __builtin_convertvector(mean, dsa_f16x2);
            p.rs_mean[at] = __builtin_bit_cast(uint32_t, hm);
          }
        }
        carry[n] = dsa_f32x4{0.f, 0.f, 0.f, 0.f};
      }
    };

    const int bp = p.block_pad;
    const int total = (nblk - 1) * bp + p.block;  // slots up to the row's last key
    const int chunks = nblk > 0 ? (total + 63) >> 6 : 0;
    int j0 = 0, o0 = 0, w0 = 0;
    int kb0 = chunks > 0 ? gblock(0) : -1, kb1 = chunks > 0 ? gblock(1) : -1;
    if (chunks > 0) {
      issue(of_k, kb0, kb1, 0);
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
      __syncthreads();
    }
    // K of the chunk has landed and V's stage is free.  Each of the two loads
    // half a chunk ahead of its use: V under the first half's scores and
    // probabilities, the next K under the second half's probabilities and
    // products.
    int closing = -1;  // the tile that ended in the chunk before
    auto step = [&](int c, auto move_c) __attribute__((always_inline)) {
      int j1 = j0, o1 = o0 + 64;
      if (o1 >= bp) { o1 -= bp; ++j1; }
      const bool more = c + 1 < chunks;
      issue(of_v, kb0, kb1, o0);
      if constexpr (kStats) {
        if (closing >= 0) close(closing);
      }
      const int kb0n = more ? gblock(j1) : -1, kb1n = more ? gblock(j1 + 1) : -1;
      if (walk_at != nullptr && kb0 >= 0)
        __hip_atomic_store(walk_at, walk_entry(bh, kb0), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
      const int second = bp - o0;  // first slot of block kb1
      const int left = total - c * 64;
      uint64_t invalid = 0;
      if (left < 64) invalid = ~0ull << left;
      if (bp > p.block) {
        const int lo = max(p.block - o0, 0);
        const int hi = min(second, 64);
        if (lo < hi) invalid |= (hi == 64 ? ~0ull : (1ull << hi) - 1) & ~((1ull << lo) - 1);
      }
      if (kb0 < 0) invalid |= second >= 64 ? ~0ull : (1ull << second) - 1;
      if (kb1 < 0 && second < 64) invalid |= ~0ull << second;
      scores(0);
      softmax(0, invalid, move_c);
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): V
      __syncthreads();
      products(0, w0);
      scores(1);
      dsa::lds_barrier();  // both waves are done with K
      if (more) issue(of_k, kb0n, kb1n, o1);
      softmax(1, invalid, move_c);
      products(1, w0);
      // Block j0 ends in this chunk (the row's last block after the walk).
      closing = kStats && second <= 64 && j0 + 1 < nblk ? j0 : -1;
      dsa::lds_barrier<true>();  // the next K, and both waves are done with V
      j0 = j1;
      o0 = o1;
      kb0 = kb0n;
      kb1 = kb1n;
      w0 = w0 + 64 >= 2 * bp ? w0 + 64 - 2 * bp : w0 + 64;
    };
    // Two loops: the first moves the references (in practice one chunk), the
    // second needs no row max and no rescale.  With the rescale inside the one
    // loop the compiler keeps two copies of the accumulators across it, which
    // three row groups have no registers for (96 of 256 each).
    int c = 0;
    while (c < chunks) {
      step(c++, std::bool_constant<true>{});
      if (bounded()) break;
    }
    while (c < chunks) step(c++, std::bool_constant<false>{});
    if constexpr (kStats) {
      if (closing >= 0) close(closing);
      if (nblk > 0) close(nblk - 1);
    }

#pragma unroll
    for (int n = 0; n < kGroups; ++n) {
      float l_tot = l_run[n] + __shfl_xor(l_run[n], 16);
      l_tot += __shfl_xor(l_tot, 32);
      if (!row_ok[n]) continue;
      const int local = 16 * (grp0 + n) + c16;
      const int tq = qb * p.block + local;
      if (split) {
        float* po = p.part + (int64_t)(wg - p.split_from) * kPartFloats;
#pragma unroll
        for (int dt = 0; dt < 8; ++dt)
          *reinterpret_cast<dsa_f32x4*>(po + local * kHeadDim + dt * 16 + q4 * 4) = oacc[n][dt];
        if (q4 == 0) {
          po[128 * 128 + local] = m_run[n];
          po[128 * 128 + 128 + local] = l_tot;
        }
        continue;
      }
      const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
      T* orow = static_cast<T*>(p.o) + b * p.o_sb + h * p.o_sh + (int64_t)tq * p.o_st;
#pragma unroll
      for (int dt = 0; dt < 8; ++dt)
        if (dt * 16 + q4 * 4 < p.head_dim)
          *reinterpret_cast<x4*>(orow + dt * 16 + q4 * 4) =
              __builtin_convertvector(oacc[n][dt] * inv, x4);
      if (p.lse && q4 == 0)
        p.lse[((int64_t)b * p.heads + h) * p.q_tokens + tq] =
            l_tot > 0.f ? m_run[n] * 0.6931471805599453f + logf(l_tot) : -INFINITY;
    }
  };
  const std::integral_constant<int, 3> three;
  const std::integral_constant<int, 2> two;
  if (wave == 0 || p.block > 80) run(three, wave * kNarrowGroups);
  else run(two, kNarrowGroups);
}

// Whole blocks of 65..96 tokens, K and V of one head within 2 GiB.
inline bool use_narrow(int32_t block, int32_t kv_tokens, int64_t k_token_stride,
                       int64_t v_token_stride) {
  if (block <= kHalfKeys || block > 96 || kv_tokens % block != 0) return false;
  const int64_t stride = std::max(k_token_stride, v_token_stride);
  return ((int64_t)kv_tokens + 64) * stride * 2 + kRowBytes <= 0x7fffffff;
}

}  // namespace bsa
