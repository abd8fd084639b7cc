// Sampled block-mass estimate for gfx950 (bf16 or fp16 Q/K).
//
// Replaces `_sampled_block_mass` (attention_backends/flex.py:205-251): per
// block b of size_b = min(T - block * b, block) tokens, S samples at local
// offsets floor((2 s + 1) size_b / (2 S)); scores of every sampled query
// against every sampled key, computed by a matmul in the input type and
// multiplied by the scale in the input type (so rounded twice to bf16 or
// fp16), plus log(size_b / S) per key sample; an fp32 softmax over all
// sampled keys; mass[h, qb, kb] = mean over the query samples of block qb of
// the sum over the key samples of block kb.
//
// Any S in 1..block (<= 128) runs on a power-of-two sample stride SP >= S:
// sample slots s >= S of every block are padding, masked out of the
// softmax (keys) and out of the mean (queries).  SP <= 32: a 32-key sub-tile
// covers 32 / SP key blocks and a wave's 32 query lanes 32 / SP query blocks,
// so block sums are lane shuffles.  SP = 64 or 128: a key block spans one or
// two whole 64-key tiles and a query block two or four waves; each wave's
// block sum goes through LDS and the workgroup adds them in a fixed order
// after the next barrier (no atomics: the mass, the input of the bit-exact
// route selection, is run-to-run deterministic).
#include <algorithm>
#include <type_traits>

#include "bsa_tiles.h"

namespace {

constexpr int kHeadDim = 128;
constexpr float kLog2e = 1.4426950408889634f;

struct MassParams {
  const void* q;  // element type T of the kernel instance
  const void* k;
  float* mass;  // [heads, blocks, blocks]
  int64_t q_st, q_sh, k_st, k_sh;
  int32_t tokens, heads, blocks, block_size, samples;  // samples: S (real)
  int32_t head_dim;  // 8..256, a multiple of 8
  float scale;      // score scale (d^-1/2 unless given)
  float logw_full;  // log(block_size / S)
  float logw_last;  // log(size of the last block / S)
  // One-sweep kernel: row-block sums of the launch's workgroups (kGroupRows
  // floats per key block and workgroup), and the launch's first workgroup.
  float* part;
  int32_t first, row_tiles;  // row_tiles: 128-row workgroups per head
};

constexpr int kGroupRows = 128;  // sampled query rows per workgroup
// The one-sweep kernel moves a row's reference once a sub-tile adds more than
// this to it: a row sum of up to 2^20 sub-tiles then stays finite.
constexpr float kMoveSum = 1152921504606846976.0f;  // 2^60

// Key blocks per slot of row sums: whole 64-key tiles of any sample count, so
// that every sub-tile stores its sums without a bound check.
__host__ __device__ constexpr int64_t part_blocks(int64_t blocks) {
  return (blocks + 63) / 64 * 64;
}

// Token of padded sample slot j (block j / SP, sample j % SP) for S real
// samples per block (flex.py:224-231); a padding slot repeats the block's
// last sample (it is masked).
template <int SP>
__device__ __forceinline__ int sampled_token(int j, int tokens, int block_size, int S) {
  const int blk = j / SP;
  int s = j % SP;
  s = s < S ? s : S - 1;
  int size = tokens - blk * block_size;
  size = size < block_size ? size : block_size;
  int local = ((2 * s + 1) * size) / (2 * S);
  local = local < size - 1 ? local : size - 1;
  return blk * block_size + local;
}

// Rounding of two fp32 values to T (round to nearest even; fp16 overflows to
// inf as torch's fp16 matmul does), returned as fp32.
template <typename T>
__device__ __forceinline__ void round_pair(float a, float b, float& ra, float& rb) {
  const dsa_f32x2 two = {a, b};
  const typename dsa::Elem<T>::x2 h = __builtin_convertvector(two, typename dsa::Elem<T>::x2);
  if constexpr (std::is_same<T, __bf16>::value) {
    const uint32_t bits = __builtin_bit_cast(uint32_t, h);
    ra = __builtin_bit_cast(float, bits << 16);
    rb = __builtin_bit_cast(float, bits & 0xFFFF0000u);
  } else {
    ra = (float)h[0];
    rb = (float)h[1];
  }
}

// One workgroup (4 waves x 32 sampled queries) scans every sampled key; the
// sampled score matrix is never written to memory.  The per-score rounding and
// softmax work outweighs the 32x32x16 MFMAs several times (VALU 92% active in two
// sweeps; 56% in one, at three waves per SIMD), so scores are rounded in pairs,
// the log2(e) scale and log-weight fold into one fma, and only the tile holding
// the sequence's last sampled keys (every tile with padding slots) pays the
// per-score checks.
// Sampled key rows are gathered straight into LDS (buffer loads with a
// per-lane row offset), double-buffered one 64-key tile ahead.
//
// kOnce: one sweep.  Each query row keeps its scores' reference fixed (the
// largest score of its first sub-tile; fp32's exponent range absorbs what
// later scores exceed it by, and a row moves its reference, and rescales what
// it has written, only past kMoveSum), writes the sum of its terms per key
// block to p.part and, after the scan, reads them back and adds the rows of
// each query block over their row totals.  Writing and reading 4 bytes per
// (row, key block) costs far less than the second sweep's rounding, fma, exp
// and add per score: 57,600 tokens x 40 heads, 16 samples: 1.04 ms (0.8 with the
// fences below at workgroup scope) against 1.58 ms.  Without a workspace (kOnce = false; also SP >= 64, whose blocks span
// waves) sweep 1 builds each query's log-sum-exp and sweep 2 sums the normalised
// probabilities per (query block, key block).  Three waves per SIMD
// (168 VGPRs): with four, the longer instances spill.
//
// kHalves: head dims up to 128 * kHalves.  Head dims above 128 stage each
// tile as two 128-dim halves (dims 0..127, then 128..) and add both halves'
// products into one fp32 accumulator before the score is rounded, as one
// matmul over all dims does.
template <typename T, int SP, bool kPad, int kHalves, bool kOnce>
__global__ void __launch_bounds__(256, kHalves == 1 ? 3 : 2) sampled_mass_kernel(MassParams p) {
  typedef dsa::Elem<T> E;
  static_assert(!kOnce || SP <= 32, "one sweep: query blocks within a wave");
  constexpr int kTileKeys = 64;
  constexpr int kHalfBytes = kTileKeys * 256;  // one 128-dim half of a tile
  constexpr bool kWide = SP >= 64;
  constexpr int KBS = kWide ? 1 : 32 / SP;  // key blocks of one 32-key sub-tile
  __shared__ __attribute__((aligned(1024))) unsigned char st0[kHalfBytes * kHalves];
  __shared__ __attribute__((aligned(1024))) unsigned char st1[kHalfBytes * kHalves];
  __shared__ float wide_part[2][4];  // kWide: per-wave block sums, by block parity

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5;
  const int qi = lane & 31;
  const int group = p.first + (int)blockIdx.x;
  const int h = group / p.row_tiles;
  const int row0 = (group % p.row_tiles) * kGroupRows;
  const int S = kPad ? p.samples : SP;
  const int ns = p.blocks * SP;
  const int tiles = (ns + kTileKeys - 1) / kTileKeys;
  const int q0 = row0 + wave * 32;  // first sampled query of this wave

  int qs = q0 + qi;
  const bool q_real = qs < ns && (qs % SP) < S;
  qs = qs < ns ? qs : ns - 1;
  const T* qrow = static_cast<const T*>(p.q) + h * p.q_sh +
                  (int64_t)sampled_token<SP>(qs, p.tokens, p.block_size, S) * p.q_st;
  typename E::x8 qf[8 * kHalves];
#pragma unroll
  for (int hf = 0; hf < kHalves; ++hf)
    dsa::load_q_fragments(qrow + 128 * hf, g, p.head_dim - 128 * hf, qf + 8 * hf);

  // The head's K rows as one raw buffer (the host keeps them within 2^31 bytes).
  const T* kbase = static_cast<const T*>(p.k) + h * p.k_sh;
  __amdgpu_buffer_rsrc_t k_rsrc[kHalves];
#pragma unroll
  for (int hf = 0; hf < kHalves; ++hf)
    k_rsrc[hf] = dsa::make_rsrc(kbase + 128 * hf,
                                (uint32_t)(((int64_t)(p.tokens - 1) * p.k_st + kHeadDim) * 2));
  const int last_block = p.blocks - 1;
  // Tiles before this one hold only full, in-range key blocks.
  const int first_tail_tile = (last_block * SP) / kTileKeys;
  // This lane's 4 chunks of tile t: LDS slot idx = (wave * 4 + j) * 64 + lane
  // holds chunk (idx & 15) ^ (row & 15) of tile row idx >> 4.  In a tile of
  // full blocks the row's token is that of tile 0 plus 64 / SP blocks per tile
  // (SP <= 64), so its offset is a per-lane constant plus a uniform one: the
  // general form (a division and a 64-bit multiply per chunk) took a fifth of
  // the scan's VALU work.
  constexpr bool kTileBlocks = SP <= kTileKeys;
  const uint32_t tile_step =
      (uint32_t)((int64_t)(kTileKeys / SP) * p.block_size * p.k_st * 2);
  uint32_t chunk_at[4];
  if constexpr (kTileBlocks) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int idx = (wave * 4 + j) * 64 + lane;
      const int row = idx >> 4;
      const int c = (idx & 15) ^ (row & 15);
      // (Blocks past a one-block sequence: those tiles take the general form.)
      const int s = row % SP < S ? row % SP : S - 1;
      const int token = row / SP * p.block_size + ((2 * s + 1) * p.block_size) / (2 * S);
      chunk_at[j] = (uint32_t)(((int64_t)token * p.k_st + c * 8) * 2);
    }
  }
  auto issue = [&](int t, unsigned char* dst) __attribute__((always_inline)) {
    const int kt0 = t * kTileKeys;
    if (kTileBlocks && t < first_tail_tile) {
      const uint32_t at = (uint32_t)t * tile_step;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int idx = (wave * 4 + j) * 64 + lane;
        const int c = (idx & 15) ^ ((idx >> 4) & 15);
#pragma unroll
        for (int hf = 0; hf < kHalves; ++hf)
          dsa::lds_load16(k_rsrc[hf], dst + hf * kHalfBytes + (wave * 4 + j) * 1024,
                          (chunk_at[j] + at) | dsa::dead_bits(c, p.head_dim - 128 * hf), 0);
      }
      return;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int idx = (wave * 4 + j) * 64 + lane;
      const int row = idx >> 4;
      const int c = (idx & 15) ^ (row & 15);
      int key = kt0 + row;
      key = key < ns ? key : ns - 1;
      const uint32_t base = (uint32_t)(
          ((int64_t)sampled_token<SP>(key, p.tokens, p.block_size, S) * p.k_st + c * 8) * 2);
#pragma unroll
      for (int hf = 0; hf < kHalves; ++hf)
        dsa::lds_load16(k_rsrc[hf], dst + hf * kHalfBytes + (wave * 4 + j) * 1024,
                        base | dsa::dead_bits(c, p.head_dim - 128 * hf), 0);
    }
  };

  const float c_full = p.logw_full * kLog2e;
  const float c_last = p.logw_last * kLog2e;
  float m2 = -INFINITY, l2 = 0.f, lse2 = 0.f;
  float wide_acc = 0.f;  // kWide: this lane's sum over the current key block
  // kOnce: this wave's row sums [key block][32 rows].
  float* const part =
      kOnce ? p.part + ((int64_t)blockIdx.x * 4 + wave) * 32 * part_blocks(p.blocks) : nullptr;
  // Makes the wave's own stores to `part` visible to its other lanes' loads.  At
  // workgroup scope, as one L1 serves them: at agent scope every wave wrote back
  // and invalidated its XCD's L2, beside the kernels of other streams (a whole
  // route update at 57,600 tokens x 40 heads 1,179 us, with this 957).
  auto settle_part = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  };

  // One tile; kTail: it may hold keys of the last block, padding slots or
  // slots past the end.
  auto compute_tile = [&](const unsigned char* lds_k, int t, int sweep, auto tail_c)
      __attribute__((always_inline)) {
    constexpr bool kTail = decltype(tail_c)::value;
    const int kt0 = t * kTileKeys;
#pragma unroll
    for (int sub = 0; sub < kTileKeys / 32; ++sub) {
      dsa_f32x16 acc;
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
      for (int hf = 0; hf < kHalves; ++hf)
#pragma unroll
        for (int dc = 0; dc < 8; ++dc) {
          const int key = sub * 32 + qi;
          const int c = dc * 2 + g;
          const typename E::x8 a = *reinterpret_cast<const typename E::x8*>(
              lds_k + hf * kHalfBytes + key * 256 + ((c ^ (key & 15)) << 4));
          acc = E::mfma32(a, qf[8 * hf + dc], acc);
        }
      // Score = T(T(q.k) * scale), as a matmul and a scale multiply in T;
      // the softmax input in log2 units is score * log2e + c with
      // c = log(block size / S) * log2e.
      float sc[16];
      [[maybe_unused]] float cws[16];
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        float a0, a1;
        round_pair<T>(acc[r], acc[r + 1], a0, a1);
        round_pair<T>(a0 * p.scale, a1 * p.scale, sc[r], sc[r + 1]);
      }
      if constexpr (kTail) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int j = kt0 + sub * 32 + 8 * (r >> 2) + 4 * g + (r & 3);
          cws[r] = j / SP == last_block ? c_last : c_full;
          if (j >= ns || (kPad && (j % SP) >= S)) sc[r] = -INFINITY;
        }
      }
      auto cw = [&](int r) __attribute__((always_inline)) {
        if constexpr (kTail) return cws[r];
        else return c_full;
      };
      if constexpr (kOnce) {
        // Key-block sums of this lane: key 8 (r >> 2) + 4 g + (r & 3) of the
        // sub-tile.  Blocks of 8 or more samples hold keys of both lane
        // halves (sum i: block i), shorter ones of one half (sum i: the block
        // of accumulator i SP).
        constexpr int kOwn = SP >= 8 ? 32 / SP : 16 / SP;
        const int kb0 = (kt0 + sub * 32) / SP;
        // (The empty asm keeps the compiler from computing it ahead of the
        // branches that need it, on every sub-tile.)
        auto row_max = [&]() __attribute__((always_inline)) {
          float log2e = kLog2e;
          asm volatile("" : "+v"(log2e));
          float mx = -INFINITY;
#pragma unroll
          for (int r = 0; r < 16; ++r) mx = fmaxf(mx, fmaf(sc[r], log2e, cw(r)));
          return dsa::pair32_max(mx);
        };
        // The reference: the largest score of the row's first sub-tile that
        // has one above -inf (0 until then, when every term is 0).
        if (__any(m2 == -INFINITY)) {
          const float mx = row_max();
          if (m2 == -INFINITY) m2 = mx;
        }
        float pk[kOwn];
        auto terms = [&]() __attribute__((always_inline)) {
          const float mref = m2 == -INFINITY ? 0.f : m2;
#pragma unroll
          for (int i = 0; i < kOwn; ++i) pk[i] = 0.f;
#pragma unroll
          for (int r = 0; r < 16; ++r)
            pk[(SP >= 8 ? 8 * (r >> 2) : r) / SP] +=
                __builtin_amdgcn_exp2f(fmaf(sc[r], kLog2e, cw(r) - mref));
          float sum = 0.f;
#pragma unroll
          for (int i = 0; i < kOwn; ++i) sum += pk[i];
          return sum;
        };
        float sum = terms();
        if (__any(!(sum <= kMoveSum))) {
          // Rows whose terms have outgrown their reference move it to their
          // largest score; both lanes of a row alike.  (A NaN row never does, and
          // must not have the wave rewrite its sums on every sub-tile.)
          const float mx = row_max();
          const bool up = mx > m2 && dsa::pair32_max(sum) > kMoveSum;
          if (__any(up)) {
            const float alpha = up ? __builtin_amdgcn_exp2f(m2 - mx) : 1.f;
            if (up) m2 = mx;
            l2 *= alpha;
            settle_part();
            for (int kb = g; kb < kb0; kb += 2) part[kb * 32 + qi] *= alpha;
            settle_part();
            sum = terms();
          }
        }
        l2 += sum;
        if constexpr (SP >= 8 && kOwn > 1) {
          // Lane half g takes block i + g: the sum over both halves' keys.
#pragma unroll
          for (int i = 0; i < kOwn; i += 2) {
            const auto both = __builtin_amdgcn_permlane32_swap(
                __float_as_uint(pk[i]), __float_as_uint(pk[i + 1]), false, false);
            part[(kb0 + i + g) * 32 + qi] = __uint_as_float(both[0]) + __uint_as_float(both[1]);
          }
        } else if constexpr (SP >= 8) {
          const float total = dsa::pair32_sum(pk[0]);
          if (g == 0) part[kb0 * 32 + qi] = total;
        } else {
#pragma unroll
          for (int i = 0; i < kOwn; ++i) {
            const int r = i * SP;
            part[(kb0 + (8 * (r >> 2) + 4 * g + (r & 3)) / SP) * 32 + qi] = pk[i];
          }
        }
      } else if (sweep == 0) {
        // Running max of x = score * log2e + c (log2e > 0: c_last differs
        // from c_full only in the tail).
        float mx = m2;
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, fmaf(sc[r], kLog2e, cw(r)));
        // While every key this lane has seen is masked (mx = -inf, as for
        // the lanes past the last sampled key when blocks * S <= 4), the
        // terms and the rescale take a finite reference and are exactly
        // zero, where -inf - (-inf) would make them NaN.
        const float mref = mx == -INFINITY ? 0.f : mx;
        float sum = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r)
          sum += __builtin_amdgcn_exp2f(fmaf(sc[r], kLog2e, cw(r) - mref));
        l2 = l2 * __builtin_amdgcn_exp2f(m2 - mref) + sum;
        m2 = mx;
      } else if constexpr (kWide) {
        float sum = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r)
          sum += __builtin_amdgcn_exp2f(fmaf(sc[r], kLog2e, cw(r) - lse2));
        wide_acc += q_real ? sum : 0.f;
      } else {
        float pk[KBS];
#pragma unroll
        for (int b = 0; b < KBS; ++b) pk[b] = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int local = 8 * (r >> 2) + 4 * g + (r & 3);
          pk[local / SP] += __builtin_amdgcn_exp2f(fmaf(sc[r], kLog2e, cw(r) - lse2));
        }
        // Sum over the SP query lanes of each query block (padding lanes
        // add zero) and both halves.
#pragma unroll
        for (int b = 0; b < KBS; ++b) {
          if (kPad && !q_real) pk[b] = 0.f;
#pragma unroll
          for (int m = 1; m < SP; m <<= 1) pk[b] += __shfl_xor(pk[b], m);
          pk[b] += __shfl_xor(pk[b], 32);
        }
        if (g == 0 && (qi % SP) == 0) {
          const int qs_first = q0 + qi;
          if (qs_first < ns) {
            const int qb = qs_first / SP;
            float* out = p.mass + ((int64_t)h * p.blocks + qb) * p.blocks;
#pragma unroll
            for (int b = 0; b < KBS; ++b) {
              const int kb = (kt0 + sub * 32) / SP + b;
              if (kb < p.blocks) out[kb] = pk[b] / (float)S;
            }
          }
        }
      }
    }
    if constexpr (kWide) {
      // Key block (kt0 / SP) complete after this tile: publish this wave's sum.
      if (sweep == 1 && ((t + 1) * kTileKeys) % SP == 0) {
        const float total = dsa::wave_total(wide_acc);
        if (lane == 0) wide_part[(kt0 / SP) & 1][wave] = total;
        wide_acc = 0.f;
      }
    }
  };
  auto compute = [&](const unsigned char* lds_k, int t, int sweep) __attribute__((always_inline)) {
    if (kPad || t >= first_tail_tile)
      compute_tile(lds_k, t, sweep, std::bool_constant<true>{});
    else
      compute_tile(lds_k, t, sweep, std::bool_constant<false>{});
  };

  // kWide: writes the mass of key block kb from the wave sums published for
  // it (after a barrier); the waves of one query block are added in order.
  auto flush_wide = [&](int kb) __attribute__((always_inline)) {
    if constexpr (kWide) {
      constexpr int kWavesPerBlock = SP / 32;
      if (tid < 4 / kWavesPerBlock) {
        const int qb = row0 / SP + tid;
        if (qb < p.blocks && kb < p.blocks) {
          float total = 0.f;
#pragma unroll
          for (int w = 0; w < kWavesPerBlock; ++w) total += wide_part[kb & 1][tid * kWavesPerBlock + w];
          p.mass[((int64_t)h * p.blocks + qb) * p.blocks + kb] = total / (float)S;
        }
      }
    }
  };

  // Step: wait for the current tile (and every older memory and LDS
  // operation), barrier (all waves' loads landed, every wave done with the
  // other stage, wave sums published), prefetch the next tile into the other
  // stage, write the key block finished by the previous tile (kWide), compute
  // the current one.
  auto step = [&](int t, int sweep, int next_t, const unsigned char* cur,
                  unsigned char* nxt) __attribute__((always_inline)) {
    // kOnce: the row sums of the previous tile, stored after the current
    // tile's loads were issued, may still be on their way.
    constexpr int kStores = !kOnce ? 0 : 2 * (SP >= 8 ? (SP == 32 ? 1 : 16 / SP) : 16 / SP);
    if (kOnce && t > 0)
      __builtin_amdgcn_s_waitcnt(0x0F70 | (kStores & 15) | ((kStores >> 4) << 14));  // vmcnt
    else
      __builtin_amdgcn_s_waitcnt(kWide ? 0x0070 : 0x0F70);  // vmcnt(0) [lgkmcnt(0)]
    __syncthreads();
    if (next_t >= 0) issue(next_t, nxt);
    if (kWide && sweep == 1 && t > 0 && (t * kTileKeys) % SP == 0) flush_wide(t * kTileKeys / SP - 1);
    compute(cur, t, sweep);
  };

  for (int sweep = 0; sweep < (kOnce ? 1 : 2); ++sweep) {
    issue(0, st0);
    for (int t = 0; t < tiles; t += 2) {
      step(t, sweep, t + 1 < tiles ? t + 1 : -1, st0, st1);
      if (t + 1 >= tiles) break;
      step(t + 1, sweep, t + 2 < tiles ? t + 2 : -1, st1, st0);
    }
    if (!kOnce && sweep == 0) {  // each query's log-sum-exp (log2 units)
      // Lanes l and l ^ 32 hold the two halves of one query's keys; both get
      // the same total (the pair's two terms in one fixed order, so a
      // contracted fma rounds alike in both lanes).
      const auto ms = __builtin_amdgcn_permlane32_swap(__float_as_uint(m2), __float_as_uint(m2),
                                                       false, false);
      const auto ls = __builtin_amdgcn_permlane32_swap(__float_as_uint(l2), __float_as_uint(l2),
                                                       false, false);
      const float ma = __uint_as_float(ms[0]), mb = __uint_as_float(ms[1]);
      const float mx = fmaxf(ma, mb);
      const float tot = __uint_as_float(ls[0]) * __builtin_amdgcn_exp2f(ma - mx) +
                        __uint_as_float(ls[1]) * __builtin_amdgcn_exp2f(mb - mx);
      lse2 = mx + __builtin_log2f(tot);
      __syncthreads();  // every wave done with st0/st1 before sweep 2 refills st0
    }
  }
  if constexpr (kWide) {  // the last key block
    dsa::lds_barrier();
    flush_wide(p.blocks - 1);
  }
  if constexpr (kOnce) {
    // mass[qb][kb] = sum over the rows of qb of part[kb][row] / total[row] / S.
    // Eight lanes read one key block's 32 rows (four each), so a wave reads
    // 1 KB of consecutive part per step.
    settle_part();
    const float total = dsa::pair32_sum(l2);
    const float weight = q_real ? 1.f / total : 0.f;
    const int sub_rows = lane & 7;
    float w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = __shfl(weight, 4 * sub_rows + i);
    constexpr int kLanes = SP >= 4 ? SP / 4 : 1;  // lanes per query block
    constexpr int kVals = SP >= 4 ? 1 : 4 / SP;   // query blocks per lane
    constexpr int kAhead = 4;                     // loads in flight per lane
    for (int k0 = lane >> 3; k0 - (lane >> 3) < p.blocks; k0 += 8 * kAhead) {
      dsa_f32x4 x[kAhead];
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        const int kb = k0 + 8 * u;
        x[u] = kb < p.blocks
                   ? *reinterpret_cast<const dsa_f32x4*>(part + kb * 32 + 4 * sub_rows)
                   : dsa_f32x4{0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        const int kb = k0 + 8 * u;
        float val[kVals];
#pragma unroll
        for (int v = 0; v < kVals; ++v) {
          val[v] = 0.f;
#pragma unroll
          for (int i = 0; i < 4 / kVals; ++i)
            val[v] = fmaf(x[u][v * (4 / kVals) + i], w[v * (4 / kVals) + i], val[v]);
        }
#pragma unroll
        for (int m = 1; m < kLanes; m <<= 1) val[0] += __shfl_xor(val[0], m);
        if (kb < p.blocks && sub_rows % kLanes == 0) {
#pragma unroll
          for (int v = 0; v < kVals; ++v) {
            const int qb = q0 / SP + sub_rows / kLanes * kVals + v;
            if (qb < p.blocks)
              p.mass[((int64_t)h * p.blocks + qb) * p.blocks + kb] = val[v] / (float)S;
          }
        }
      }
    }
  }
}

bool aligned16(const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15u) == 0; }

template <typename T, int kHalves, bool kOnce>
void launch_mass(const MassParams& p, int sp, bool pad, int groups, hipStream_t stream) {
#define DSA_MASS(SPV, PADV)                                                           \
  hipLaunchKernelGGL((sampled_mass_kernel<T, SPV, PADV, kHalves, kOnce>),             \
                     dim3((unsigned)groups), dim3(256), 0, stream, p)
  if (!pad) {
    switch (sp) {
      case 1: DSA_MASS(1, false); break;
      case 2: DSA_MASS(2, false); break;
      case 4: DSA_MASS(4, false); break;
      case 8: DSA_MASS(8, false); break;
      case 16: DSA_MASS(16, false); break;
      default: DSA_MASS(32, false); break;
    }
  } else {
    switch (sp) {
      case 4: DSA_MASS(4, true); break;
      case 8: DSA_MASS(8, true); break;
      case 16: DSA_MASS(16, true); break;
      case 32: DSA_MASS(32, true); break;
      case 64: if constexpr (!kOnce) DSA_MASS(64, true); break;
      default: if constexpr (!kOnce) DSA_MASS(128, true); break;
    }
  }
#undef DSA_MASS
}

template <typename T>
void launch_mass(const MassParams& p, int sp, bool pad, bool once, int groups,
                 hipStream_t stream) {
  if (p.head_dim > kHeadDim)
    once ? launch_mass<T, 2, true>(p, sp, pad, groups, stream)
         : launch_mass<T, 2, false>(p, sp, pad, groups, stream);
  else
    once ? launch_mass<T, 1, true>(p, sp, pad, groups, stream)
         : launch_mass<T, 1, false>(p, sp, pad, groups, stream);
}

// Power-of-two sample stride of S samples per block.
int sample_stride(int32_t samples) {
  int sp = 1;
  while (sp < samples) sp <<= 1;
  return sp;
}

// One-sweep workspace: a slot of row sums per workgroup, for every workgroup or
// as many chip-fulls as kSlotBytes holds, and at least one; a call of more runs in
// launches of whole chip-fulls over the same slots.  A CU holds three of the
// kernel's workgroups (four waves each, three per SIMD), two above head dim 128.
// (57,600 tokens x 40 heads, 16 samples, 2,280 workgroups: 598 MB in one launch,
// 1,042 us; in launches of two chip-fulls 1,056 us, of one 1,060.  Workgroups that
// stay and take one group after the other are no faster than launches of one.)
constexpr int64_t kChipGroups = 3 * 256, kChipGroupsWide = 2 * 256;
constexpr int64_t kSlotBytes = (int64_t)1 << 30;

int64_t slot_bytes(int64_t blocks) {
  return part_blocks(blocks) * kGroupRows * (int64_t)sizeof(float);
}

}  // namespace

extern "C" size_t dsa_sampled_mass_workspace_bytes(int32_t tokens, int32_t heads,
                                                   int32_t block_size, int32_t samples) {
  if (tokens <= 0 || heads <= 0 || block_size <= 0 || block_size > 128 || samples <= 0 ||
      samples > block_size)
    return 0;
  const int sp = sample_stride(samples);
  if (sp > 32) return 0;
  const int64_t blocks = ((int64_t)tokens + block_size - 1) / block_size;
  const int64_t groups = (blocks * sp + kGroupRows - 1) / kGroupRows * heads;
  const int64_t chips = std::max<int64_t>(1, kSlotBytes / (kChipGroups * slot_bytes(blocks)));
  return (size_t)(std::min(groups, chips * kChipGroups) * slot_bytes(blocks));
}

extern "C" int dsa_sampled_mass(const void* q, const void* k, int32_t dtype,
                                const int64_t* strides, int32_t tokens, int32_t heads,
                                int32_t head_dim, int32_t block_size, int32_t samples,
                                float scale, float* mass, hipStream_t stream) {
  return dsa_sampled_mass_ws(q, k, dtype, strides, tokens, heads, head_dim, block_size, samples,
                             scale, mass, nullptr, 0, stream);
}

extern "C" int dsa_sampled_mass_ws(const void* q, const void* k, int32_t dtype,
                                   const int64_t* strides, int32_t tokens, int32_t heads,
                                   int32_t head_dim, int32_t block_size, int32_t samples,
                                   float scale, float* mass, void* workspace,
                                   size_t workspace_bytes, hipStream_t stream) {
  dsa::clear_error();
  if (!q || !k || !mass || !strides)
    return dsa::set_error(DSA_EINVAL, "dsa_sampled_mass: null pointer");
  if (dtype != DSA_BF16 && dtype != DSA_F16)
    return dsa::set_error(DSA_EUNSUPPORTED, "dsa_sampled_mass: dtype %d unsupported (bf16 or fp16)",
                          dtype);
  if (tokens <= 0 || heads <= 0 || block_size <= 0)
    return dsa::set_error(DSA_EINVAL, "dsa_sampled_mass: tokens/heads/block must be positive");
  if (head_dim <= 0 || head_dim > 2 * kHeadDim || head_dim % 8 != 0)
    return dsa::set_error(DSA_EUNSUPPORTED,
                          "dsa_sampled_mass: head_dim %d unsupported (a multiple of 8 up to 256)",
                          head_dim);
  if (block_size > 128)
    return dsa::set_error(DSA_EUNSUPPORTED, "dsa_sampled_mass: block_size %d unsupported (<= 128)",
                          block_size);
  if (samples <= 0 || samples > block_size)
    return dsa::set_error(DSA_EINVAL, "route_samples must be in [1, block_size]");
  if (!(scale > 0.f)) return dsa::set_error(DSA_EINVAL, "dsa_sampled_mass: scale must be > 0");
  if (!aligned16(q) || !aligned16(k))
    return dsa::set_error(DSA_EINVAL, "dsa_sampled_mass: q/k must be 16-byte aligned");
  for (int i = 0; i < 4; ++i)
    if (strides[i] % 8 != 0 || strides[i] < 0)
      return dsa::set_error(DSA_EINVAL,
                            "dsa_sampled_mass: stride %d not a non-negative multiple of 8", i);
  if (((int64_t)(tokens - 1) * strides[2] + kHeadDim) * 2 > 0x7fffffff)
    return dsa::set_error(DSA_EUNSUPPORTED,
                          "dsa_sampled_mass: one head's K rows must span < 2 GiB");
  if (workspace_bytes > 0 && (!workspace || !aligned16(workspace)))
    return dsa::set_error(DSA_EINVAL, "dsa_sampled_mass: workspace must be 16-byte aligned");
  const int sp = sample_stride(samples);
  MassParams p;
  p.q = q;
  p.k = k;
  p.mass = mass;
  p.q_st = strides[0]; p.q_sh = strides[1]; p.k_st = strides[2]; p.k_sh = strides[3];
  p.tokens = tokens;
  p.heads = heads;
  p.block_size = block_size;
  p.samples = samples;
  p.head_dim = head_dim;
  p.blocks = (tokens + block_size - 1) / block_size;
  if ((int64_t)p.blocks * sp > 0x3fffffff)
    return dsa::set_error(DSA_EUNSUPPORTED, "dsa_sampled_mass: too many sampled tokens");
  p.scale = scale;
  // fp32 log of an fp32 quotient, as torch's (sizes.float() / samples).log().
  const int last = tokens - (p.blocks - 1) * block_size;
  p.logw_full = logf((float)block_size / (float)samples);
  p.logw_last = logf((float)last / (float)samples);
  const int ns = p.blocks * sp;
  p.row_tiles = (ns + kGroupRows - 1) / kGroupRows;
  const int64_t groups = (int64_t)p.row_tiles * heads;
  if (groups > 0x7fffffff)
    return dsa::set_error(DSA_EINVAL, "dsa_sampled_mass: grid too large");
  // Padded instances for sample counts that are not a power of two, and for
  // 64 and 128 samples (key and query blocks wider than a sub-tile or wave).
  const bool pad = sp != samples || sp > 32;
  // One sweep where the workspace holds a chip-full of row sums, or all.
  const int64_t slots = std::min<int64_t>(
      groups, workspace ? (int64_t)workspace_bytes / slot_bytes(p.blocks) : 0);
  const bool once = sp <= 32 && slots >= std::min(groups, kChipGroups);
  p.part = once ? static_cast<float*>(workspace) : nullptr;
  const int64_t chip = head_dim > kHeadDim ? kChipGroupsWide : kChipGroups;
  const int64_t step = !once || slots == groups ? groups : slots / chip * chip;
  for (int64_t first = 0; first < groups; first += step) {
    p.first = (int32_t)first;
    const int n = (int)std::min(step, groups - first);
    if (dtype == DSA_F16) launch_mass<_Float16>(p, sp, pad, once, n, stream);
    else launch_mass<__bf16>(p, sp, pad, once, n, stream);
  }
  return dsa::check_launch("dsa_sampled_mass");
}
