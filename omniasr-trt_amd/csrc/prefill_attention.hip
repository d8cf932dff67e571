// Causal attention over whole contexts for gfx950: the prefill's
//     F.scaled_dot_product_attention(q, k, v, is_causal=True)
// (src/omniasr_trt/decode.py:163-164) over the cache rows ``kernels.rope_kv`` has just written.  Query p of context
// b attends to keys [0, p] of its cache row; fp32 accumulation, bf16 in and out, head_dim 128, 256 or 512.
#include <math.h>

#include <algorithm>

#include "attn_tiles.h"
#include "common.h"

namespace omni {

// Query p of context b attends to keys [0, p] of its cache row; one workgroup per (query block, head, context), the
// longest blocks first; every kernel keeps a lazy softmax reference and masks only the tiles on the diagonal.
typedef short v4i16_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4i16_t lds_v4i16;
typedef __attribute__((address_space(3))) const char lds_char;

struct PrefillArgs {
  const uint16_t* q;    // [B * width, H, D] bf16
  const uint16_t* k;    // cache rows: element strides s_row / s_head, key rows contiguous (D elements)
  const uint16_t* v;
  const int64_t* slots;  // [B] cache row of each context
  int64_t s_row, s_head, cache_rows;
  int width, H;
  float scale_log2;
  uint16_t* out;  // [B * width, H, D] bf16
  int units8, group;  // head dim 512 in chains: heads x contexts / 8, and how many of them are listed together
};

// Workgroup -> (query block j counted from the longest, head h, context b).  The dispatcher hands consecutive
// workgroups to the 8 XCDs in turn; when heads x contexts is a multiple of 8, XCD x gets units (head, context)
// x, x + 8, ... one after another, all query blocks of a unit together (longest first), so each unit's K / V rows
// are brought into one XCD's L2 rather than into all eight.  Only speed depends on the dispatch order.
constexpr bool kPfXcd = true;
struct PfBlock {
  int j, h, b;
};
__device__ __forceinline__ PfBlock pf_block(int nqb, int H, int B) {
  if (!kPfXcd || (H * B) % 8 != 0) return PfBlock{(int)blockIdx.x, (int)blockIdx.y, (int)blockIdx.z};
  const int L = (int)blockIdx.x + nqb * ((int)blockIdx.y + H * (int)blockIdx.z);
  const int x = L % 8, k = L / 8;
  const int unit = (k / nqb) * 8 + x;
  return PfBlock{k % nqb, unit % H, unit / H};
}

// Head dim 256: one workgroup of kPwWaves waves per (query block, head, context).  The block's
// NG = kPwSub * M groups of 16 queries (M = kPwWaves / (D/128)): group gi holds queries qb + 16 gi .. + 15.  Wave w
// holds the 128-dimension slice sl = w % (D/128) of q and O for the groups m + M u (m = w / (D/128), u < kPwSub).
// Per 32-key tile (K and V through LDS once for all waves):
//   1. each wave writes its slice's partial scores S^T = K_sl Q_sl^T of its groups to LDS;  barrier;
//   2. wave w runs the softmax of groups w, w + kPwWaves, ...: adds the D/128 partials in slice order, moves the
//      lazy reference max when needed, and publishes the group's P operand (bf16) and, when the reference max
//      moved, its 16 rescale factors;  barrier;
//   3. each wave rescales its O_sl of a group when told to and adds P V_sl.
// So each group's softmax runs once, not once per slice.  K has one LDS buffer (the next tile's goes in after
// barrier 1, when every wave has read this one), V two (the next tile's goes in during step 3 of this one, into the
// buffer the previous tile's P V read before barrier 1).
constexpr int kPwWaves = 8;
constexpr int kPwSub = 3;  // 16-query groups per wave

__global__ __launch_bounds__(64 * kPwWaves) __attribute__((amdgpu_waves_per_eu(2, 2))) void prefill_attn_wide_kernel(
    PrefillArgs a) {
  constexpr int D = 256;
  constexpr int NSL = D / 128, M = kPwWaves / NSL, NG = kPwSub * M, QW = 16 * NG;
  constexpr int OWN = (NG + kPwWaves - 1) / kPwWaves;  // groups whose softmax one wave runs, at most
  constexpr int kRowB = D * 2 + 16;                     // LDS bytes per key row, padded against bank conflicts
  constexpr int kRowChunks = D / 8;                     // 16-byte chunks per key row
  constexpr int kChunks = 32 * kRowChunks / (64 * kPwWaves);  // chunks of K (or of V) per thread per tile
  static_assert(NSL * M == kPwWaves && kChunks * 64 * kPwWaves == 32 * kRowChunks, "whole slices and chunks");
  __shared__ __attribute__((aligned(16))) char kl[32 * kRowB];     // K: 32 key rows
  __shared__ __attribute__((aligned(16))) char vl[2][32 * kRowB];  // V: two tiles
  __shared__ f32x4_t part[NG][NSL][2][64];  // partial scores: [group][slice][block mb][lane]
  __shared__ u32x4_t pex[NG][64];           // P operand of each group: [group][lane]
  __shared__ float alx[NG][16];             // rescale factor of each query of a group (when rflag)
  __shared__ int rflag[NG];                 // the group's reference max moved on this tile
  __shared__ float lsum[NG][16];            // probability sum of each query, at the end
  const int nqb = (a.width + QW - 1) / QW;
  const PfBlock blk = pf_block(nqb, a.H, (int)gridDim.z);
  const int qb = (nqb - 1 - blk.j) * QW;  // the longest blocks first
  const int h = blk.h, b = blk.b;
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int sl = w % NSL, m = w / NSL;
  const int64_t slot = clamp64(a.slots[b], 0, a.cache_rows - 1);
  const uint16_t* kbase = a.k + slot * a.s_row + h * a.s_head;
  const uint16_t* vbase = a.v + slot * a.s_row + h * a.s_head;
  const int kend = min(qb + QW, a.width);
  const int nt = (kend + 31) / 32;

  // Global -> LDS through one set of staging registers: thread tid moves 16-byte chunks tid, tid + 64 kPwWaves, ...
  // of a tile's K or V rows.  Rows past the context read its last key (finite: masked by the causal limit).
  u32x4_t stage[kChunks];
  auto fetch = [&](int t, const uint16_t* base) {
#pragma unroll
    for (int e = 0; e < kChunks; ++e) {
      const int ci = tid + e * 64 * kPwWaves, r = ci / kRowChunks, col = ci % kRowChunks;
      const int key = min(t * 32 + r, a.width - 1);
      stage[e] = *reinterpret_cast<const u32x4_t*>(base + (int64_t)key * D + col * 8);
    }
  };
  auto put = [&](char* dst) {
#pragma unroll
    for (int e = 0; e < kChunks; ++e) {
      const int ci = tid + e * 64 * kPwWaves, r = ci / kRowChunks, col = ci % kRowChunks;
      *reinterpret_cast<u32x4_t*>(dst + r * kRowB + col * 16) = stage[e];
    }
  };
  // Whether group gi sees the tile starting at key0: a live group whose last query reaches the tile's first key.
  auto sees = [&](int gi, int key0) { return qb + 16 * gi < a.width && key0 <= qb + 16 * gi + 15; };

  u32x4_t qop[kPwSub][4];  // lane (c, g): q[qb + 16 gi + c][128 sl + 32 s2 + 8g .. +7] (0 past the end)
  f32x4_t o[kPwSub][8];    // output column c of block e: dimension 128 sl + 16 e + c
#pragma unroll
  for (int u = 0; u < kPwSub; ++u) {
    const int row = qb + 16 * (m + M * u) + c;
    const bool live = row < a.width;
    const uint16_t* qrow = a.q + ((int64_t)(b * a.width + (live ? row : 0)) * a.H + h) * D + 128 * sl + g * 8;
#pragma unroll
    for (int s2 = 0; s2 < 4; ++s2)
      qop[u][s2] = live ? *reinterpret_cast<const u32x4_t*>(qrow + s2 * 32) : u32x4_t{0u, 0u, 0u, 0u};
#pragma unroll
    for (int e = 0; e < 8; ++e) o[u][e] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  SoftmaxState st[OWN];  // the softmax state of groups w + kPwWaves r
#pragma unroll
  for (int r = 0; r < OWN; ++r) st[r] = SoftmaxState{-INFINITY, -INFINITY, 0.f};

  fetch(0, kbase);
  put(kl);
  fetch(0, vbase);
  put(vl[0]);
  if (nt > 1) fetch(1, kbase);
  lds_barrier();
  for (int t = 0; t < nt; ++t) {
    const int key0 = t * 32;
    // 1. partial scores of this wave's groups over its slice
    {
      u32x4_t kf[2][4];
#pragma unroll
      for (int mb = 0; mb < 2; ++mb) {
        const int rk = 8 * (c >> 2) + 4 * mb + (c & 3);
#pragma unroll
        for (int s2 = 0; s2 < 4; ++s2)
          kf[mb][s2] = *reinterpret_cast<const u32x4_t*>(&kl[rk * kRowB + 256 * sl + g * 16 + s2 * 64]);
      }
#pragma unroll
      for (int u = 0; u < kPwSub; ++u) {
        const int gi = m + M * u;
        if (!sees(gi, key0)) continue;
#pragma unroll
        for (int mb = 0; mb < 2; ++mb) {
          f32x4_t acc = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int s2 = 0; s2 < 4; ++s2)
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, kf[mb][s2]),
                                                          __builtin_bit_cast(bf16x8_t, qop[u][s2]), acc, 0, 0, 0);
          part[gi][sl][mb][lane] = acc;
        }
      }
    }
    lds_barrier();
    if (t + 1 < nt) {
      put(kl);             // every wave has read this tile's K
      fetch(t + 1, vbase);  // the next V, in flight during steps 2 and 3
    }
    // 2. the softmax of this wave's own groups
#pragma unroll
    for (int r = 0; r < OWN; ++r) {
      const int gi = w + kPwWaves * r;
      if (gi >= NG || !sees(gi, key0)) continue;
      const int q0 = qb + 16 * gi;
      f32x4_t sum[2];
#pragma unroll
      for (int mb = 0; mb < 2; ++mb) {
        sum[mb] = part[gi][0][mb][lane];
#pragma unroll
        for (int s3 = 1; s3 < NSL; ++s3) sum[mb] += part[gi][s3][mb][lane];
      }
      float sv[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) sv[j] = sum[j >> 2][j & 3];
      const int lim = q0 + c + 1;
      if (!(key0 + 31 <= q0)) {  // not every query of the group sees the whole tile
#pragma unroll
        for (int j = 0; j < 8; ++j) sv[j] = key0 + 8 * g + j < lim ? sv[j] : -INFINITY;
      }
      bool over = false;
#pragma unroll
      for (int j = 0; j < 8; ++j) over |= sv[j] > st[r].thr;
      const bool moved = __any(over);
      if (moved) {
        float mx = sv[0];
#pragma unroll
        for (int j = 1; j < 8; ++j) mx = fmaxf(mx, sv[j]);
        mx = fmaxf(mx, __shfl_xor(mx, 16, kWave));
        mx = fmaxf(mx, __shfl_xor(mx, 32, kWave));
        const float m_new = fmaxf(st[r].m_ref, mx * a.scale_log2);
        const float alpha = __builtin_amdgcn_exp2f(st[r].m_ref - (m_new == -INFINITY ? 0.f : m_new));  // -inf: 0
        st[r].l_run *= alpha;
        if (g == 0) alx[gi][c] = alpha;
        st[r].m_ref = m_new;
        st[r].thr = m_new == -INFINITY ? -INFINITY : (m_new + kLazyLog2) / a.scale_log2;
      }
      if (lane == 0) rflag[gi] = moved ? 1 : 0;
      const float m_use = st[r].m_ref == -INFINITY ? 0.f : st[r].m_ref;
      float p[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        p[j] = __builtin_amdgcn_exp2f(__builtin_fmaf(sv[j], a.scale_log2, -m_use));
        st[r].l_run += p[j];
      }
      u32x4_t pop;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        pop[q] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t{p[2 * q], p[2 * q + 1]}), bf16x2_t));
      pex[gi][lane] = pop;
    }
    lds_barrier();
    // 3. O_sl += P V_sl for this wave's groups (rescaled first when the group's reference max moved)
    {
      u32x4_t pop[kPwSub];
#pragma unroll
      for (int u = 0; u < kPwSub; ++u) {
        const int gi = m + M * u;
        if (!sees(gi, key0)) continue;
        if (rflag[gi]) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float al = alx[gi][4 * g + i];
#pragma unroll
            for (int e = 0; e < 8; ++e) o[u][e][i] *= al;
          }
        }
        pop[u] = pex[gi][lane];
      }
      // V operands by transpose reads from this wave's slice of the rows: within 16 lanes, lane 4r + q points at key r,
      // dimensions 4q .. + 3, and lane c receives dimension c of the four keys.
      const int rr = c >> 2, q4 = c & 3;
      const lds_char* vls = (const lds_char*)vl[t & 1];  // vl lives in LDS
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int off = (8 * g + rr) * kRowB + 256 * sl + (16 * e + 4 * q4) * 2;
        const v4i16_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(vls + off));
        const v4i16_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(vls + off + 4 * kRowB));
        u32x4_t bop;
        bop[0] = (uint32_t)(uint16_t)lo[0] | ((uint32_t)(uint16_t)lo[1] << 16);
        bop[1] = (uint32_t)(uint16_t)lo[2] | ((uint32_t)(uint16_t)lo[3] << 16);
        bop[2] = (uint32_t)(uint16_t)hi[0] | ((uint32_t)(uint16_t)hi[1] << 16);
        bop[3] = (uint32_t)(uint16_t)hi[2] | ((uint32_t)(uint16_t)hi[3] << 16);
#pragma unroll
        for (int u = 0; u < kPwSub; ++u) {
          if (!sees(m + M * u, key0)) continue;
          o[u][e] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, pop[u]),
                                                            __builtin_bit_cast(bf16x8_t, bop), o[u][e], 0, 0, 0);
        }
      }
    }
    if (t + 1 < nt) {
      put(vl[(t + 1) & 1]);  // read last by tile t - 1's P V, before this tile's first barrier
      if (t + 2 < nt) fetch(t + 2, kbase);
    }
  }

  // ---- probability sums from the softmax owners, then each group's 16 output rows of this wave's slice
#pragma unroll
  for (int r = 0; r < OWN; ++r) {
    const int gi = w + kPwWaves * r;
    if (gi >= NG) continue;
    float l_tot = st[r].l_run + __shfl_xor(st[r].l_run, 16, kWave);
    l_tot += __shfl_xor(l_tot, 32, kWave);
    if (g == 0) lsum[gi][c] = l_tot;
  }
  lds_barrier();
#pragma unroll
  for (int u = 0; u < kPwSub; ++u) {
    const int gi = m + M * u;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int qq = qb + 16 * gi + 4 * g + i;
      if (qq >= a.width) continue;
      const float li = lsum[gi][4 * g + i];
      const float div = li > 0.f ? li : 1.f;
      uint16_t* orow = a.out + ((int64_t)(b * a.width + qq) * a.H + h) * D + 128 * sl;
#pragma unroll
      for (int e = 0; e < 8; ++e) orow[16 * e + c] = (uint16_t)pack_bf16x2(o[u][e][i] / div, 0.f);
    }
  }
}

// Head dim 512: one workgroup of 8 waves per 64 queries, two kinds of waves side by side on each SIMD.  Waves 0..3
// ("scores") compute S^T = K Q^T, the softmax and P; waves 4..7 ("values") compute O^T += V^T P^T one 64-key tile
// behind, so the softmax of a tile runs beside the matrix work of the one before, and a wave holds either Q (32 queries
// x 512 dimensions, 128 registers) or O (64 queries x 128 dimensions, 128 registers), never both.  Both products are
// v_mfma_f32_32x32x16_bf16.  One barrier per tile.
//
//  * Score wave w: queries 32 (w & 1) .. + 31, keys 32 (w >> 1) .. + 31 of the tile, all 512 dimensions.  Lane (x =
//    lane % 32, g = lane / 32) gets query x's scores of keys 8 (i / 4) + 4g + i % 4, i < 16, and writes them as
//    probabilities to LDS, 8 at a time: exactly the lane's B operand of O^T += V^T P^T.
//  * Value wave w: dimensions 128w .. + 127 of all 64 queries.  V comes straight from memory into registers (each
//    wave reads its own quarter of every row: nothing to share through LDS) in 16-byte loads, a whole tile ahead; a lane
//    swap and a byte permute per operand dword transpose it.  Rows past the context read 0 (buffer bounds).  These
//    waves also bring the next tile's K rows to LDS (global_load_lds, one 1 KB row each, rows 1040 bytes apart so
//    that the 32 rows of an operand read start on different banks).
//  * Softmax reference: a query's reference is the maximum of the first tile, and moves only when a score exceeds it
//    by 2^kWsGuard (probabilities are relative, so fp32 and bf16 lose nothing; only their range is used).  Then, and
//    on the first tile, the tile's two key halves exchange their maxima, P is written again and O is rescaled, between
//    two more barriers (uniform over the workgroup: a flag every wave reads after the tile's barrier).
//
// What bounds a tile (64 queries x 64 keys): 2048 clocks of matrix work per SIMD, 2048 of the CU's vector memory path
// (128 KB of K and V at 64 bytes a clock), 1860 of LDS; as a value wave issues its loads and its products in one order, a
// tile takes ~3000 (1.3 us) where one context leaves CUs idle, and ~5200 (2.5 us, 39% of it matrix work) with every CU
// reading its XCD's L2.  The kernel this replaced added the partial scores of four 128-dimension slices through LDS, with
// three barriers per 32 keys of 96 queries (5500 clocks for 1536 of matrix work).  Measured, 8 heads: 8 contexts x 2048
// 521 -> 357 us (770 TFLOP/s; in chains 329, see ws_group); one context of 1433, where the longest block is the launch,
// 110 -> 38 us.  Tried: 8-byte V loads of the operand's own rows, 390 / 45 us (the memory path takes a load instruction
// per 64 lanes, not only its bytes); the loads spread between the products, 390-430 us (the tile's rows arrive later and
// its products compete with the scores'); K rows brought by the score waves, 404 us; wave priorities, no change.
constexpr int kWsD = 512, kWsQ = 64, kWsK = 64;
constexpr int kWsRow = kWsD * 2 + 16;  // LDS bytes per K row
constexpr int kWsAhead = 4;
constexpr float kWsGuard = 16.0f;
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ f32x16_t mfma32(u32x4_t a, u32x4_t b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0,
                                                 0, 0);
}

// A wave-uniform pointer in scalar registers.
__device__ __forceinline__ const char* scalar_pointer(const void* p) {
  const uint64_t u = reinterpret_cast<uint64_t>(p);
  return reinterpret_cast<const char*>((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)u) |
                                       (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(u >> 32)) << 32);
}

// Chains: a workgroup fills a CU's LDS, so with more blocks than CUs each block's start (first K tile and Q, 6-7 us)
// and end (2-3 us) stood between the tiles of two blocks.  In a chain the next block's first tile is the tile after the
// last: its K and V are on the way and its scores run beside the last values of the block before.  XCD x's blocks, those
// of units (head, context) x, x + 8, .., are listed group after group of ``group`` units, within a group the longest
// blocks first, and dealt to the XCD's kWsPerXcd workgroups there and back, so that long and short blocks even out.
constexpr int kWsPerXcd = 32;  // workgroups at a time: one per CU

// The longest chain of an XCD's workgroups, in tiles (and one for each block), with ``group`` units listed together: the
// deal of prefill_attn_ws_kernel's ``place``, block after block.
inline int ws_longest(int nqb, int units8, int group) {
  int tiles[kWsPerXcd] = {}, c = 0, step = 1;
  for (int g0 = 0; g0 < units8; g0 += group) {
    const int members = std::min(group, units8 - g0);
    for (int t = nqb; t > 0; --t) {
      for (int m = 0; m < members; ++m) {
        tiles[c] += t + 1;
        c += step;
        if (c == kWsPerXcd || c < 0) {  // there and back: the end's workgroup takes two in a row
          step = -step;
          c += step;
        }
      }
    }
  }
  return *std::max_element(tiles, tiles + kWsPerXcd);
}

// The units in a group, 0 for no chains: what is predicted to end first, in tiles.
//  * No chains: an even share of the XCD's tiles and two for each block's start and end, and nqb / 4 for what the last
//    blocks leave idle.
//  * Groups of up to 8 units, or one of all: the longest chain of the deal (whether groups end with a round decides: at
//    8 x 1433 two units at a time take 201 us, all 193, no chains 199, at 8 x 1536 199, 209 and 228), 0.1% longer for each
//    block of a group past 128, whose K and V the XCD's L2 no longer holds (16 x 1024, even chains all: 214 us with 2
//    units, 225 with 8, 253 with 16), and 2% for a unit alone (8 x 2048 336, with 2 330).
// Below two rounds nothing evens out (2 contexts x 1433, 1.4 rounds: 49.5 us in chains, 47.9 without), nor with one unit,
// whose longest block is the launch (1 x 4100: 152, 146).
// Measured at 103 shapes, 8 heads, 2 to 16 contexts x 330 to 3000, every group size, repeated on one state: the choice is
// within 1% of the best one on the mean, 14% at most (16 x 640, 126 us against 111).  us, 8 contexts x width, without
// chains / in the chosen groups: 500 42 / 37, 1984 317 (none chosen; 343 with all 8), 2048 360 / 330, 2049 369 / 354, 2300
// 432 / 398, 2560 507 / 488, 3000 640 (none); 5 x 1024 84 / 74; 12 x 500 78 / 64; 16 x 1536 443 / 391.  The choice takes
// the host ~2 ns for each block of each candidate.
inline int ws_group(int nqb, int units8) {
  if ((int64_t)nqb * units8 < 2 * kWsPerXcd || units8 < 2) return 0;
  const float n = (float)nqb;
  float least = (float)units8 * n * ((n + 1.f) * 0.5f + 2.f) / kWsPerXcd + 0.25f * n;
  int pick = 0;
  for (int i = 1; i <= std::min(units8, 9); ++i) {
    const int group = i == 9 ? units8 : i;
    const float spilled = (float)std::max((int64_t)group * nqb - 128, (int64_t)0);
    const float tiles =
        (float)ws_longest(nqb, units8, group) * (1.f + 0.001f * spilled) * (group == 1 ? 1.02f : 1.f);
    if (tiles < least) {
      least = tiles;
      pick = group;
    }
  }
  return pick;
}

// A query block of a workgroup at head dim 512, its chain's ``round``-th.
struct WsBlock {
  int round, qb, h, b;
};
struct WsTile {  // key tile t of a block
  WsBlock blk;
  int t;
  const char *kbase, *vbase;
};

template <bool kChain>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void prefill_attn_ws_kernel(PrefillArgs a) {
  constexpr int D = kWsD;
  __shared__ __attribute__((aligned(16))) char kls[2][kWsK * kWsRow];
  __shared__ u32x4_t ps[2][2][4][64];  // [tile parity][query half][16-key step][lane]
  __shared__ float mxs[2][kWsQ];       // a tile's maxima by key half, when the reference moves
  __shared__ float als[kWsQ];          // then: the factors O is rescaled by
  __shared__ float lsum[2][2][2][kWsQ];  // [parity of the block in the chain]: probability sums by key half, lane half
  __shared__ int moved[4];             // by tile % 4: a score passed the guard
  const int nqb = (a.width + kWsQ - 1) / kWsQ;
  const int tid = threadIdx.x, lane = tid & 63, x = lane & 31, g = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (tid < 4) moved[tid] = 0;
  // The workgroup's block of a round, from its XCD's list; false past its end.
  auto place = [&](WsBlock& blk, int round) {
    const int c = (int)blockIdx.x / 8;
    const int p = round * kWsPerXcd + (round & 1 ? kWsPerXcd - 1 - c : c);
    if (p >= a.units8 * nqb) return false;
    const int full = a.group * nqb, g0 = p / full * a.group, r = p % full, members = min(a.group, a.units8 - g0);
    const int unit = (g0 + r % members) * 8 + (int)blockIdx.x % 8;
    blk = WsBlock{round, (nqb - 1 - r / members) * kWsQ, unit % a.H, unit / a.H};
    return true;
  };
  auto first = [&]() {
    WsBlock blk;
    if constexpr (kChain) {
      place(blk, 0);
    } else {
      const PfBlock one = pf_block(nqb, a.H, (int)gridDim.z);
      blk = WsBlock{0, (nqb - 1 - one.j) * kWsQ, one.h, one.b};  // the longest blocks first
    }
    return blk;
  };
  auto next = [&](WsBlock& blk) {  // false (and blk as it was): that was the last
    if constexpr (kChain) return place(blk, blk.round + 1);
    return false;
  };

  if (w < 4) {  // ------------------------------------------------------------------------------ scores
    const int qh = w & 1, kh = w >> 1;
    // K operands in a ring kWsAhead steps ahead of the products: an LDS read takes a few products' time to arrive.
    u32x4_t kf[kWsAhead];
    auto k_at = [&](int t, int s) {
      return *reinterpret_cast<const u32x4_t*>(&kls[t & 1][(32 * kh + x) * kWsRow + g * 16 + s * 32]);
    };
    WsBlock blk = first();
    int t = 0;  // counted over the workgroup's blocks, as is all LDS
    for (int odd = 0;; odd ^= 1) {
      const int qb = blk.qb, query = qb + 32 * qh + x, t_last = t + qb / kWsK;  // the last tile holds the diagonal
      u32x4_t q[D / 16];  // q[query][16s + 8g .. + 7] (past the end the last query's: its results are not stored)
      {
        const uint16_t* qrow = a.q + ((int64_t)(blk.b * a.width + min(query, a.width - 1)) * a.H + blk.h) * D + g * 8;
#pragma unroll
        for (int s = 0; s < D / 16; ++s) q[s] = *reinterpret_cast<const u32x4_t*>(qrow + s * 16);
      }
      float m_ref = -INFINITY, thr = -INFINITY, l_run = 0.f;
      if (t == 0) {
        lds_barrier();  // the first K tile
#pragma unroll
        for (int s = 0; s < kWsAhead; ++s) kf[s] = k_at(0, s);
      }
      for (; t <= t_last; ++t) {
        f32x16_t s0, s1;
#pragma unroll
        for (int i = 0; i < 16; ++i) s0[i] = s1[i] = 0.f;
#pragma unroll
        for (int s = 0; s < D / 16; ++s) {
          if (s & 1) s1 = mfma32(kf[s % kWsAhead], q[s], s1);
          else s0 = mfma32(kf[s % kWsAhead], q[s], s0);
          if (s + kWsAhead < D / 16) {
            kf[s % kWsAhead] = k_at(t, s + kWsAhead);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one product, one LDS read
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          }
        }
        float sv[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) sv[i] = s0[i] + s1[i];
        if (t == t_last) {
          const int rel = 32 * qh + x - (32 * kh + 4 * g);  // keys 8 (i / 4) + i % 4 <= rel are seen
#pragma unroll
          for (int i = 0; i < 16; ++i) sv[i] = 8 * (i >> 2) + (i & 3) <= rel ? sv[i] : -INFINITY;
        }
        bool over = false;
#pragma unroll
        for (int i = 0; i < 16; ++i) over |= sv[i] > thr;
        if (__any(over) && lane == 0) moved[t & 3] = 1;
        float lt = 0.f;
        auto put_p = [&](float m) {
          lt = 0.f;
#pragma unroll
          for (int s = 0; s < 2; ++s) {
            u32x4_t pop;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(sv[8 * s + 2 * e], a.scale_log2, -m));
              const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(sv[8 * s + 2 * e + 1], a.scale_log2, -m));
              lt += p0 + p1;
              pop[e] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t{p0, p1}), bf16x2_t));
            }
            ps[t & 1][qh][2 * kh + s][lane] = pop;
          }
        };
        put_p(m_ref == -INFINITY ? 0.f : m_ref);
        lds_barrier();
        const int again = moved[t & 3];  // uniform over the workgroup
#pragma unroll
        for (int s = 0; s < kWsAhead; ++s) kf[s] = k_at(t + 1, s);  // (past the last tile: unused)
        if (w == 0 && lane == 0) moved[(t + 2) & 3] = 0;
        if (again) {
          float mx = sv[0];
#pragma unroll
          for (int i = 1; i < 16; ++i) mx = fmaxf(mx, sv[i]);
          mx = fmaxf(mx, __shfl_xor(mx, 32, kWave));
          if (g == 0) mxs[kh][32 * qh + x] = mx;
          lds_barrier();
          const float m_new = fmaxf(m_ref, fmaxf(mxs[0][32 * qh + x], mxs[1][32 * qh + x]) * a.scale_log2);
          const float alpha = __builtin_amdgcn_exp2f(m_ref - (m_new == -INFINITY ? 0.f : m_new));  // m_ref = -inf: 0
          if (kh == 0 && g == 0) als[32 * qh + x] = alpha;
          l_run *= alpha;
          m_ref = m_new;
          thr = m_new == -INFINITY ? -INFINITY : (m_new + kWsGuard) / a.scale_log2;
          put_p(m_ref == -INFINITY ? 0.f : m_ref);
          lds_barrier();
        }
        l_run += lt;
      }
      lsum[odd][kh][g][32 * qh + x] = l_run;
      if (!next(blk)) break;
    }
    lds_barrier();
    return;
  }

  // ---------------------------------------------------------------------------------------------- values
  const int vw = w - 4;
  // [query half][e]: row r is dimension 128 vw + 8 (r % 16) + 4 (r / 16) + e, column x query x of the half
  f32x16_t o[2][4];
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[u][e][i] = 0.f;
  // K rows 16 vw .. + 15 of tile t to LDS, one row (64 lanes x 16 bytes) per load; rows past the context read its last
  // key (finite: masked).
  auto bring_k = [&](const WsTile& c, int n) {  // as tile n of the workgroup
    const __amdgpu_buffer_rsrc_t kr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(c.kbase), 0, -1, 0x00020000);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int key = min(c.t * kWsK + 16 * vw + r, a.width - 1);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          kr, (__attribute__((address_space(3))) void*)&kls[n & 1][(16 * vw + r) * kWsRow], 16, lane * 16,
          (int)((uint32_t)key * (D * 2)), 0,
          0);
    }
  };
  // V of 16-key step s of tile t: lane (c = x % 16, u = x / 16, g) loads keys 16s + 8u + 4g + j, dimensions 128 vw + 8c
  // .. + 7, j < 4.  A buffer resource per step, its size what is left of the context's rows: scalar work only, and rows
  // past the end read 0.
  const uint32_t vlane = (uint32_t)((8 * (x >> 4) + 4 * g) * D + 128 * vw + 8 * (x & 15)) * 2;
  const uint32_t vbytes = (uint32_t)a.width * (D * 2);
  u32x4_t v[4][4];
  auto load_v = [&](const WsTile& c, int s) {
    const uint32_t off = (uint32_t)(c.t * kWsK + 16 * s) * (D * 2);
    uint32_t used = min(off, vbytes);
    asm("" : "+s"(used));  // kept scalar (the saturating subtraction it would become is a vector instruction)
    const __amdgpu_buffer_rsrc_t vr =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(c.vbase) + off, 0, vbytes - used, 0x00020000);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      v[s][j] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(vr, vlane + j * D * 2, 0, 0));
  };
  u32x4_t p[2][2];  // steps s, s + 1 of tile t
  auto read_p = [&](int t, int s) {
#pragma unroll
    for (int u = 0; u < 2; ++u) p[u][s & 1] = ps[t & 1][u][s][lane];
  };
  // O^T += V^T P^T for the workgroup's tile t; ``ahead``: the next tile's V loads as its registers fall free.  Step
  // s + 1's operands are built beside step s's products; the scheduler keeps each step's loads behind the permutes that read their registers.
  auto attend_v = [&](int t, const WsTile* ahead) {
    u32x4_t vop[2][4];
    auto operands = [&](int s) {
      // The lanes of a pair (u = 0, 1) hold 8 dimensions of 4 keys each; swapped, 4 dimensions (8c + 4u ..) of 8 keys:
      // lo[j] of key 16s + 4g + j, hi[j] of key 16s + 8 + 4g + j.
      u32x2_t lo[4], hi[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int d = 0; d < 2; ++d) {
          const auto r = __builtin_amdgcn_permlane16_swap(v[s][j][d], v[s][j][2 + d], false, false);
          lo[j][d] = r[0];
          hi[j][d] = r[1];
        }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t sel = (e & 1) ? 0x07060302u : 0x05040100u;
#pragma unroll
        for (int q2 = 0; q2 < 2; ++q2) {
          vop[s & 1][e][q2] = __builtin_amdgcn_perm(lo[2 * q2 + 1][e >> 1], lo[2 * q2][e >> 1], sel);
          vop[s & 1][e][2 + q2] = __builtin_amdgcn_perm(hi[2 * q2 + 1][e >> 1], hi[2 * q2][e >> 1], sel);
        }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) asm volatile("" : "+v"(vop[s & 1][e]));  // built here, not where first used
    };
    operands(0);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      __builtin_amdgcn_sched_barrier(0);
      if (ahead) load_v(*ahead, s);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int u = 0; u < 2; ++u) o[u][e] = mfma32(vop[s & 1][e], p[u][s & 1], o[u][e]);
      if (s < 2) read_p(t, s + 2);
      if (s < 3) operands(s + 1);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // After tile t's barrier: its probabilities, and O rescaled when the reference moved on it (O holds the tiles
  // before it).
  auto take_p = [&](int t) {
    const int again = moved[t & 3];
    read_p(t, 0);
    read_p(t, 1);
    if (!again) return;
    lds_barrier();
    lds_barrier();
    read_p(t, 0);
    read_p(t, 1);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const float al = als[32 * u + x];
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[u][e][i] *= al;
    }
  };
  auto output = [&](const WsBlock& blk, int odd) {  // O of a finished block; then O is 0 again
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int query = blk.qb + 32 * u + x;
      const float l = (lsum[odd][0][0][32 * u + x] + lsum[odd][0][1][32 * u + x]) +
                      (lsum[odd][1][0][32 * u + x] + lsum[odd][1][1][32 * u + x]);
      const float inv = l > 0.f ? 1.f / l : 1.f;
      uint16_t* orow = a.out + ((int64_t)(blk.b * a.width + query) * a.H + blk.h) * D + 128 * vw + 32 * g;
      auto pair = [&](float lo, float hi) {
        return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t{lo * inv, hi * inv}), bf16x2_t));
      };
      if (query < a.width) {
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
          for (int i = 0; i < 4; ++i) {  // dimensions 64r + 32g + 8i + 4k + e, k = 0, 1
            u32x4_t out;
#pragma unroll
            for (int k = 0; k < 2; ++k) {
              const int at = 4 * (r + 2 * k) + i;
              out[2 * k] = pair(o[u][0][at], o[u][1][at]);
              out[2 * k + 1] = pair(o[u][2][at], o[u][3][at]);
            }
            *reinterpret_cast<u32x4_t*>(orow + 64 * r + 8 * i) = out;
          }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[u][e][i] = 0.f;
    }
  };
  auto open = [&](WsTile& c) {  // the block's first tile
    const int64_t slot = clamp64(a.slots[c.blk.b], 0, a.cache_rows - 1);
    c.kbase = scalar_pointer(a.k + slot * a.s_row + c.blk.h * a.s_head);
    c.vbase = scalar_pointer(a.v + slot * a.s_row + c.blk.h * a.s_head);
    c.t = 0;
  };
  auto advance = [&](WsTile& c) {  // false (and c as it was): no more tiles
    if (c.t < c.blk.qb / kWsK) {
      ++c.t;
      return true;
    }
    if (!next(c.blk)) return false;
    open(c);
    return true;
  };
  WsTile at, ahead;  // the tiles whose V and whose K come next
  at.blk = first();
  open(at);
  bring_k(at, 0);
  landed_barrier();
  ahead = at;
  bool more = advance(ahead);
  bring_k(ahead, 1);
#pragma unroll
  for (int s = 0; s < 4; ++s) load_v(at, s);
  landed_barrier();
  take_p(0);
  int n = 1, odd = 0;
  while (more) {  // tile n's scores, tile n - 1's values
    const WsBlock was = at.blk;
    at = ahead;
    more = advance(ahead);
    bring_k(ahead, n + 1);  // unconditional (past the last tile: that tile again, not used): no wait joins a branch
    attend_v(n - 1, &at);
    // vmcnt(16): tile n + 1's K rows are in LDS, tile n's 16 V loads, issued after them, stay in flight (lds_barrier
    // would wait for those too).  This wave's LDS reads of the tile are in registers by now.
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0x4f70);
    __builtin_amdgcn_s_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    if (kChain && at.t == 0) {
      output(was, odd);
      odd ^= 1;
    }
    take_p(n);
    ++n;
  }
  attend_v(n - 1, nullptr);
  lds_barrier();
  output(at.blk, odd);
}

// Head dim 128: 256 queries per workgroup, four pairs of a score wave and a value wave (see prefill_attn_ws_kernel), each
// pair its own 64 queries against the same 64-key tiles.  Score wave p of step t multiplies tile t (K from LDS, Q in
// registers) beside the softmax of tile t - 1, so its matrix and vector work overlap within the wave; value wave p
// accumulates tile t - 2.  A pair keeps its own softmax reference (a lane's two queries see every key of the tile
// through lanes x and x + 32), so a moved reference costs no barrier: the factors wait in LDS for the value wave.
// K and V rows go to LDS by direct loads (score waves bring V, value waves K: neither reads what it brings, so its
// loads are waited for at the step's barrier alone, landed_barrier), 1 KB = 4 rows each, 16-byte chunks permuted within
// a row so that the operand reads spread over the banks: chunk c of key r at position c ^ (r % 16) in K, c ^ 4 (r % 4)
// in V.
//
// What bounds a tile (a pair's 64 queries x 64 keys): 2048 clocks of matrix work on its SIMD beside ~1900 of the score
// wave's vector work (64 exponentials per lane at a quarter rate), one barrier per tile.  The kernel this replaced ran
// both in one wave, one after the other, on 16 x 16 products with 192 queries per workgroup.  Measured, 32 heads, before
// and after: 4 contexts x 1777 203 -> 147 us (705 TFLOP/s), 8 x 2048 405 -> 362 us (760), one of 1433 64 -> 42 us, 8 of
// 130 16 -> 13 us.  Tried: fmaxf in place of max3, 157 / 387 us; K operands 3 steps ahead (3 registers spilled) with
// the products and the vector work interleaved by sched_group_barrier, 151 / 378 us; wave priorities, no change.
constexpr int kPairQ = 256, kPairK = 64;

// Without the copy of each operand that fmaxf makes to quiet a signalling NaN (a product has none).  The compiler does
// not see an instruction that reads a, b, c here: a caller with values of the matrix unit waits for them first.
__device__ __forceinline__ float max3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void prefill_attn_pairs_kernel(
    PrefillArgs a) {
  constexpr int D = 128;
  __shared__ __attribute__((aligned(16))) char kls[2][kPairK * D * 2];
  __shared__ __attribute__((aligned(16))) char vls[2][kPairK * D * 2];
  __shared__ u32x4_t ps[4][2][2][4][64];  // [pair][tile parity][query half][16-key step][lane]
  __shared__ float als[4][4][64];         // [pair][tile % 4]: O's factors, when the reference moved
  __shared__ int moved[4][4];
  __shared__ float lsum[4][2][64];        // [pair][lane half]
  const int nqb = (a.width + kPairQ - 1) / kPairQ;
  const PfBlock blk = pf_block(nqb, a.H, (int)gridDim.z);
  const int qb = (nqb - 1 - blk.j) * kPairQ;  // the longest blocks first
  const int h = blk.h, b = blk.b;
  const int tid = threadIdx.x, lane = tid & 63, x = lane & 31, g = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), pr = w & 3;
  const int64_t slot = clamp64(a.slots[b], 0, a.cache_rows - 1);
  const char* kbase = scalar_pointer(a.k + slot * a.s_row + h * a.s_head);
  const char* vbase = scalar_pointer(a.v + slot * a.s_row + h * a.s_head);
  const int nt = (min(qb + kPairQ, a.width) + kPairK - 1) / kPairK;
  const int qp = qb + 64 * pr;
  const int dq = qp < a.width ? qp / kPairK : -1;  // the pair's last tile, which holds its diagonal (-1: no queries)

  // Rows 16 pr .. + 15 of tile t to LDS; rows past the context read its last key (finite: masked).  ``swap``: the chunk
  // permutation of key row r of a 16-row group.
  auto bring = [&](const __amdgpu_buffer_rsrc_t rsrc, char* dst, int t, auto swap) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int r = 4 * j + (lane >> 4);
      const int key = min(t * kPairK + 16 * pr + r, a.width - 1);
      const uint32_t from = (uint32_t)key * (D * 2) + (uint32_t)((lane & 15) ^ swap(r)) * 16;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rsrc, (__attribute__((address_space(3))) void*)(dst + (16 * pr + 4 * j) * (D * 2)), 16, from, 0, 0, 0);
    }
  };

  if (w < 4) {  // ------------------------------------------------------------------------------ scores
    const __amdgpu_buffer_rsrc_t vr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(vbase), 0, -1, 0x00020000);
    auto bring_v = [&](int t) { bring(vr, vls[t & 1], t, [](int r) { return 4 * (r & 3); }); };
    u32x4_t q[2][D / 16];  // q[query][16s + 8g .. + 7], query qp + 32u + x
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const uint16_t* qrow =
          a.q + ((int64_t)(b * a.width + min(qp + 32 * u + x, a.width - 1)) * a.H + h) * D + g * 8;
#pragma unroll
      for (int s = 0; s < D / 16; ++s) q[u][s] = *reinterpret_cast<const u32x4_t*>(qrow + s * 16);
    }
    float m_ref[2] = {-INFINITY, -INFINITY}, thr[2] = {-INFINITY, -INFINITY}, l_run[2] = {0.f, 0.f};
    const int klane = x * (D * 2) + ((g ^ (x & 15)) * 16);
    auto k_at = [&](int t, int m, int s) {
      return *reinterpret_cast<const u32x4_t*>(&kls[t & 1][32 * m * (D * 2) + (klane ^ (32 * s))]);
    };
    typedef f32x16_t Scores[2][2];  // [key half m][query half u]
    f32x16_t zero;
#pragma unroll
    for (int i = 0; i < 16; ++i) zero[i] = 0.f;
    // One 16-key step's probabilities of query half u: keys 16 (2m + hf) .., as the value wave's operand.
    auto put_p = [&](const Scores& sc, int t, int m, int hf, int u, float mu) {
      u32x4_t pop;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[m][u][8 * hf + 2 * e], a.scale_log2, -mu));
        const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[m][u][8 * hf + 2 * e + 1], a.scale_log2, -mu));
        l_run[u] += p0 + p1;
        pop[e] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t{p0, p1}), bf16x2_t));
      }
      ps[pr][t & 1][u][2 * m + hf][lane] = pop;
    };
    // The reference of tile t's scores (masked on the pair's last tile).
    auto refer = [&](Scores& sc, int t) {
      // max3's operands come from the matrix unit: every product has written its result after 24 wait states.
      asm volatile("s_nop 15\n\ts_nop 7" : "+v"(sc[0][0]), "+v"(sc[0][1]), "+v"(sc[1][0]), "+v"(sc[1][1]));
      if (t == dq) {
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            const int rel = 32 * u + x - (32 * m + 4 * g);  // keys 8 (i / 4) + i % 4 <= rel are seen
#pragma unroll
            for (int i = 0; i < 16; ++i) sc[m][u][i] = 8 * (i >> 2) + (i & 3) <= rel ? sc[m][u][i] : -INFINITY;
          }
      }
      float mx[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        mx[u] = max3(sc[0][u][0], sc[1][u][0], sc[0][u][1]);
        mx[u] = max3(mx[u], sc[1][u][1], sc[1][u][1]);
#pragma unroll
        for (int i = 2; i < 16; ++i) mx[u] = max3(mx[u], sc[0][u][i], sc[1][u][i]);
      }
      const bool move = __any(mx[0] > thr[0] || mx[1] > thr[1]);
      if (lane == 0) moved[pr][t & 3] = move ? 1 : 0;
      if (move) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const float top = fmaxf(mx[u], __shfl_xor(mx[u], 32, kWave));
          const float m_new = fmaxf(m_ref[u], top * a.scale_log2);
          const float alpha = __builtin_amdgcn_exp2f(m_ref[u] - (m_new == -INFINITY ? 0.f : m_new));  // m_ref = -inf: 0
          if (g == 0) als[pr][t & 3][32 * u + x] = alpha;
          l_run[u] *= alpha;
          m_ref[u] = m_new;
          thr[u] = m_new == -INFINITY ? -INFINITY : (m_new + kWsGuard) / a.scale_log2;
        }
      }
    };
    // Step t: tile t's products into ``to``, the softmax of tile t - 1's scores ``from`` beside them.
    auto step = [&](const Scores& from, Scores& to, int t, bool soft) {
      u32x4_t kf[2] = {k_at(t, 0, 0), k_at(t, 1, 0)};
      const float m0 = m_ref[0] == -INFINITY ? 0.f : m_ref[0], m1 = m_ref[1] == -INFINITY ? 0.f : m_ref[1];
#pragma unroll
      for (int s = 0; s < D / 16; ++s) {
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
          for (int u = 0; u < 2; ++u) to[m][u] = mfma32(kf[m], q[u][s], s == 0 ? zero : to[m][u]);
        if (s + 1 < D / 16) {
#pragma unroll
          for (int m = 0; m < 2; ++m) kf[m] = k_at(t, m, s + 1);
        }
        if (soft) put_p(from, t - 1, s >> 2, (s >> 1) & 1, s & 1, s & 1 ? m1 : m0);
      }
      refer(to, t);
    };
    auto finish = [&](const Scores& from, int t) {  // the pair's last tile
      const float m0 = m_ref[0] == -INFINITY ? 0.f : m_ref[0], m1 = m_ref[1] == -INFINITY ? 0.f : m_ref[1];
#pragma unroll
      for (int s = 0; s < 8; ++s) put_p(from, t, s >> 2, (s >> 1) & 1, s & 1, s & 1 ? m1 : m0);
#pragma unroll
      for (int u = 0; u < 2; ++u) lsum[pr][g][32 * u + x] = l_run[u];
    };
    Scores sa, sb;
    lds_barrier();  // the first K tile (these waves have brought nothing yet)
    if (dq >= 0) step(sb, sa, 0, false);
    lds_barrier();
    int t = 1;
    for (; t + 1 <= dq; t += 2) {
      bring_v(t - 1);
      step(sa, sb, t, true);
      landed_barrier();
      bring_v(t);
      step(sb, sa, t + 1, true);
      landed_barrier();
    }
    if (t <= dq) {  // one more, then its scores are in sb
      bring_v(t - 1);
      step(sa, sb, t, true);
      landed_barrier();
      bring_v(t);
      finish(sb, t);
      landed_barrier();
      t += 2;
    } else if (dq >= 0) {
      bring_v(t - 1);
      finish(sa, t - 1);
      landed_barrier();
      t += 1;
    }
    for (; t <= nt + 1; ++t) {
      if (t <= nt) bring_v(t - 1);
      landed_barrier();
    }
    return;
  }

  // ---------------------------------------------------------------------------------------------- values
  const __amdgpu_buffer_rsrc_t kr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(kbase), 0, -1, 0x00020000);
  auto bring_k = [&](int t) { bring(kr, kls[t & 1], t, [](int r) { return r; }); };
  f32x16_t o[2][4];  // [query half][e]: row 16k + 4q + i is dimension 32e + 8q + 4k + i, column x query x of the half
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[u][e][i] = 0.f;
  // V operands by transpose reads: within 16 lanes (k = lane / 16 % 2), lane 4r + q points at key 4g + r, dimensions
  // 32e + 8q + 4k .., and lane 4q + i receives dimension 32e + 8q + 4k + i of the four keys.
  const int r = (lane & 15) >> 2, q4 = lane & 3, k2 = (lane >> 4) & 1;
  int vlane[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) vlane[e] = (4 * g + r) * (D * 2) + (e ^ r) * 64 + q4 * 16 + k2 * 8;
  auto attend_v = [&](int t) {
    u32x4_t p[2][4];
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int u = 0; u < 2; ++u) p[u][s] = ps[pr][t & 1][u][s][lane];
    if (moved[pr][t & 3]) {  // wave-uniform
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const float al = als[pr][t & 3][32 * u + x];
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[u][e][i] *= al;
      }
    }
    const lds_char* vt = (const lds_char*)vls[t & 1];
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const v4i16_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(vt + vlane[e] + s * 16 * D * 2));
        const v4i16_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(vt + vlane[e] + (s * 16 + 8) * D * 2));
        const u32x2_t l2 = __builtin_bit_cast(u32x2_t, lo), h2 = __builtin_bit_cast(u32x2_t, hi);
        const u32x4_t vop = {l2[0], l2[1], h2[0], h2[1]};
#pragma unroll
        for (int u = 0; u < 2; ++u) o[u][e] = mfma32(vop, p[u][s], o[u][e]);
      }
  };
  bring_k(0);
  landed_barrier();
  for (int t = 0; t <= nt + 1; ++t) {
    if (t + 1 < nt) bring_k(t + 1);
    if (t >= 2 && t - 2 <= dq) attend_v(t - 2);
    landed_barrier();
  }
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int query = qp + 32 * u + x;
    if (query >= a.width) continue;
    const float l = lsum[pr][0][32 * u + x] + lsum[pr][1][32 * u + x];
    const float inv = l > 0.f ? 1.f / l : 1.f;
    uint16_t* orow = a.out + ((int64_t)(b * a.width + query) * a.H + h) * D + 8 * g;
    auto pair = [&](float lo, float hi) {
      return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t{lo * inv, hi * inv}), bf16x2_t));
    };
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) {  // dimensions 32e + 16 rb + 8g .. + 7
        u32x4_t out;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const int at = 4 * (rb + 2 * k);
          out[2 * k] = pair(o[u][e][at], o[u][e][at + 1]);
          out[2 * k + 1] = pair(o[u][e][at + 2], o[u][e][at + 3]);
        }
        *reinterpret_cast<u32x4_t*>(orow + 32 * e + 16 * rb) = out;
      }
  }
}

// Head dim 128 in blocks of 192 queries, for the launches of small_blocks: one workgroup of 4 waves, two workgroups per
// CU.  The block's 32-key tiles go through LDS once for all of its waves (double-buffered: tile t + 1's global loads are
// in flight during tile t's math).  Each wave holds kPfSub groups of 16 queries: per tile it reads the K fragments and,
// by LDS transpose reads, the V operands once, then runs S^T = K Q^T, the lazy softmax (causal limit as the key limit,
// skipped on tiles the whole group sees) and O += P V for every group that sees the tile.  What bounds it is that its
// products and its softmax share one wave: a tile takes ~1.7 times as long as in the pairs kernel, but a CU holds two.
constexpr int kPfWaves = 4;
constexpr int kPfSub = 3;  // 16-query groups per wave (3: 255 VGPRs, two waves per SIMD; measured fastest of 1-4)
constexpr int kPfQueries = 16 * kPfSub * kPfWaves;
constexpr int kPfRow = 128 * 2 + 16;  // LDS bytes per key row: 256 B of data, padded against bank conflicts
constexpr int kPfStage = 32;          // keys per LDS stage (one barrier each), a multiple of the 32-key MFMA tile
constexpr int kPfThreads = 64 * kPfWaves;
constexpr int kPfChunks = kPfStage * 16 / kPfThreads;  // 16-byte chunks of K (and of V) per thread per stage
static_assert(kPfChunks * kPfThreads == kPfStage * 16, "a stage is whole chunks per thread");

// Whether a launch at head dim 128 takes blocks of 192 queries, two per CU, rather than the pairs kernel's 256, one per
// CU: where the pairs kernel needs more than one round of its 256 workgroups and
//  * both sizes give the same number of blocks per unit, so that this one has half the rounds, and the 192 are at most 5/6
//    full on the mean (past that its time grows with the queries, the pairs kernel's does not);
//  * or, with one block more per unit at two or four blocks of 256, the pairs kernel's last round is nearly empty and this
//    kernel takes fewer rounds (with three, the blocks of that round are the short ones, and it costs little).
// Pairs kernel / this one, us: 160 units (5 contexts x 32 heads) x 257 27.3 / 22.7, x 300 27.4 / 24.8, x 385 33.5 / 30.6, x 384
// 30.0 / 32.2 (full: pairs); 256 x 257 29.0 / 24.2; 320 x 129 22.0 / 18.8; 130 x 512 40.7 / 32.9, 192 x 512 42.2 / 48.3
// (as many rounds: pairs); 96 x 800 50.8 / 47.0, 96 x 640 35.4 / 41.5 (three blocks: pairs).
inline bool small_blocks(int width, int64_t units) {
  constexpr int kCus = 256;
  const int n = (width + kPairQ - 1) / kPairQ, small = (width + kPfQueries - 1) / kPfQueries;
  const int64_t blocks = n * units, rounds = (blocks + kCus - 1) / kCus;
  if (rounds < 2) return false;
  if (n == small) return width <= kPfQueries * 5 / 6 * n;
  const int64_t small_rounds = (small * units + 2 * kCus - 1) / (2 * kCus), last = blocks % kCus;
  if (small != n + 1 || (n != 2 && n != 4) || last == 0 || small_rounds >= rounds) return false;
  return last <= 96 || (2 * small_rounds <= rounds && last <= 128);
}

// The softmax step of one 16-query group for one tile: mask (key0 + j >= lim), lazy reference max, this lane's
// 8 probabilities packed as the P operand.  (The same arithmetic as attend().)
template <int NB>
__device__ __forceinline__ u32x4_t softmax_tile(float (&sv)[8], float c_scale, SoftmaxState& st, f32x4_t (&o)[NB],
                                                int g, int key0, int lim, bool whole) {
  bool over = false;
  if (!whole) {  // whole (wave-uniform): every query of the group sees every key of the tile
#pragma unroll
    for (int j = 0; j < 8; ++j) sv[j] = key0 + j < lim ? sv[j] : -INFINITY;
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) over |= sv[j] > st.thr;
  if (__any(over)) {
    float mx = sv[0];
#pragma unroll
    for (int j = 1; j < 8; ++j) mx = fmaxf(mx, sv[j]);
    mx = fmaxf(mx, __shfl_xor(mx, 16, kWave));
    mx = fmaxf(mx, __shfl_xor(mx, 32, kWave));
    const float m_new = fmaxf(st.m_ref, mx * c_scale);
    rescale<NB>(st.m_ref, m_new == -INFINITY ? 0.f : m_new, st.l_run, o, g);
    st.m_ref = m_new;
    st.thr = m_new == -INFINITY ? -INFINITY : (m_new + kLazyLog2) / c_scale;
  }
  const float m_use = st.m_ref == -INFINITY ? 0.f : st.m_ref;
  float p[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    p[j] = __builtin_amdgcn_exp2f(__builtin_fmaf(sv[j], c_scale, -m_use));
    st.l_run += p[j];
  }
  u32x4_t pop;
#pragma unroll
  for (int w = 0; w < 4; ++w)
    pop[w] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t{p[2 * w], p[2 * w + 1]}), bf16x2_t));
  return pop;
}

__global__ __launch_bounds__(64 * kPfWaves) __attribute__((amdgpu_waves_per_eu(2, 2))) void prefill_attn_kernel(
    PrefillArgs a) {
  constexpr int D = 128, KS = D / 32;
  __shared__ __attribute__((aligned(16))) char lds[2][2][kPfStage * kPfRow];  // [buffer][K, V][key rows]
  const int nqb = (a.width + kPfQueries - 1) / kPfQueries;
  const PfBlock blk = pf_block(nqb, a.H, (int)gridDim.z);
  const int qb = (nqb - 1 - blk.j) * kPfQueries;  // the longest blocks first
  const int h = blk.h, b = blk.b;
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t slot = clamp64(a.slots[b], 0, a.cache_rows - 1);
  const uint16_t* kbase = a.k + slot * a.s_row + h * a.s_head;
  const uint16_t* vbase = a.v + slot * a.s_row + h * a.s_head;
  const int kend = min(qb + kPfQueries, a.width);  // keys the block's last query sees
  const int nt = (kend + kPfStage - 1) / kPfStage;

  // Global -> LDS: thread tid moves 16-byte chunks tid, tid + kPfThreads, ... of the stage's K and of its V (kPfStage rows x
  // 256 B each).  Rows past the context read its last key (finite: masked by the causal limit, never NaN).
  u32x4_t stage[2 * kPfChunks];
  auto fetch = [&](int t) {
#pragma unroll
    for (int e = 0; e < kPfChunks; ++e) {
      const int ci = tid + e * kPfThreads, r = ci >> 4, col = ci & 15;
      const int key = min(t * kPfStage + r, a.width - 1);
      stage[e] = *reinterpret_cast<const u32x4_t*>(kbase + (int64_t)key * D + col * 8);
      stage[kPfChunks + e] = *reinterpret_cast<const u32x4_t*>(vbase + (int64_t)key * D + col * 8);
    }
  };
  auto put = [&](int buf) {
#pragma unroll
    for (int e = 0; e < kPfChunks; ++e) {
      const int ci = tid + e * kPfThreads, r = ci >> 4, col = ci & 15;
      *reinterpret_cast<u32x4_t*>(&lds[buf][0][r * kPfRow + col * 16]) = stage[e];
      *reinterpret_cast<u32x4_t*>(&lds[buf][1][r * kPfRow + col * 16]) = stage[kPfChunks + e];
    }
  };

  // The wave's groups: queries q0[u] + c, u < kPfSub (group u of wave w: block rows 16 (w + kPfWaves u)).
  int q0[kPfSub];
  u32x4_t qop[kPfSub][KS];  // B operand of S^T = K Q^T: lane (c, g) holds q[q0 + c][32s + 8g .. +7] (0 past the end)
  SoftmaxState st[kPfSub];
  f32x4_t o[kPfSub][D / 16];
#pragma unroll
  for (int u = 0; u < kPfSub; ++u) {
    q0[u] = qb + 16 * (w + kPfWaves * u);
    const bool live = q0[u] + c < a.width;
    const uint16_t* qrow = a.q + ((int64_t)(b * a.width + (live ? q0[u] + c : 0)) * a.H + h) * D + g * 8;
#pragma unroll
    for (int s2 = 0; s2 < KS; ++s2)
      qop[u][s2] = live ? *reinterpret_cast<const u32x4_t*>(qrow + s2 * 32) : u32x4_t{0u, 0u, 0u, 0u};
    st[u] = SoftmaxState{-INFINITY, -INFINITY, 0.f};
#pragma unroll
    for (int nb = 0; nb < D / 16; ++nb) o[u][nb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }

  fetch(0);
  put(0);
  __syncthreads();
  for (int t = 0; t < nt; ++t) {
    fetch(t + 1 < nt ? t + 1 : t);  // unconditional: the last iteration re-reads its own tile (cache hit)
    // The stage's 32-key MFMA tiles in turn.
#pragma unroll
    for (int sub = 0; sub < kPfStage / 32; ++sub) {
    const int key0 = t * kPfStage + sub * 32;
    // Groups that see the tile (wave-uniform): a live group whose last query reaches the tile's first key.
    bool act[kPfSub];
    bool any = false;
#pragma unroll
    for (int u = 0; u < kPfSub; ++u) {
      act[u] = q0[u] < a.width && key0 <= q0[u] + 15;
      any |= act[u];
    }
    if (any) {
      const char* kl = lds[t & 1][0] + sub * 32 * kPfRow;
      const char* vl = lds[t & 1][1] + sub * 32 * kPfRow;
      u32x4_t pop[kPfSub];
      {
        u32x4_t kf[2][KS];
#pragma unroll
        for (int mb = 0; mb < 2; ++mb) {
          const int rk = 8 * (c >> 2) + 4 * mb + (c & 3);
#pragma unroll
          for (int s2 = 0; s2 < KS; ++s2) kf[mb][s2] = *reinterpret_cast<const u32x4_t*>(kl + rk * kPfRow + g * 16 + s2 * 64);
        }
#pragma unroll
        for (int u = 0; u < kPfSub; ++u) {
          if (!act[u]) continue;
          f32x4_t sacc[2];
#pragma unroll
          for (int mb = 0; mb < 2; ++mb) {
            sacc[mb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s2 = 0; s2 < KS; ++s2)
              sacc[mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, kf[mb][s2]),
                                                                 __builtin_bit_cast(bf16x8_t, qop[u][s2]), sacc[mb],
                                                                 0, 0, 0);
          }
          float sv[8];
#pragma unroll
          for (int j = 0; j < 8; ++j) sv[j] = sacc[j >> 2][j & 3];
          pop[u] = softmax_tile<D / 16>(sv, a.scale_log2, st[u], o[u], g, key0 + 8 * g, q0[u] + c + 1,
                                        key0 + 31 <= q0[u]);
        }
      }
      {
        // V operands by transpose reads: in lane group g (keys 8g .. 8g + 7) lane 4r + q points at key
        // 8g + 4h + r, dimensions 16e + 4q .. 16e + 4q + 3 (h = 0, 1), and ds_read_b64_tr_b16 hands lane c the
        // four keys' dimension 16e + c: block e's B operand, output column c = dimension 16e + c.
        const int rr = c >> 2, q4 = c & 3;
        const lds_char* vls = (const lds_char*)vl;  // vl points into LDS
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int off = (8 * g + rr) * kPfRow + (16 * e + 4 * q4) * 2;
          const v4i16_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(vls + off));
          const v4i16_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(vls + off + 4 * kPfRow));
          u32x4_t bop;
          bop[0] = (uint32_t)(uint16_t)lo[0] | ((uint32_t)(uint16_t)lo[1] << 16);
          bop[1] = (uint32_t)(uint16_t)lo[2] | ((uint32_t)(uint16_t)lo[3] << 16);
          bop[2] = (uint32_t)(uint16_t)hi[0] | ((uint32_t)(uint16_t)hi[1] << 16);
          bop[3] = (uint32_t)(uint16_t)hi[2] | ((uint32_t)(uint16_t)hi[3] << 16);
#pragma unroll
          for (int u = 0; u < kPfSub; ++u) {
            if (!act[u]) continue;
            o[u][e] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, pop[u]),
                                                              __builtin_bit_cast(bf16x8_t, bop), o[u][e], 0, 0, 0);
          }
        }
      }
    }
    }
    put((t + 1) & 1);
    __syncthreads();
  }

  // ---- each group's 16 output rows: O / l, rounded to bf16
#pragma unroll
  for (int u = 0; u < kPfSub; ++u) {
    float l_tot = st[u].l_run + __shfl_xor(st[u].l_run, 16, kWave);
    l_tot += __shfl_xor(l_tot, 32, kWave);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float li = __shfl(l_tot, 4 * g + i, kWave);
      const int qq = q0[u] + 4 * g + i;
      if (qq >= a.width) continue;
      const float div = li > 0.f ? li : 1.f;
      uint16_t* orow = a.out + ((int64_t)(b * a.width + qq) * a.H + h) * D;
#pragma unroll
      for (int e = 0; e < 8; ++e) orow[16 * e + c] = (uint16_t)pack_bf16x2(o[u][e][i] / div, 0.f);  // dim 16e + c
    }
  }
}

}  // namespace omni

extern "C" int omni_prefill_attention(const void* q, const void* k_cache, const void* v_cache, int64_t stride_row,
                                      int64_t stride_head, int64_t stride_pos, int64_t cache_len,
                                      int64_t cache_rows, const int64_t* slots, int32_t contexts, int32_t width,
                                      int32_t heads, int32_t head_dim, float scale, void* out, int32_t dtype,
                                      void* stream) {
  if (contexts < 0 || width < 0 || heads <= 0 || cache_rows <= 0) return OMNI_ERR_INVALID;
  if (dtype != OMNI_BF16) return OMNI_ERR_DTYPE;
  if ((head_dim != 128 && head_dim != 256 && head_dim != 512) || stride_pos != head_dim) return OMNI_ERR_SHAPE;
  if (!(scale > 0.f) || width > cache_len) return OMNI_ERR_INVALID;
  if (contexts == 0 || width == 0) return OMNI_OK;
  if (!q || !k_cache || !v_cache || !slots || !out) return OMNI_ERR_INVALID;
  if (((uintptr_t)q | (uintptr_t)out | (uintptr_t)k_cache | (uintptr_t)v_cache) & 15u) return OMNI_ERR_INVALID;
  if ((stride_row | stride_head) % 8 != 0) return OMNI_ERR_INVALID;
  if ((int64_t)contexts * width * heads >= (int64_t{1} << 31) / head_dim) return OMNI_ERR_INVALID;
  omni::PrefillArgs a;
  a.q = (const uint16_t*)q;
  a.k = (const uint16_t*)k_cache;
  a.v = (const uint16_t*)v_cache;
  a.slots = slots;
  a.s_row = stride_row;
  a.s_head = stride_head;
  a.cache_rows = cache_rows;
  a.width = width;
  a.H = heads;
  a.scale_log2 = scale * 1.4426950408889634f;
  a.out = (uint16_t*)out;
  hipStream_t s = (hipStream_t)stream;
  if (head_dim == 128) {
    if (omni::small_blocks(width, (int64_t)heads * contexts)) {
      dim3 grid((width + omni::kPfQueries - 1) / omni::kPfQueries, heads, contexts);
      omni::prefill_attn_kernel<<<grid, omni::kPfThreads, 0, s>>>(a);
    } else {
      dim3 grid((width + omni::kPairQ - 1) / omni::kPairQ, heads, contexts);
      omni::prefill_attn_pairs_kernel<<<grid, 512, 0, s>>>(a);
    }
  } else if (head_dim == 512) {
    const int nqb = (width + omni::kWsQ - 1) / omni::kWsQ, units = heads * contexts;
    dim3 grid(nqb, heads, contexts);
    a.units8 = units / 8;
    a.group = units % 8 == 0 ? omni::ws_group(nqb, a.units8) : 0;
    if (a.group) {
      omni::prefill_attn_ws_kernel<true><<<8 * omni::kWsPerXcd, 512, 0, s>>>(a);
    } else {
      omni::prefill_attn_ws_kernel<false><<<grid, 512, 0, s>>>(a);
    }
  } else {
    const int qw = 16 * omni::kPwSub * (omni::kPwWaves / 2);  // queries per workgroup
    dim3 grid((width + qw - 1) / qw, heads, contexts);
    omni::prefill_attn_wide_kernel<<<grid, 64 * omni::kPwWaves, 0, s>>>(a);
  }
  return omni_launch_status();
}
