// The beam search step's choice, for gfx950: each group's N best offers over its N rows x V tokens, from the LM
// head's log-probabilities or logits (src/omniasr_trt/beam.py:165-175):
//   logp  = the input itself (OMNI_SELECT_LOGP: torch's own F.log_softmax output, so the choice is the reference's
//           bit for bit), or (OMNI_SELECT_LOGITS) log_softmax(logits) per row computed here in the model's dtype
//           (bf16): fp32 max, fp32 sum of exp(x - max) in this kernel's own order, logsum = log(sum),
//           logp = bf16((x - max) - logsum) -- the arithmetic of torch's kernel but not its summation order, so a
//           logp on a bf16 rounding boundary can round the other way;
//   offer = score + logp, or with length_norm, once the group's row 0 has tokens, (score * count + logp) / (count + 1),
//           each operation rounded to fp32 in that order (torch's element-wise kernels, no fused multiply-add);
//           a finished row offers -inf everywhere except EOS, at its frozen score;
//   best, flat = offers.view(S, N * V).topk(N), sorted best first: ties in value go to the lower flat index
//           (torch.topk leaves the order of equal values unspecified).
//
// Layout: one 256-thread workgroup per row (the log-softmax needs the whole row; a row is ~20 KB, so one workgroup
// per row spreads the group's reads over N CUs): the row's max and sum are two workgroup reductions in a fixed order;
// each offer's value becomes a 32-bit number ordered as the choice is.  The N-th largest of a wave's threads' bests is a
// floor under the row's N best, so only the offers at or above the largest floor (few more than N) become 64-bit keys,
// value above inverted index, and wave 0 ranks them by counting.  What bounds it is that chain at one row's size, not the
// 20 KB: as N rounds of a 64-bit scan of all offers and a wave-wide maximum, at three levels, the launch took 18 us (now
// 11) at 8 groups x 5 beams x 10288; those rounds remain for rows with more than 256 offers at the floor (equal values).
// The row writes them through to the device's coherence point (the rows of a group run on different XCDs, whose L2s
// are not coherent) and takes the group's ticket; the last row of the group reads the N rows' lists and merges them
// into the group's N best.  Every selection is by (value, index), so the result does not depend on which row
// finishes last.
#include <limits.h>
#include <math.h>

#include "common.h"

namespace omni {

constexpr int kSelThreads = 256;
constexpr int kSelWaves = kSelThreads / kWave;
constexpr int kSelMaxBeams = 16;
constexpr int kSelCand = 256;  // candidates of a row in LDS (and the N x N keys of a group, at most 256)

// An offer and its flat index as one 64-bit key whose unsigned order is the choice's order: the value's bits mapped
// to an order-preserving unsigned integer (negative values bit-inverted, positive ones with the sign bit set; -0 as
// +0, so equal values stay equal) above the index inverted (a lower index is the larger key).  Keys are unique, and 0
// is below every offer's key, in its value half as in the whole.
__device__ __forceinline__ uint32_t sel_order(float v) {
  const uint32_t b = v == 0.f ? 0u : __float_as_uint(v);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ uint64_t sel_key(uint32_t order, int i) {
  return ((uint64_t)order << 32) | (uint64_t)(0xffffffffu - (uint32_t)i);
}
__device__ __forceinline__ float sel_value(uint64_t k) {
  const uint32_t u = (uint32_t)(k >> 32);
  return __uint_as_float((u & 0x80000000u) ? (u & 0x7fffffffu) : ~u);
}
__device__ __forceinline__ int64_t sel_index(uint64_t k) { return (int64_t)(0xffffffffu - (uint32_t)k); }

__device__ __forceinline__ uint64_t sel_wave_max(uint64_t k) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const uint32_t lo = __shfl_xor((uint32_t)k, o, kWave), hi = __shfl_xor((uint32_t)(k >> 32), o, kWave);
    const uint64_t ok = ((uint64_t)hi << 32) | lo;
    k = ok > k ? ok : k;
  }
  return k;
}

// The wave's largest 32-bit value, on the data-parallel lane moves (a cross-lane read through LDS takes ~10 times as
// long): within rows of 16 lanes, then across them; lanes without a source take 0.
template <int kCtrl>
__device__ __forceinline__ uint32_t sel_dpp_max(uint32_t v) {
  const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, kCtrl, 0xf, 0xf, false);
  return o > v ? o : v;
}
__device__ __forceinline__ uint32_t sel_wave_max32(uint32_t v) {
  v = sel_dpp_max<0x111>(v);  // row_shr 1, 2, 4, 8: lane 15 of each row holds the row's
  v = sel_dpp_max<0x112>(v);
  v = sel_dpp_max<0x114>(v);
  v = sel_dpp_max<0x118>(v);
  v = sel_dpp_max<0x142>(v);  // row_bcast 15, 31: lane 63 holds the wave's
  v = sel_dpp_max<0x143>(v);
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// keys[0 .. m) in LDS, unique: lanes' own keys (lane, lane + 64, ...) by rank; ``put(rank, key)`` for the n best.
template <typename Put>
__device__ __forceinline__ void sel_rank(const uint64_t* keys, int m, int n, Put put) {
  for (int i = lane_id(); i < m; i += kWave) {
    const uint64_t mine = keys[i];
    int rank = 0;
#pragma unroll 4
    for (int j = 0; j < m; ++j) rank += keys[j] > mine;
    if (rank < n) put(rank, mine);
  }
}

__device__ __forceinline__ float sel_block_reduce(float v, float* red, bool is_max) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const float ov = __shfl_xor(v, o, kWave);
    v = is_max ? fmaxf(v, ov) : v + ov;
  }
  if (lane_id() == 0) red[threadIdx.x / kWave] = v;
  __syncthreads();
  float t = red[0];
#pragma unroll
  for (int w = 1; w < kSelWaves; ++w) t = is_max ? fmaxf(t, red[w]) : t + red[w];  // the same order in every thread
  __syncthreads();
  return t;
}

struct SelectArgs {
  const uint16_t* logits;
  int64_t logits_stride;
  int beams, vocab;
  const float* score;
  const int64_t* count;
  const uint8_t* ended;
  int length_norm;
  int64_t eos;
  float* best;
  int64_t* flat;
  uint64_t* cand;  // [rows][beams] keys of each row's best, written through
  int* tickets;    // [groups], zero before and after
  int logp_in;     // 1: the input rows are log-probabilities already (no log-softmax here)
};

// CPT: 8-logit chunks per thread (V <= 8 x 256 x CPT).
template <int CPT>
__global__ __launch_bounds__(kSelThreads) void beam_select_kernel(SelectArgs a) {
#pragma clang fp contract(off)
  __shared__ float red[kSelWaves];
  __shared__ uint64_t cand[kSelCand];
  __shared__ uint32_t wave_floor[kSelWaves];
  __shared__ int n_cand;
  const int row = blockIdx.x, n = a.beams, V = a.vocab;
  const int g = row / n, b = row - g * n;
  const int tid = threadIdx.x, lane = lane_id(), wave = tid / kWave;
  const uint16_t* lr = a.logits + (int64_t)row * a.logits_stride;
  u32x4_t x[CPT];
#pragma unroll
  for (int c = 0; c < CPT; ++c) {
    const int ci = tid + c * kSelThreads;
    x[c] = ci * 8 < V ? *reinterpret_cast<const u32x4_t*>(lr + ci * 8) : u32x4_t{0u, 0u, 0u, 0u};
  }
  const float score = a.score[row];
  const int64_t cnt = a.count[row];
  const bool ended = a.ended[row] != 0;
  const bool norm = a.length_norm && a.count[(int64_t)g * n] > 0;

  float m = 0.f, logsum = 0.f;
  if (!a.logp_in) {  // block-uniform
    m = -INFINITY;
#pragma unroll
    for (int c = 0; c < CPT; ++c)
      if ((tid + c * kSelThreads) * 8 < V) {
#pragma unroll
        for (int e = 0; e < 8; ++e) m = fmaxf(m, bf16x8_elem(x[c], e));
      }
    m = sel_block_reduce(m, red, true);
    float sum = 0.f;
#pragma unroll
    for (int c = 0; c < CPT; ++c)
      if ((tid + c * kSelThreads) * 8 < V) {
#pragma unroll
        for (int e = 0; e < 8; ++e) sum += expf(bf16x8_elem(x[c], e) - m);
      }
    sum = sel_block_reduce(sum, red, false);
    logsum = logf(sum);
  }

  // The row's offers' orders (past V: 0, never chosen).
  uint32_t ord[CPT * 8];
  const float cf = (float)cnt, c1 = (float)(cnt + 1);
  uint32_t cur = 0;  // this thread's best
#pragma unroll
  for (int c = 0; c < CPT; ++c)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int v = (tid + c * kSelThreads) * 8 + e;
      const float lp = a.logp_in ? bf16x8_elem(x[c], e) : round_through_bf16((bf16x8_elem(x[c], e) - m) - logsum);
      float o;
      if (norm) {
        const float t = score * cf;
        o = (t + lp) / c1;
      } else {
        o = score + lp;
      }
      const uint32_t order = sel_order(o);
      ord[c * 8 + e] = v < V ? (order > 1u ? order : 1u) : 0u;
      cur = ord[c * 8 + e] > cur ? ord[c * 8 + e] : cur;
    }

  // The row's candidates, in LDS.  A finished row offers EOS at its score and -inf elsewhere: its N best are among EOS
  // and the first N + 1 tokens.  Otherwise n threads of a wave hold an offer of at least the n-th largest of the
  // threads' bests, so the row's N best are at or above the largest of the waves' N-th: few more than N unless values
  // tie.
  if (tid == 0) n_cand = 0;
  if (!ended) {  // block-uniform
    uint32_t floor_w = 0;
    for (int j = 0; j < n; ++j) {
      floor_w = sel_wave_max32(cur);
      const uint64_t at = __ballot(cur == floor_w);
      if (lane == __ffsll((unsigned long long)at) - 1) cur = 0;
    }
    if (lane == 0) wave_floor[wave] = floor_w;
  }
  __syncthreads();
  if (ended) {
    const int few = n + 1 < V ? n + 1 : V;
    if (tid < few) cand[tid] = sel_key(sel_order(tid == a.eos ? score : -INFINITY), b * V + tid);
    if (tid == 0) {
      const bool extra = a.eos >= few && a.eos < V;
      if (extra) cand[few] = sel_key(sel_order(score), b * V + (int)a.eos);
      n_cand = few + (extra ? 1 : 0);
    }
  } else {
    uint32_t least = wave_floor[0];
#pragma unroll
    for (int w = 1; w < kSelWaves; ++w) least = wave_floor[w] > least ? wave_floor[w] : least;
    least = least > 1u ? least : 1u;
#pragma unroll
    for (int i = 0; i < CPT * 8; ++i)
      if (ord[i] >= least) {
        const int at = __hip_atomic_fetch_add(&n_cand, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (at < kSelCand) cand[at] = sel_key(ord[i], b * V + (tid + (i >> 3) * kSelThreads) * 8 + (i & 7));
      }
  }
  __syncthreads();
  const int found = n_cand;  // block-uniform
  if (found > kSelCand) {  // many equal values: each wave's N best in N rounds, in the candidates' place
    __syncthreads();
    uint64_t prev = ~0ull, mine = 0;
    for (int j = 0; j < n; ++j) {
      uint64_t best = 0;
#pragma unroll
      for (int i = 0; i < CPT * 8; ++i) {
        const uint64_t k = ord[i] ? sel_key(ord[i], b * V + (tid + (i >> 3) * kSelThreads) * 8 + (i & 7)) : 0ull;
        best = k < prev && k > best ? k : best;
      }
      best = sel_wave_max(best);
      if (lane == j) mine = best;
      prev = best;
    }
    if (lane < n) cand[wave * n + lane] = mine;
    __syncthreads();
  }
  if (wave != 0) return;
  const int have = found > kSelCand ? kSelWaves * n : found;

  // The row's list, written through; then the group's ticket.
  uint64_t* crow = a.cand + (int64_t)row * n;
  sel_rank(cand, have, n, [&](int rank, uint64_t k) {
    __hip_atomic_store(crow + rank, k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  });
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0);
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  int ticket = 0;
  if (lane == 0) ticket = __hip_atomic_fetch_add(a.tickets + g, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  ticket = __shfl(ticket, 0, kWave);
  if (ticket != n - 1) return;

  // The group's last row: the N lists (N x N <= 256 keys, read at the coherence point), merged.
  const uint64_t* cg = a.cand + (int64_t)g * n * n;
  uint64_t gk[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int f = lane + q * kWave;
    gk[q] = __hip_atomic_load(cg + (f < n * n ? f : 0), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
#pragma unroll
  for (int q = 0; q < 4; ++q)
    if (lane + q * kWave < n * n) cand[lane + q * kWave] = gk[q];
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");  // this wave's own reads follow
  __builtin_amdgcn_s_waitcnt(0xc07f);                              // lgkmcnt(0): the keys are in LDS
  sel_rank(cand, n * n, n, [&](int rank, uint64_t k) {
    a.best[(int64_t)g * n + rank] = sel_value(k);
    a.flat[(int64_t)g * n + rank] = sel_index(k);
  });
  if (lane == 0) __hip_atomic_store(a.tickets + g, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace omni

extern "C" size_t omni_beam_select_workspace(int32_t groups, int32_t beams) {
  if (groups <= 0 || beams <= 0) return 0;
  return (size_t)groups * beams * beams * sizeof(uint64_t);
}

extern "C" int omni_beam_select(const void* logits, int64_t logits_stride, int32_t groups, int32_t beams,
                                int32_t vocab, const float* score, const int64_t* count, const uint8_t* ended,
                                int32_t length_norm, int64_t eos, float* best, int64_t* flat, void* workspace,
                                size_t workspace_bytes, int32_t* tickets, int32_t input_kind, int32_t dtype,
                                void* stream) {
  if (dtype != OMNI_BF16) return OMNI_ERR_DTYPE;
  if (input_kind != OMNI_SELECT_LOGP && input_kind != OMNI_SELECT_LOGITS) return OMNI_ERR_INVALID;
  if (groups < 0 || beams < 1 || beams > omni::kSelMaxBeams || vocab < beams) return OMNI_ERR_INVALID;
  if (vocab % 8 != 0 || vocab > 8 * omni::kSelThreads * 8) return OMNI_ERR_SHAPE;
  if (groups == 0) return OMNI_OK;
  if ((int64_t)beams * vocab >= INT_MAX) return OMNI_ERR_SHAPE;
  if (!logits || !score || !count || !ended || !best || !flat || !tickets || logits_stride < vocab ||
      logits_stride % 8)
    return OMNI_ERR_INVALID;
  if (!workspace || workspace_bytes < omni_beam_select_workspace(groups, beams)) return OMNI_ERR_WORKSPACE;
  omni::SelectArgs a{static_cast<const uint16_t*>(logits), logits_stride, beams, vocab, score, count, ended,
                     length_norm, eos, best, flat, static_cast<uint64_t*>(workspace), tickets,
                     input_kind == OMNI_SELECT_LOGP ? 1 : 0};
  const int rows = groups * beams, cpt = (vocab / 8 + omni::kSelThreads - 1) / omni::kSelThreads;
  hipStream_t s = (hipStream_t)stream;
  if (cpt <= 2)
    omni::beam_select_kernel<2><<<rows, omni::kSelThreads, 0, s>>>(a);
  else if (cpt <= 4)
    omni::beam_select_kernel<4><<<rows, omni::kSelThreads, 0, s>>>(a);
  else if (cpt <= 6)
    omni::beam_select_kernel<6><<<rows, omni::kSelThreads, 0, s>>>(a);
  else
    omni::beam_select_kernel<8><<<rows, omni::kSelThreads, 0, s>>>(a);
  return omni_launch_status();
}
