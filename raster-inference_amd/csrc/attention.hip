// Causal prefill attention on int8 MFMA (det_attention_prefill,
// det_kernels.rs:575-651): the q.k and weight.v products of every (head,
// query) row exactly, as wrapping int64 sums, from int8 limb products.
//
// An int32 x is split into signed bytes with an offset, three where its whole
// group fits 24 bits and four otherwise:
//   x = c0 + 256 c1 + 65536 c2 + C3,               C3 = 32896    (x in [-2^23, 2^23)),
//   x = c0 + 256 c1 + 65536 c2 + 2^24 c3 + C4,     C4 = 8421504,
// c_j the signed bytes of (x + 2^23) ^ 0x808080 or of x ^ 0x808080. The groups
// are one row of Q or K (its head dims), and 64 keys x 256 dims of V. A softmax weight w
// lies in [0, 65536]; only the first argmax row can hold 65536 (every other
// weight is at most half), so w is split as two bytes of w ^ 0x8080 plus 32896
// with that row clamped to 65535, and the clamped unit goes with the residual
// into one extra product extra * v[argmax]. With x' = x - C (C the group's
// offset, C_q and C_k below those of the two rows):
//   sum_d q_d k_d = sum_{i,j} 256^(i+j) sum_d c_i(q_d) c_j(k_d)
//                   + C_q sum_d k_d + C_k sum_d q'_d,
//   sum_r w_r v_r = sum_{i,j} 256^(i+j) sum_r a_i(w_r) c_j(v_r)
//                   + 32896 sum_r v'_r + sum_r C_v(r) w_r + extra v[argmax]
// in wrapping int64. The limb products with the same i + j share one int32
// MFMA accumulator: at most four pairs of 128 x 128 over at most 512 head
// dims (q.k), two pairs over at most 16000 keys (weight.v), both below 2^31.
// Normalised rows take three limbs, so a (query, key) pair costs 9 + 6
// products of one byte each per head dim (16 + 12 with four limbs of
// everything and three of the weights).
//
// Pipeline: limb tiles of Q, of K and of V (transposed, dims x keys) with
// their offset sums; then, in chunks of queries whose score rows stay within
// kScoreBytes (half the Infinity Cache, and what bounds the work area): the
// scores of every (head, query, key in the window), the softmax of every row
// in place, the weighted sums.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "det_arith.h"
#include "kernels.h"
#include "wave.h"

namespace det {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int64_t kC4 = kAttnC4;   // offset of the four-limb split
constexpr int64_t kC3 = kAttnC3;   // offset of the three-limb split and of the weights
constexpr uint32_t kOp = kAttnOp;  // one MFMA operand block: 64 lanes x 16 bytes

// Query rows t in [0, n_queries) attend to keys [start_t, end_t).
struct AttnRange {
  uint64_t start, end;
};
__device__ inline AttnRange attn_range(const AttnMfmaArgs& a, uint64_t t) {
  uint64_t end = t + 1 + a.causal_offset;
  uint64_t start = (a.window && end > a.window) ? end - a.window : 0;
  if (start > a.avail) start = a.avail;
  if (end > a.avail) end = a.avail;
  return {start, end > start ? end : start};
}

// The first key of the score rows of the 32 queries around t: the 64-key
// substep of their union window's start (a score row holds keys from there on).
__device__ inline uint64_t score_base(const AttnMfmaArgs& a, uint64_t t) {
  return attn_range(a, t & ~uint64_t(31)).start & ~uint64_t(63);
}

// 16 int32 -> four 16-byte limb vectors and the sum of x - C
__device__ inline int64_t split4(const int32_t (&x)[16], bool wide, v4i (&limb)[4]) {
  uint32_t w[4][4];
  const int64_t s = attn_split16(x, wide, w);
#pragma unroll
  for (int j = 0; j < 4; ++j) limb[j] = v4i{int(w[j][0]), int(w[j][1]), int(w[j][2]), int(w[j][3])};
  return s;
}

// Q or K rows to limb blocks. Block (row tile T, substep s, limb j) at
// ((T * nsub + s) * 4 + j) * kOp: lane l holds row 16 T + (l & 15), dims
// [64 s + 16 (l >> 4), +16) (limb 3 of a narrow row is zero). One wave per
// substep; sums[row] = attn_pack_sum of the row. Rows
// past n take zero limbs and a zero sum. One launch for both matrices: blocks
// of Q's heads, then of K's. grid (heads, most tiles), block 64 * nsub.
struct SplitRows {
  const int32_t* x;
  uint64_t ld, n, ntiles;
  int8_t* limbs;
  int64_t* sums;
  uint32_t heads;  // 0: the rows' producer has written these
};
__global__ __launch_bounds__(512) void k_attn_split_rows(SplitRows q, SplitRows k, uint32_t hd) {
  __shared__ int64_t part[8][16];
  __shared__ uint32_t wide16[8];  // bit i: row i has a wide value in the wave's dims
  const bool is_q = blockIdx.x < q.heads;
  const uint32_t h = is_q ? blockIdx.x : blockIdx.x - q.heads, T = blockIdx.y;
  const uint64_t ld = is_q ? q.ld : k.ld, n = is_q ? q.n : k.n, ntiles = is_q ? q.ntiles : k.ntiles;
  const int32_t* __restrict__ x = is_q ? q.x : k.x;
  int8_t* __restrict__ limbs = is_q ? q.limbs : k.limbs;
  int64_t* __restrict__ sums = is_q ? q.sums : k.sums;
  if (T >= ntiles) return;  // (workgroup-uniform)
  const uint32_t s = threadIdx.x >> 6, l = threadIdx.x & 63;
  const uint32_t nsub = hd / 64;
  const uint64_t row = uint64_t(T) * 16 + (l & 15);
  const uint32_t d0 = 64 * s + 16 * (l >> 4);
  int32_t v[16];
  if (row < n) {
    const int4* p = reinterpret_cast<const int4*>(x + row * ld + uint64_t(h) * hd + d0);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int4 t = p[q];
      v[4 * q] = t.x, v[4 * q + 1] = t.y, v[4 * q + 2] = t.z, v[4 * q + 3] = t.w;
    }
  } else {
#pragma unroll
    for (int e = 0; e < 16; ++e) v[e] = int32_t(kC3);
  }
  const uint64_t wb = __ballot(attn_wide16(v));
  if (l == 0) wide16[s] = uint32_t((wb | (wb >> 16) | (wb >> 32) | (wb >> 48)) & 0xffffu);
  __syncthreads();
  uint32_t wm = 0;
  for (uint32_t q = 0; q < nsub; ++q) wm |= wide16[q];
  const bool wide = (wm >> (l & 15)) & 1u;
  v4i limb[4];
  int64_t sm = split4(v, wide, limb);
  int8_t* blk = limbs + ((uint64_t(h) * ntiles + T) * nsub + s) * 4 * kOp + l * 16;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    *reinterpret_cast<v4i*>(blk + j * kOp) = limb[j];
  // the four lane groups of a row, then the substeps
  sm += __shfl_xor(sm, 16, 64);
  sm += __shfl_xor(sm, 32, 64);
  if (l < 16) part[s][l] = sm;
  __syncthreads();
  if (threadIdx.x < 16) {
    int64_t t = 0;
    for (uint32_t q = 0; q < nsub; ++q) t += part[q][threadIdx.x];
    sums[uint64_t(h) * ntiles * 16 + uint64_t(T) * 16 + threadIdx.x] = attn_pack_sum(t, (wm >> threadIdx.x) & 1u);
  }
}

// V to transposed limb blocks: block (dim tile D, key substep ks, limb j) at
// ((D * nks + ks) * 4 + j) * kOp: lane l holds dim 16 D + (l & 15), keys
// [64 ks + 16 (l >> 4), +16) (keys past avail have zero limbs). The substep's
// 256 dims of grid z take four limbs (vwide[(kvh * gridDim.z + z) * nks + ks]
// = 1) when any of their values needs them. vblk[ks][dim] = sum over the
// substep's keys of v - C. grid (kv heads, nks, ceil(hd / 256)), a wave per dim
// tile, block 64 * min(hd / 16, 16).
__global__ __launch_bounds__(1024) void k_attn_split_v(const int32_t* __restrict__ v, uint64_t ld, uint64_t avail,
                                                       uint32_t hd, uint64_t nks, int8_t* __restrict__ limbs,
                                                       int64_t* __restrict__ vblk, uint32_t* __restrict__ vwide) {
  const uint32_t kvh = blockIdx.x, ks = blockIdx.y, l = threadIdx.x & 63;
  const uint32_t ndt = hd / 16, D = blockIdx.z * 16 + (threadIdx.x >> 6);
  const uint64_t k0 = uint64_t(ks) * 64 + 16 * (l >> 4);
  const bool on = D < ndt;  // (wave-uniform)
  const uint32_t dim = 16 * (on ? D : ndt - 1) + (l & 15);
  int32_t x[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    const uint64_t r = k0 + e;
    x[e] = (on && r < avail) ? v[r * ld + uint64_t(kvh) * hd + dim] : 0;
  }
  const bool wide = __syncthreads_or(attn_wide16(x)) != 0;
  if (threadIdx.x == 0) vwide[(uint64_t(kvh) * gridDim.z + blockIdx.z) * nks + ks] = wide;
  if (!on) return;
#pragma unroll
  for (int e = 0; e < 16; ++e)
    if (k0 + e >= avail) x[e] = int32_t(wide ? kC4 : kC3);
  v4i limb[4];
  int64_t sm = split4(x, wide, limb);
  int8_t* blk = limbs + ((uint64_t(kvh) * ndt + D) * nks + ks) * 4 * kOp + l * 16;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (j < 3 || wide) *reinterpret_cast<v4i*>(blk + j * kOp) = limb[j];
  sm += __shfl_xor(sm, 16, 64);
  sm += __shfl_xor(sm, 32, 64);
  if (l < 16) vblk[(uint64_t(kvh) * nks + ks) * hd + dim] = sm;
}

// Ring of LDS stages filled by global_load_lds copies: a wave waits for its own
// copies of the stage it is about to use (copies complete in issue order; N may
// stay outstanding) and for its LDS reads, and a bare barrier then makes every wave's visible and
// leaves the later stages' copies in flight.
template <int N>
__device__ __forceinline__ void ring_barrier(bool more) {
  static_assert(N < 64, "vmcnt range");
  asm volatile("" ::: "memory");
  if (more) __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | ((N >> 4) << 14));
  else __builtin_amdgcn_s_waitcnt(7 << 4);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
// One 1 KB copy: 16 bytes per lane from src (per lane) to dst + 16 lane.
__device__ __forceinline__ void ring_copy(const int8_t* src, int8_t* dst) {
  __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)src,
                                   (void __attribute__((address_space(3)))*)dst, 16, 0, 0);
}

// Scores of 16 queries (limb operands in registers) against one key tile in
// LDS: lane l holds, in component r, key 16 J + 4 (l >> 4) + r and query
// 16 T + (l & 15), so each lane stores four consecutive keys of one query. NL
// limbs of both operands; the offsets of a row are those of its own split.
template <int NSUB, int NL>
__device__ __forceinline__ void score_tile(const v4i (&q)[NSUB][NL], const v4i* kt, uint32_t l, int64_t qpack,
                                           const int64_t* kpack, int32_t* dst, bool on) {
  v4i acc[2 * NL - 1];
#pragma unroll
  for (int s = 0; s < 2 * NL - 1; ++s) acc[s] = v4i{0, 0, 0, 0};
#pragma unroll
  for (int s = 0; s < NSUB; ++s)
#pragma unroll
    for (int j = 0; j < NL; ++j) {
      const v4i k = kt[(s * NL + j) * 64 + l];
#pragma unroll
      for (int i = 0; i < NL; ++i) acc[i + j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(k, q[s][i], acc[i + j], 0, 0, 0);
    }
  const uint64_t qs = uint64_t(qpack >> 1), cq = (qpack & 1) ? uint64_t(kC4) : uint64_t(kC3);
  int32_t out[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int64_t kp = kpack[4 * (l >> 4) + r];
    const uint64_t ksp = uint64_t(kp >> 1);
    uint64_t dot;
    if constexpr (NL == 3) {
      dot = uint64_t(kC3) * (ksp + qs + uint64_t(NSUB * 64) * uint64_t(kC3));
    } else {
      const uint64_t ck = (kp & 1) ? uint64_t(kC4) : uint64_t(kC3);
      dot = cq * (ksp + uint64_t(NSUB * 64) * ck) + ck * qs;
    }
#pragma unroll
    for (int s = 0; s < 2 * NL - 1; ++s) dot += uint64_t(int64_t(acc[s][r])) << (8 * s);
    out[r] = requant(int64_t(dot));
  }
  if (on) *reinterpret_cast<int4*>(dst) = make_int4(out[0], out[1], out[2], out[3]);
}

// Scores: block (kv head, NW weight-stationary tiles of 16 queries x one of
// the G heads, span of key tiles from the first one its queries attend to).
// Wave w keeps the limb operands of head w % G, query tile w / G in registers
// and multiplies every key tile of the span with them; the key tiles (3 or 4
// KB per 64 head dims) stream through a ring of four LDS stages of KS tiles,
// so each is read once per block for all its rows, and no wave waits for its
// own operands. (Key tiles held in registers and queries in LDS, each wave
// loading its own key tiles, left the loads exposed: 1643 queries, 8 heads of
// 256, 65 us.) A block all of whose rows take three limbs reads and multiplies
// no fourth one. A tile of 16 x 16 that touches the query tile's union window
// is written whole; the softmax drops the positions outside a query's window.
// grid (kv heads, groups of NW / G query tiles, spans), block 64 NW.
constexpr int kScoreStages = 4;
constexpr uint32_t kScoreSpan = 64;  // most key tiles per block
template <int NSUB, int NW, int NL>
__device__ __forceinline__ void score_block(const AttnMfmaArgs& a, int8_t* ring, const int64_t* kpk, uint32_t kvh,
                                            uint32_t h, uint32_t hq, uint64_t t_lo, uint64_t tc, bool q_on,
                                            uint64_t j0, uint64_t j1, uint32_t l, uint32_t wave) {
  asm volatile("" : "+v"(l));  // (the two forms' addresses, computed ahead of the choice, would spill)
  constexpr int KS = NSUB == 1 ? 4 : (NSUB == 2 ? 2 : 1);  // key tiles per stage
  constexpr int SLOTS = KS * NSUB * NL, LPW = (SLOTS + NW - 1) / NW;
  const uint64_t t_end = a.t0 + a.crow_used, t = t_lo + (l & 15);
  const uint32_t ntile = uint32_t(j1 - j0), nst = (ntile + KS - 1) / KS;
  const int8_t* kb = a.klimbs + uint64_t(kvh) * a.nkt * NSUB * 4 * kOp;  // (wave-uniform)
  auto copy_stage = [&](uint32_t st) {
#pragma unroll
    for (int u = 0; u < LPW; ++u) {
      uint32_t c = wave * LPW + u;
      if (c >= uint32_t(SLOTS)) c = SLOTS - 1;  // (spare slots copy the last block again)
      uint64_t J = j0 + uint64_t(st) * KS + c / (NSUB * NL);
      if (J >= j1) J = j1 - 1;
      ring_copy(kb + ((J * NSUB + c / NL % NSUB) * 4 + c % NL) * kOp + l * 16,
                ring + ((st % kScoreStages) * SLOTS + c) * kOp);
    }
  };
  copy_stage(0);
  const uint64_t T = tc / 16;
  const int64_t qpack = a.qsum[uint64_t(hq) * a.nqt * 16 + T * 16 + (l & 15)];
  const int8_t* qb = a.qlimbs + (uint64_t(hq) * a.nqt + T) * NSUB * 4 * kOp;  // (wave-uniform)
  v4i q[NSUB][NL];
#pragma unroll
  for (int s = 0; s < NSUB; ++s)
#pragma unroll
    for (int i = 0; i < NL; ++i) q[s][i] = *reinterpret_cast<const v4i*>(qb + (s * 4 + i) * kOp + l * 16);
#pragma unroll
  for (int p = 1; p < kScoreStages - 1; ++p)
    if (uint32_t(p) < nst) copy_stage(p);
  const uint64_t kmin = attn_range(a, tc).start, kmax = attn_range(a, tc + 15 < t_end ? tc + 15 : t_end - 1).end;
  int32_t* row = a.scores + (uint64_t(h) * a.crow + (t - a.t0)) * a.srow + 4 * (l >> 4);
  const uint64_t kbase = score_base(a, tc);
  const bool on = q_on && t < t_end;
  for (uint32_t st = 0; st < nst; ++st) {
    ring_barrier<(kScoreStages - 2) * LPW>(st + kScoreStages - 1 <= nst);
    if (st + kScoreStages - 1 < nst) copy_stage(st + kScoreStages - 1);
    const v4i* base = reinterpret_cast<const v4i*>(ring + (st % kScoreStages) * SLOTS * kOp);
#pragma unroll
    for (int u = 0; u < KS; ++u) {
      const uint32_t jl = st * KS + u;
      const uint64_t key0 = (j0 + jl) * 16;
      if (!q_on || jl >= ntile || key0 >= kmax || key0 + 16 <= kmin) continue;  // (wave-uniform)
      score_tile<NSUB, NL>(q, base + u * NSUB * NL * 64, l, qpack, kpk + jl * 16, row + (key0 - kbase), on);
    }
  }
}
template <int NSUB, int NW>
__global__ __launch_bounds__(64 * NW, NSUB <= 4 ? 4 : 2) void k_attn_scores_mfma(AttnMfmaArgs a, uint32_t span) {
  extern __shared__ __attribute__((aligned(16))) int8_t ring[];  // [stage][key tile][substep][limb][lane]
  __shared__ int64_t kpk[kScoreSpan * 16];
  const uint32_t l = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t kvh = blockIdx.x, G = a.groups, QT = NW / G;
  const uint64_t t_end = a.t0 + a.crow_used;
  // the block's keys: its share of the union window of its queries
  const uint64_t tb = a.t0 + uint64_t(blockIdx.y) * 16 * QT;
  const uint64_t tb_hi = tb + 16 * QT < t_end ? tb + 16 * QT - 1 : t_end - 1;
  const uint64_t j0 = attn_range(a, tb).start / 16 + uint64_t(blockIdx.z) * span;
  uint64_t j1 = (attn_range(a, tb_hi).end + 15) / 16;
  j1 = j1 < j0 + span ? j1 : j0 + span;
  if (j0 >= j1) return;  // (workgroup-uniform)
  // this wave's queries
  const uint32_t h = kvh * G + wave % G;
  const uint64_t t_lo = tb + 16 * (wave / G);
  const bool q_on = wave < G * QT && t_lo < t_end;  // (wave-uniform)
  const uint64_t tc = q_on ? t_lo : tb;
  const uint32_t hq = q_on ? h : kvh * G;
  bool wl = a.qsum[uint64_t(hq) * a.nqt * 16 + (tc & ~uint64_t(15)) + (l & 15)] & 1;
  const uint32_t ntile = uint32_t(j1 - j0);
  for (uint32_t i = threadIdx.x; i < ntile * 16; i += 64 * NW) {
    const int64_t kp = a.ksum[(uint64_t(kvh) * a.nkt + j0) * 16 + i];
    kpk[i] = kp;
    wl = wl || (kp & 1);
  }
  const bool wide = __syncthreads_or(wl) != 0;  // (no load is outstanding from here on)
  if (wide) score_block<NSUB, NW, 4>(a, ring, kpk, kvh, h, hq, t_lo, tc, q_on, j0, j1, l, wave);
  else score_block<NSUB, NW, 3>(a, ring, kpk, kvh, h, hq, t_lo, tc, q_on, j0, j1, l, wave);
}

template <int NSUB, int NW>
void launch_scores_nw(const AttnMfmaArgs& m, uint64_t nkv, hipStream_t s) {
  constexpr int KS = NSUB == 1 ? 4 : (NSUB == 2 ? 2 : 1);
  constexpr uint32_t lds = kScoreStages * KS * NSUB * 4 * kOp;
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_attn_scores_mfma<NSUB, NW>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  (void)attr;
  const uint64_t rows = 16 * (NW / m.groups), y = (m.crow_used + rows - 1) / rows;
  // key tiles of the query blocks' union windows: the most of one block, and all
  auto tiles = [&](uint64_t b) {
    const uint64_t lo = m.t0 + b * rows, hi = std::min(lo + rows, m.t0 + m.crow_used);  // queries [lo, hi)
    const uint64_t end = std::min(hi + m.causal_offset, m.avail);
    const uint64_t start = m.window && lo + 1 + m.causal_offset > m.window ? lo + 1 + m.causal_offset - m.window : 0;
    return end > start ? (end + 15) / 16 - start / 16 : 0;
  };
  uint64_t most = 0, all = 0;
  for (uint64_t b = 0; b < y; ++b) {
    const uint64_t n = tiles(b);
    most = std::max(most, n);
    all += nkv * n;
  }
  uint32_t span = kScoreSpan;
  // Spans short enough for two blocks per CU up to 256 head dims (their ring
  // and registers leave room for two) and one block on every other CU beyond
  // (128 KB of ring, 32 KB of query operands per wave to load first). Never
  // less than eight tiles left 100 queries of 4 heads of 512 on four blocks:
  // 17.0 us, now 6.8; 8/2 heads of 256 at 300 queries 15.8 -> 7.4.
  constexpr uint64_t want = NSUB <= 4 ? 512 : 128;
  while (span > 1 && all < want * span) span /= 2;
  const dim3 grid(unsigned(nkv), unsigned(y), unsigned(std::max<uint64_t>((most + span - 1) / span, 1)));
  hipLaunchKernelGGL((k_attn_scores_mfma<NSUB, NW>), grid, dim3(64 * NW), lds, s, m, span);
}
template <int NSUB>
void launch_scores_nsub(const AttnMfmaArgs& m, uint64_t nkv, hipStream_t s) {
  if (m.groups == 3) launch_scores_nw<NSUB, 6>(m, nkv, s);
  else launch_scores_nw<NSUB, 8>(m, nkv, s);
}

// Softmax of every (head, query) row of the chunk: the first argmax, the exp
// sum, the weights. The weights replace the scores in place as 16-bit values
// w ^ 0x8080 at the start of the row (the r-th key at byte 2 r), zero outside
// the window, over the 64-key substeps of the union window of the 32 queries
// that share a score row's first key. A row's scores, then its exp terms, are
// kept in LDS, so that the three passes are rolled loops (unrolled over
// registers they were 66 to 130 KB of code, more than the instruction cache of
// two CUs: 46 us against now 38 for 1000 rows of 16 heads in windows of 512). Terms 16 or more below the
// maximum are zero exactly, and 64 keys that have only such terms skip the exp
// series and the weights (rows of 256 normalised dims have scores of standard
// deviation 16).
// wtot: the row's weights' sum; extra: what the first argmax row holds past
// its (clamped) 16-bit weight, the residual included.
struct RowSpan {
  uint64_t k0;    // the score row's first key
  uint32_t n;     // keys of the row
  uint32_t w0, w1;  // the window, relative to k0
};
__device__ inline RowSpan row_span(const AttnMfmaArgs& a, uint64_t t) {
  const AttnRange w = attn_range(a, t);
  const uint64_t p_hi = (t | 31) < a.n_queries ? (t | 31) : a.n_queries - 1;
  const uint64_t K0 = score_base(a, t), K1 = (attn_range(a, p_hi).end + 63) & ~uint64_t(63);
  return {K0, uint32_t(K1 - K0), uint32_t(w.start - K0), uint32_t(w.end - K0)};
}
// An exp term (at most 2^32, and otherwise below 2^32 - 65000) in 32 bits, all ones for 2^32.
__device__ inline uint32_t pack_term(int64_t v) { return v >> 32 ? 0xffffffffu : uint32_t(v); }
__device__ inline int64_t unpack_term(uint32_t e) { return int64_t(uint64_t(e) + (e == 0xffffffffu)); }
// A term's weight, clamped to 16 bits (only the first argmax row's is 65536);
// `total` adds the unclamped one. (sum is at least 2^32, the maximum's term,
// and below 2^61: at most 16000 rows.)
__device__ inline uint32_t term_weight(uint32_t e, int64_t sum, uint64_t M, int64_t& total) {
  const int32_t w = softmax_weight_r(unpack_term(e), sum, M);
  total += w;
  return uint32_t(w > 65535 ? 65535 : w);
}
// The row's extras: the first argmax row's weight (its exp term is that of gap
// 0) and the residual, added to it with saturation.
__device__ inline void put_row_extras(const AttnMfmaArgs& a, uint32_t h, uint64_t t, bool on, int64_t ws, int64_t sum,
                                      uint64_t M, uint64_t argmax) {
  const uint64_t o = uint64_t(h) * a.n_queries + t;
  const int32_t wm = on ? softmax_weight_r(int64_t(1) << 32, sum, M) : 0;
  const int32_t res = sub_sat(kOneAct, sat32(ws)), kept = wm > 65535 ? 65535 : wm;
  a.extra[o] = on ? add_sat(wm, res) - kept : 0;
  a.argm[o] = on ? uint32_t(argmax) : 0;
  a.wtot[o] = uint32_t(ws - (wm - kept));
}

// Windows of at most kSoftmaxShort keys: one wave per row, one key per lane and
// step, from the window's own first key on (steps over the union window were a
// quarter more at 512 keys). grid (heads, ceil(chunk rows / 4)), block 256.
constexpr uint32_t kSoftmaxShort = 1024;
__global__ __launch_bounds__(256) void k_attn_softmax_short(AttnMfmaArgs a) {
  __shared__ uint32_t row[4][kSoftmaxShort];
  const uint32_t h = blockIdx.x, l = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint64_t t = a.t0 + uint64_t(blockIdx.y) * 4 + wave;
  if (t >= a.t0 + a.crow_used) return;
  const RowSpan s = row_span(a, t);
  const uint32_t cnt = s.w1 - s.w0, steps = (cnt + 63) / 64;
  int32_t* srow = a.scores + (uint64_t(h) * a.crow + (t - a.t0)) * a.srow;
  const int32_t* src = srow + s.w0;
  uint16_t* wrow = reinterpret_cast<uint16_t*>(srow);
  uint32_t* x = row[wave];
  int32_t mxl = INT32_MIN;
#pragma unroll 4
  for (uint32_t c = 0; c < steps; ++c) {
    const uint32_t r = 64 * c + l;
    const int32_t v = src[r < cnt ? r : cnt - 1];
    x[r] = uint32_t(v);
    mxl = v > mxl ? v : mxl;
  }
  const int32_t mx = int32_t(wave_max64(mxl));
  uint32_t mi = 0xffffffffu;  // the first argmax (wave-uniform)
  int64_t sum = 0;            // (below 2^63)
  for (uint32_t c = 0; c < steps; ++c) {
    const uint32_t r = 64 * c + l;
    const int32_t v = int32_t(x[r]);
    const uint32_t gap = r < cnt ? uint32_t(mx) - uint32_t(v) : 0xffffffffu;  // (mx >= v)
    uint32_t e = 0;
    if (__any(gap < (1u << 20))) {
      const uint64_t top = __ballot(gap == 0);
      if (mi == 0xffffffffu && top) mi = 64 * c + uint32_t(__builtin_ctzll(top));
      const int64_t term = gap < (1u << 20) ? softmax_exp(v, mx) : 0;
      sum += term;
      e = pack_term(term);
    }
    x[r] = e;
  }
  sum = wave_sum_wrap64(sum);
  const uint64_t M = cnt ? softmax_recip(sum) : 0;
  int64_t ws = 0;
  for (uint32_t c = 0; c < steps; ++c) {
    const uint32_t r = 64 * c + l, e = x[r];
    uint32_t w = 0;
    if (__any(e)) w = term_weight(e, sum, M, ws);
    if (r < cnt) wrow[s.w0 + r] = uint16_t(w ^ 0x8080u);
  }
  for (uint32_t k = l; k < s.w0; k += 64) wrow[k] = 0x8080u;
  for (uint32_t k = s.w1 + l; k < s.n; k += 64) wrow[k] = 0x8080u;
  ws = wave_sum_wrap64(ws);
  if (l == 0) put_row_extras(a, h, t, cnt != 0, ws, sum, M, s.k0 + s.w0 + mi);  // (callers keep every window non-empty)
}

// Longer windows: R waves per row, four consecutive keys per lane and 256 R
// keys per step over the union window. grid (heads, chunk rows), block 64 R,
// LDS 4 bytes per key of whole steps.
template <int R>
__global__ __launch_bounds__(64 * R) void k_attn_softmax_long(AttnMfmaArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint4 terms[];  // [step][lane of the row]
  __shared__ int64_t red[4][R];
  const uint32_t h = blockIdx.x, l = threadIdx.x & 63, wave = threadIdx.x >> 6, lane = threadIdx.x;
  const uint64_t t = a.t0 + blockIdx.y;
  // all-reduce over the row's waves (slot: one per use)
  auto row_reduce = [&](int slot, int64_t v, auto op) {
    if (l == 0) red[slot][wave] = v;
    __syncthreads();
    int64_t r = red[slot][0];
#pragma unroll
    for (int w = 1; w < R; ++w) r = op(r, red[slot][w]);
    return r;
  };
  const auto max = [](int64_t x, int64_t y) { return x > y ? x : y; };
  const auto add = [](int64_t x, int64_t y) { return int64_t(uint64_t(x) + uint64_t(y)); };
  const RowSpan s = row_span(a, t);
  int32_t* srow = a.scores + (uint64_t(h) * a.crow + (t - a.t0)) * a.srow;
  uint16_t* wrow = reinterpret_cast<uint16_t*>(srow);
  constexpr uint32_t STEP = 256 * R;
  const uint32_t steps = (s.n + STEP - 1) / STEP;
  int32_t mxl = INT32_MIN;
#pragma unroll 4
  for (uint32_t c = 0; c < steps; ++c) {
    const uint32_t k = STEP * c + 4 * lane;
    const int4 v = *reinterpret_cast<const int4*>(srow + (k < s.n ? k : s.n - 4));
    int32_t x[4] = {v.x, v.y, v.z, v.w};
    // positions outside the window take the lowest value (only the steps at
    // its ends hold any)
    if (STEP * c < s.w0 || STEP * (c + 1) > s.w1) {  // (uniform)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (k + e < s.w0 || k + e >= s.w1) x[e] = INT32_MIN;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) mxl = x[e] > mxl ? x[e] : mxl;
    terms[64 * R * c + lane] = make_uint4(x[0], x[1], x[2], x[3]);
  }
  const int32_t mx = int32_t(row_reduce(0, wave_max64(mxl), max));  // the maximum score itself
  // gaps below 2^20 belong to the window, unless the maximum is so low that
  // the masked positions' gaps are below it as well
  const bool low = mx < INT32_MIN + (1 << 20);
  uint32_t first = 0xffffffffu;  // this lane's first position of the maximum
  int64_t sum = 0;               // (below 2^63)
  for (uint32_t c = 0; c < steps; ++c) {
    const uint4 v = terms[64 * R * c + lane];
    const uint32_t x[4] = {v.x, v.y, v.z, v.w};
    uint32_t e[4] = {0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t k = STEP * c + 4 * lane + q;
      const uint32_t gap = uint32_t(mx) - x[q];  // (mx >= x[q])
      bool in = gap < (1u << 20);
      if (low) in = in && k >= s.w0 && k < s.w1;
      if (__any(in)) {
        if (gap == 0 && in) first = k < first ? k : first;
        const int64_t term = in ? softmax_exp(int32_t(x[q]), mx) : 0;
        sum += term;
        e[q] = pack_term(term);
      }
    }
    terms[64 * R * c + lane] = make_uint4(e[0], e[1], e[2], e[3]);
  }
  sum = row_reduce(1, wave_sum_wrap64(sum), add);
  const bool on = s.w1 > s.w0;  // (callers keep every window non-empty)
  const uint64_t M = on ? softmax_recip(sum) : 0;
  int64_t ws = 0;
  for (uint32_t c = 0; c < steps; ++c) {
    const uint32_t k = STEP * c + 4 * lane;
    const uint4 v = terms[64 * R * c + lane];
    const uint32_t e[4] = {v.x, v.y, v.z, v.w};
    uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (__any(e[q])) w[q] = term_weight(e[q], sum, M, ws);
    if (k < s.n)
      *reinterpret_cast<uint2*>(wrow + k) =
          make_uint2((w[0] | (w[1] << 16)) ^ 0x80808080u, (w[2] | (w[3] << 16)) ^ 0x80808080u);
  }
  ws = row_reduce(2, wave_sum_wrap64(ws), add);
  const uint32_t mi = ~uint32_t(row_reduce(3, wave_max64(int64_t(~first)), max));  // the first argmax, relative to k0
  if (lane == 0) put_row_extras(a, h, t, on, ws, sum, M, s.k0 + mi);
}
template <int R>
void launch_softmax_long(const AttnMfmaArgs& m, uint64_t nh, uint64_t keys, hipStream_t s) {
  const uint32_t lds = uint32_t((keys + 256 * R - 1) / (256 * R) * (256 * R) * 4);
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_attn_softmax_long<R>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, 80 << 10);
  (void)attr;
  hipLaunchKernelGGL(k_attn_softmax_long<R>, dim3(unsigned(nh), unsigned(m.crow_used)), dim3(64 * R), lds, s, m);
}
void launch_softmax(const AttnMfmaArgs& m, uint64_t nh, hipStream_t s) {
  // the chunk's longest window and score row
  const uint64_t last = std::min<uint64_t>(m.t0 + m.crow_used + m.causal_offset, m.avail);
  const uint64_t window = m.window ? std::min(last, m.window) : last;
  if (window <= kSoftmaxShort) {
    hipLaunchKernelGGL(k_attn_softmax_short, dim3(unsigned(nh), unsigned((m.crow_used + 3) / 4)), dim3(256), 0, s, m);
    return;
  }
  // four waves per row while four rows' terms fit a CU's LDS (9000 queries of 4
  // heads of 64: 1357 us against 1378 with eight), eight beyond (15000 queries
  // 4192 against 4782; sixteen 5157)
  if (m.srow <= 10240) launch_softmax_long<4>(m, nh, m.srow, s);
  else launch_softmax_long<8>(m, nh, m.srow, s);
}

// Weighted sums: block (kv head, 16 queries, group of 8 dim tiles), wave w on
// dim tile 8 dg + w for the weight tiles of the GB (group size) heads. A 64-key
// substep's weights (two bytes each, 2 KB per head) and the waves' V limbs
// (3 KB each) come through a ring of four LDS stages; the two limbs of a weight
// operand are taken apart in registers. Loads into registers one substep
// ahead left their latency exposed (1.5 us per substep; 0.9 with the ring,
// 72 queries x 79 substeps). A window that holds a four-limb V substep takes a
// ring of three stages with all four limbs (read from global memory when they
// came, they cost a third of the time). The rows' extras and the argmax rows'
// values are read ahead of the loop, and the first stage's copies come before
// any other load: with the chain of two loads behind the loop the kernel took
// 15.0 us in a layer of 120 rows, whose caches are cold, now 10.0. 32 queries
// per block halve the V traffic but leave half the blocks: 1643 queries 172 us
// for the whole attention against 158, 5000 queries the same. Lane l holds, in
// component r, query 4 (l >> 4) + r and dim 16 D + (l & 15). Blocks of the
// longest windows come first. grid (kv heads, query tiles, ceil(dim tiles / 8)), block 512.
template <int GB, int VL>
struct WsumShape {
  static constexpr int NA = GB;                 // weight tiles, one per head
  static constexpr int RPW = (2 * NA + 7) / 8;  // weight copies per wave and stage
  static constexpr int STAGE = 8 * RPW + 8 * VL;  // 1 KB slots: weight halves, then the waves' limbs j
  static constexpr int NB = VL == 3 ? 4 : 3;      // stages
  static constexpr uint32_t lds = NB * STAGE * kOp;
};
// A wave's sources, this lane's bytes: its weight halves at the start of the
// score rows, its V limbs of the cache's first substep.
template <int RPW>
struct WsumSrc {
  const int8_t* w[RPW];
  const int8_t* v;
  uint32_t ksb;  // substep at the start of the score rows
};
// Limbs [j0, j1) of substep ks (and with j0 = 0 the weights) to stage `st` of the ring.
template <int GB, int VL>
__device__ __forceinline__ void wsum_copy(const WsumSrc<WsumShape<GB, VL>::RPW>& src, int8_t* st, uint32_t ks,
                                          uint32_t wave, int j0, int j1) {
  constexpr int NA = GB, RPW = WsumShape<GB, VL>::RPW;
  if (j0 == 0)
#pragma unroll
    for (int u = 0; u < RPW; ++u) {
      uint32_t c = wave * RPW + u;
      if (c >= 2 * NA) c = 2 * NA - 1;  // (spare slots copy the last half again)
      ring_copy(src.w[u] + uint64_t(ks - src.ksb) * 128, st + c * kOp);
    }
#pragma unroll
  for (int j = 0; j < VL; ++j)
    if (j >= j0 && j < j1) ring_copy(src.v + (uint64_t(ks) * 4 + j) * kOp, st + (8 * RPW + j * 8 + wave) * kOp);
}
// The K loop over substeps [ks0, ks1), whose first stage's weights and first
// three limbs are on their way; `ahead` runs once the other first stages are.
template <int GB, int VL, class Ahead>
__device__ __forceinline__ void wsum_loop(const WsumSrc<WsumShape<GB, VL>::RPW>& src, int8_t* ring, uint32_t ks0,
                                          uint32_t ks1, const uint64_t (&vbits)[4], uint32_t l, uint32_t wave,
                                          v4i (&acc)[GB][5], int32_t& wide_sum, Ahead&& ahead) {
  using S = WsumShape<GB, VL>;
  constexpr int NA = GB, RPW = S::RPW, NB = S::NB, LPW = RPW + VL;
  const uint32_t nst = ks1 - ks0;
  const uint64_t vb0 = vbits[0], vb1 = vbits[1], vb2 = vbits[2], vb3 = vbits[3];
  if (VL == 4 && nst) wsum_copy<GB, VL>(src, ring, ks0, wave, 3, 4);
#pragma unroll
  for (int p = 1; p < NB - 1; ++p)
    if (uint32_t(p) < nst) wsum_copy<GB, VL>(src, ring + p * S::STAGE * kOp, ks0 + p, wave, 0, VL);
  ahead();
  for (uint32_t st = 0; st < nst; ++st) {
    ring_barrier<(NB - 2) * LPW>(st + NB - 1 <= nst);
    if (st + NB - 1 < nst)
      wsum_copy<GB, VL>(src, ring + ((st + NB - 1) % NB) * S::STAGE * kOp, ks0 + st + NB - 1, wave, 0, VL);
    const int8_t* base = ring + (st % NB) * S::STAGE * kOp + l * 16;
    v4i b[VL];
#pragma unroll
    for (int j = 0; j < VL; ++j) b[j] = *reinterpret_cast<const v4i*>(base + (8 * RPW + j * 8 + wave) * kOp);
    const uint64_t vword = st < 128 ? (st < 64 ? vb0 : vb1) : (st < 192 ? vb2 : vb3);
    const bool wide = VL == 4 && ((vword >> (st & 63)) & 1);  // (workgroup-uniform)
#pragma unroll
    for (int g = 0; g < NA; ++g) {
      const v4i x = *reinterpret_cast<const v4i*>(base + 2 * g * kOp);
      const v4i y = *reinterpret_cast<const v4i*>(base + (2 * g + 1) * kOp);
      v4i w[2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        w[0][q] = int(__builtin_amdgcn_perm(uint32_t(x[2 * q + 1]), uint32_t(x[2 * q]), 0x06040200u));
        w[1][q] = int(__builtin_amdgcn_perm(uint32_t(x[2 * q + 1]), uint32_t(x[2 * q]), 0x07050301u));
        w[0][q + 2] = int(__builtin_amdgcn_perm(uint32_t(y[2 * q + 1]), uint32_t(y[2 * q]), 0x06040200u));
        w[1][q + 2] = int(__builtin_amdgcn_perm(uint32_t(y[2 * q + 1]), uint32_t(y[2 * q]), 0x07050301u));
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j)
          acc[g][i + j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[i], b[j], acc[g][i + j], 0, 0, 0);
      if (VL == 4 && wide)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          acc[g][i + 3] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[i], b[VL - 1], acc[g][i + 3], 0, 0, 0);
    }
    if (VL == 4 && wide && wave < NA)
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        const v4i x = *reinterpret_cast<const v4i*>(base + (2 * wave + hf) * kOp);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint32_t d = uint32_t(x[q]) ^ 0x80808080u;
          wide_sum += int32_t((d & 0xffffu) + (d >> 16));
        }
      }
  }
}
// OVER: the outputs share memory with V, whose argmax rows then come from its
// limbs (as a branch of one kernel this cost layers of 16 to 800 rows 2-3 %).
template <int GB, bool OVER>
__global__ __launch_bounds__(512) void k_attn_wsum_mfma(AttnMfmaArgs a) {
  constexpr int NA = GB, RPW = WsumShape<GB, 3>::RPW;
  extern __shared__ __attribute__((aligned(16))) int8_t ring[];  // [stage][weight halves, V limbs][lane]
  __shared__ int32_t wsw[NA][16];  // sum of the weights over four-limb V substeps
  const uint32_t l = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t kvh = blockIdx.x;
  const uint64_t t_lo = a.t0 + uint64_t(gridDim.y - 1 - blockIdx.y) * 16;
  const uint32_t ndt = a.hd / 16, D = blockIdx.z * 8 + wave;
  const bool d_on = D < ndt;
  const uint32_t G = a.groups;
  const uint64_t t_end = a.t0 + a.crow_used;  // past the chunk's last query
  const uint64_t t_hi = t_lo + 15 < t_end ? t_lo + 15 : t_end - 1;
  const uint64_t kmin = attn_range(a, t_lo).start, kmax = attn_range(a, t_hi).end;
  const uint32_t ks0 = uint32_t(kmin / 64), ks1 = uint32_t((kmax + 63) / 64);  // key substeps of the union window
  const uint32_t nvh = (a.hd + 255) / 256;
  const uint32_t* vw = a.vwide + (uint64_t(kvh) * nvh + blockIdx.z / 2) * a.nks;
  // this wave's copies: weight slot c is half c & 1 (keys 16 g + 8 half .., g
  // the lane group) of tile c >> 1, lane l its query l & 15
  WsumSrc<RPW> src;
#pragma unroll
  for (int u = 0; u < RPW; ++u) {
    uint32_t c = wave * RPW + u;
    if (c >= 2 * NA) c = 2 * NA - 1;
    const uint32_t ai = c >> 1;
    const uint64_t t = t_lo + (l & 15);
    const uint64_t row = uint64_t(kvh * G + ai) * a.crow + ((t < t_end ? t : t_end - 1) - a.t0);
    src.w[u] = reinterpret_cast<const int8_t*>(a.scores + row * a.srow) + 32 * (l >> 4) + 16 * (c & 1);
  }
  const uint32_t Dc = d_on ? D : ndt - 1, dim = 16 * Dc + (l & 15);
  src.v = a.vlimbs + (uint64_t(kvh) * ndt + Dc) * a.nks * 4 * kOp + l * 16;
  src.ksb = uint32_t(score_base(a, t_lo) / 64);
  if (ks0 < ks1) wsum_copy<GB, 3>(src, ring, ks0, wave, 0, 3);
  // the window's four-limb V substeps (bit st % 64 of word st / 64; at most
  // 16000 keys), and the rows' extras
  uint64_t vbits[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const uint32_t k = ks0 + 64 * c + l;
    vbits[c] = __ballot(k < ks1 && vw[k < ks1 ? k : ks0]);
  }
  int32_t extra[NA][4], vmax[NA][4];
  uint32_t wtot[NA][4], argm[NA][4];
#pragma unroll
  for (int g = 0; g < NA; ++g)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const uint64_t t = t_lo + 4 * (l >> 4) + r;
      const uint64_t o = uint64_t(kvh * G + g) * a.n_queries + (t < t_end ? t : t_end - 1);
      argm[g][r] = a.argm[o];
      extra[g][r] = a.extra[o];
      wtot[g][r] = a.wtot[o];
    }
  int64_t vs = 0;
  auto ahead = [&] {
#pragma unroll
    for (int g = 0; g < NA; ++g)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const uint32_t key = argm[g][r];
        if constexpr (!OVER) {
          vmax[g][r] = a.v[uint64_t(key) * a.kv_ld + uint64_t(kvh) * a.hd + dim];
        } else {
          const int8_t* c = src.v - l * 16 + uint64_t(key / 64) * 4 * kOp + (key / 16 % 4 * 16 + (l & 15)) * 16 + key % 16;
          vmax[g][r] = c[0] + c[kOp] * 256 + c[2 * kOp] * 65536 + int32_t(kC3);
          if (vw[key / 64]) vmax[g][r] += int32_t(uint32_t(c[3 * kOp]) << 24) + int32_t(kC4 - kC3);
        }
      }
    // sum of v' over the window's substeps: lane group g takes every fourth one,
    // eight loads at a time (one after the other they cost more than the products)
    for (uint32_t k = ks0 + (l >> 4); k < ks1; k += 32) {
      int64_t x[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const uint32_t kk = k + 4 * u;
        x[u] = a.vblk[(uint64_t(kvh) * a.nks + (kk < ks1 ? kk : ks0)) * a.hd + dim];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) vs += k + 4 * u < ks1 ? x[u] : 0;
    }
  };
  v4i acc[NA][5];
#pragma unroll
  for (int g = 0; g < NA; ++g)
#pragma unroll
    for (int s = 0; s < 5; ++s) acc[g][s] = v4i{0, 0, 0, 0};
  int32_t wide_sum = 0;  // of weight tile `wave`, this lane's query and keys
  if (vbits[0] | vbits[1] | vbits[2] | vbits[3])  // (workgroup-uniform)
    wsum_loop<GB, 4>(src, ring, ks0, ks1, vbits, l, wave, acc, wide_sum, ahead);
  else
    wsum_loop<GB, 3>(src, ring, ks0, ks1, vbits, l, wave, acc, wide_sum, ahead);
  // (the sums as 32-bit registers here: else their widening moves into the two
  // loops and the pairs do not fit)
#pragma unroll
  for (int g = 0; g < NA; ++g)
#pragma unroll
    for (int s = 0; s < 5; ++s) asm volatile("" : "+v"(acc[g][s]));
  vs += __shfl_xor(vs, 16, 64);
  vs += __shfl_xor(vs, 32, 64);
  wide_sum += __shfl_xor(wide_sum, 16, 64);
  wide_sum += __shfl_xor(wide_sum, 32, 64);
  if (wave < NA && l < 16) wsw[wave][l] = wide_sum;
  __syncthreads();
  if (!d_on) return;
#pragma unroll
  for (int g = 0; g < NA; ++g) {
    const uint32_t h = kvh * G + g;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const uint32_t qi = 4 * (l >> 4) + r;
      const uint64_t t = t_lo + qi;
      if (t >= t_end) continue;
      uint64_t dot = 0;
#pragma unroll
      for (int s = 0; s < 5; ++s) dot += uint64_t(int64_t(acc[g][s][r])) << (8 * s);
      dot += uint64_t(kC3) * uint64_t(vs) + uint64_t(kC3) * uint64_t(wtot[g][r]) +
             uint64_t(kC4 - kC3) * uint64_t(int64_t(wsw[g][qi]));
      dot += uint64_t(int64_t(extra[g][r]) * int64_t(vmax[g][r]));
      a.out[t * a.out_ld + uint64_t(h) * a.hd + dim] = requant(int64_t(dot));
    }
  }
}
template <int GB, bool OVER>
void launch_wsum_over(const AttnMfmaArgs& m, uint64_t nkv, hipStream_t s) {
  constexpr uint32_t lds = std::max(WsumShape<GB, 3>::lds, WsumShape<GB, 4>::lds);
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_attn_wsum_mfma<GB, OVER>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  (void)attr;
  const dim3 grid(unsigned(nkv), unsigned((m.crow_used + 15) / 16), unsigned((m.hd / 16 + 7) / 8));
  hipLaunchKernelGGL((k_attn_wsum_mfma<GB, OVER>), grid, dim3(512), lds, s, m);
}
template <int GB>
void launch_wsum(const AttnMfmaArgs& m, uint64_t nkv, hipStream_t s) {
  if (m.v_overwritten) launch_wsum_over<GB, true>(m, nkv, s);
  else launch_wsum_over<GB, false>(m, nkv, s);
}
// Score rows (int32) of one chunk of queries. At 5000 queries, 8 heads of 256:
// 64 MB 1.29 ms, 128 MB 0.94 ms, 256 MB 0.84 ms (four chunks), 384 MB 0.86 ms;
// 3500 queries 0.64, 0.49, 0.46 and 0.41 ms (each chunk ends on a partly filled
// device). 256 MB keeps the whole work area within its bound up to 16000 rows
// of that shape.
constexpr uint64_t kScoreBytes = uint64_t(256) << 20;

// Keys of a score row: every key, or with a window the union window of 32
// queries in whole 64-key substeps.
uint64_t score_row(const AttnArgs& a) {
  const uint64_t all = (a.avail + 63) / 64 * 64;
  return a.window ? std::min(all, (std::min(a.window, all) + 31 + 63) / 64 * 64 + 64) : all;
}

// Queries per chunk: whole tiles of 32 unless one chunk holds every query.
uint64_t attn_chunk_rows(const AttnArgs& a) {
  const uint64_t per = uint64_t(a.num_heads) * score_row(a) * 4;
  const uint64_t fit = std::max<uint64_t>(kScoreBytes / per, 32) / 32 * 32;
  return std::min<uint64_t>(a.n_queries, fit);
}

}  // namespace

// Work area of the MFMA path (zero when it does not apply): limb blocks of Q,
// K and V, their offset sums, a chunk's score rows and the per-row extras.
uint64_t attn_mfma_bytes(const AttnArgs& a) {
  if (a.seqs || !a.causal || a.ring_cap || a.hd % 64 != 0 || a.hd > 512 || a.num_heads == 0 || a.groups == 0 ||
      a.num_heads % a.groups != 0 || a.groups > 4 ||
      a.n_queries < 16 || a.avail == 0 || a.q_ld % 4 != 0 || a.kv_ld % 4 != 0 ||
      reinterpret_cast<uintptr_t>(a.q) % 16 != 0 || reinterpret_cast<uintptr_t>(a.k) % 16 != 0)
    return 0;
  const uint64_t nh = a.num_heads, nkv = nh / a.groups, nsub = a.hd / 64;
  const uint64_t nqt = (a.n_queries + 15) / 16, nkt = (a.avail + 15) / 16, nks = (a.avail + 63) / 64;
  uint64_t b = 0;
  b += nh * nqt * nsub * 4 * kOp;            // Q limbs
  b += nkv * nkt * nsub * 4 * kOp;           // K limbs
  b += nkv * (a.hd / 16) * nks * 4 * kOp;    // V limbs
  b += nh * nqt * 16 * 8 + nkv * nkt * 16 * 8 + nkv * nks * a.hd * 8;  // offset sums
  b += nkv * ((a.hd + 255) / 256) * nks * 4;  // V widths
  b += nh * attn_chunk_rows(a) * score_row(a) * 4;   // scores / weights of a chunk
  b += nh * a.n_queries * 12;                // extras, argmax rows, weight sums
  return b + 4096;
}

// What the work area takes with every query's full score row in it at once.
uint64_t attn_mfma_unchunked_bytes(const AttnArgs& a) {
  const uint64_t b = attn_mfma_bytes(a);
  const uint64_t rows = uint64_t(a.num_heads) * 4;
  return b == 0 ? 0 : b + rows * (a.n_queries * ((a.avail + 63) / 64 * 64) - attn_chunk_rows(a) * score_row(a));
}

bool attn_mfma_plan(const AttnArgs& a, AttnMfmaArgs& m) {
  const uint64_t need = attn_mfma_bytes(a);
  void* work = a.work;
  if (need == 0 || !work || a.work_bytes < need) return false;
  m = AttnMfmaArgs{};
  const uint64_t nh = a.num_heads, nkv = nh / a.groups, nsub = a.hd / 64;
  m.hd = a.hd;
  m.groups = a.groups;
  m.n_queries = a.n_queries;
  m.avail = a.avail;
  m.window = a.window;
  m.causal_offset = a.causal_offset;
  m.nqt = (a.n_queries + 15) / 16;
  m.nkt = (a.avail + 15) / 16;
  m.nks = (a.avail + 63) / 64;
  m.srow = score_row(a);
  m.crow = attn_chunk_rows(a);
  m.v = a.v;
  m.kv_ld = a.kv_ld;
  // (V is read again while outputs are written, unless they share memory: its limbs then)
  const uintptr_t v0 = reinterpret_cast<uintptr_t>(a.v), o0 = reinterpret_cast<uintptr_t>(a.out);
  const uint64_t v_bytes = ((a.avail - 1) * a.kv_ld + nkv * a.hd) * 4;
  const uint64_t o_bytes = ((a.n_queries - 1) * a.out_ld + nh * a.hd) * 4;
  m.v_overwritten = v0 < o0 + o_bytes && o0 < v0 + v_bytes;
  m.out = a.out;
  m.out_ld = a.out_ld;
  auto carve = [&](uint64_t bytes) {
    uint8_t* p = static_cast<uint8_t*>(work);
    work = p + ((bytes + 255) / 256) * 256;
    return p;
  };
  m.qlimbs = reinterpret_cast<int8_t*>(carve(nh * m.nqt * nsub * 4 * kOp));
  m.klimbs = reinterpret_cast<int8_t*>(carve(nkv * m.nkt * nsub * 4 * kOp));
  m.vlimbs = reinterpret_cast<int8_t*>(carve(nkv * (a.hd / 16) * m.nks * 4 * kOp));
  m.qsum = reinterpret_cast<int64_t*>(carve(nh * m.nqt * 16 * 8));
  m.ksum = reinterpret_cast<int64_t*>(carve(nkv * m.nkt * 16 * 8));
  m.vblk = reinterpret_cast<int64_t*>(carve(nkv * m.nks * a.hd * 8));
  m.vwide = reinterpret_cast<uint32_t*>(carve(nkv * ((a.hd + 255) / 256) * m.nks * 4));
  m.scores = reinterpret_cast<int32_t*>(carve(nh * m.crow * m.srow * 4));
  m.extra = reinterpret_cast<int32_t*>(carve(nh * a.n_queries * 4));
  m.argm = reinterpret_cast<uint32_t*>(carve(nh * a.n_queries * 4));
  m.wtot = reinterpret_cast<uint32_t*>(carve(nh * a.n_queries * 4));
  return true;
}

bool launch_attention_mfma(const AttnArgs& a, void* work, uint64_t work_bytes, hipStream_t s) {
  AttnArgs aw = a;
  aw.work = work;
  aw.work_bytes = work_bytes;
  AttnMfmaArgs m;
  if (!attn_mfma_plan(aw, m)) return false;
  const uint64_t nh = a.num_heads, nkv = nh / a.groups, nsub = a.hd / 64;
  const unsigned th = unsigned(64 * nsub);
  // Q rows: heads are the row segments of q; K rows: kv heads of k (unless
  // the rows' producer wrote their blocks)
  const SplitRows sq{a.q, a.q_ld, a.n_queries, m.nqt, m.qlimbs, m.qsum, (a.split_done & 1) ? 0 : uint32_t(nh)};
  const SplitRows sk{a.k, a.kv_ld, a.avail, m.nkt, m.klimbs, m.ksum, (a.split_done & 2) ? 0 : uint32_t(nkv)};
  if (sq.heads + sk.heads)
    hipLaunchKernelGGL(k_attn_split_rows,
                       dim3(sq.heads + sk.heads,
                            unsigned(std::max(sq.heads ? m.nqt : 0, sk.heads ? m.nkt : 0))),
                       dim3(th), 0, s, sq, sk, a.hd);
  const unsigned vth = unsigned(64 * std::min<uint64_t>(a.hd / 16, 16));
  hipLaunchKernelGGL(k_attn_split_v, dim3(unsigned(nkv), unsigned(m.nks), unsigned((a.hd + 255) / 256)), dim3(vth), 0, s, a.v,
                     a.kv_ld, a.avail, a.hd, m.nks, m.vlimbs, m.vblk, m.vwide);
  for (m.t0 = 0; m.t0 < m.n_queries; m.t0 += m.crow) {
    m.crow_used = std::min<uint64_t>(m.crow, m.n_queries - m.t0);
    switch (nsub) {
      case 1: launch_scores_nsub<1>(m, nkv, s); break;
      case 2: launch_scores_nsub<2>(m, nkv, s); break;
      case 3: launch_scores_nsub<3>(m, nkv, s); break;
      case 4: launch_scores_nsub<4>(m, nkv, s); break;
      case 5: launch_scores_nsub<5>(m, nkv, s); break;
      case 6: launch_scores_nsub<6>(m, nkv, s); break;
      case 7: launch_scores_nsub<7>(m, nkv, s); break;
      default: launch_scores_nsub<8>(m, nkv, s); break;
    }
    launch_softmax(m, nh, s);
    switch (a.groups) {
      case 1: launch_wsum<1>(m, nkv, s); break;
      case 2: launch_wsum<2>(m, nkv, s); break;
      case 3: launch_wsum<3>(m, nkv, s); break;
      default: launch_wsum<4>(m, nkv, s); break;
    }
  }
  return true;
}

}  // namespace det
