// Causal prefill attention on int8 MFMA (det_attention_prefill,
// det_kernels.rs:575-651): the q.k and weight.v products of every (head,
// query) row exactly, as wrapping int64 sums, from int8 limb products.
//
// An int32 x is split into signed bytes with an offset, three where its whole
// group fits 24 bits and four otherwise:
//   x = c0 + 256 c1 + 65536 c2 + C3,               C3 = 32896    (x in [-2^23, 2^23)),
//   x = c0 + 256 c1 + 65536 c2 + 2^24 c3 + C4,     C4 = 8421504,
// c_j the signed bytes of (x + 2^23) ^ 0x808080 or of x ^ 0x808080. The groups
// are one row of Q or K (its head dims), and 64 keys of V. A softmax weight w
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
// past n take zero limbs and a zero sum. grid (heads, tiles), block 64 * nsub.
__global__ __launch_bounds__(512) void k_attn_split_rows(const int32_t* __restrict__ x, uint64_t ld, uint64_t n,
                                                         uint32_t hd, uint64_t ntiles, int8_t* __restrict__ limbs,
                                                         int64_t* __restrict__ sums) {
  __shared__ int64_t part[8][16];
  __shared__ uint32_t wide16[8];  // bit i: row i has a wide value in the wave's dims
  const uint32_t h = blockIdx.x, T = blockIdx.y, s = threadIdx.x >> 6, l = threadIdx.x & 63;
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
// [64 ks + 16 (l >> 4), +16) (keys past avail have zero limbs). The substep
// takes four limbs (vwide[kvh * nks + ks] = 1) when any of its values needs
// them. vblk[ks][dim] = sum over the substep's keys of v - C. grid (kv heads,
// nks), block 64 * min(hd / 16, 16) (waves loop over the dim tiles, at most
// two each up to 512 dims).
__global__ __launch_bounds__(1024) void k_attn_split_v(const int32_t* __restrict__ v, uint64_t ld, uint64_t avail,
                                                       uint32_t hd, uint64_t nks, int8_t* __restrict__ limbs,
                                                       int64_t* __restrict__ vblk, uint32_t* __restrict__ vwide) {
  const uint32_t kvh = blockIdx.x, ks = blockIdx.y, l = threadIdx.x & 63;
  const uint32_t ndt = hd / 16, nw = blockDim.x >> 6;
  const uint64_t k0 = uint64_t(ks) * 64 + 16 * (l >> 4);
  int32_t x[2][16];
  bool wl = false;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const uint32_t D = (threadIdx.x >> 6) + u * nw;
    const uint32_t dim = 16 * (D < ndt ? D : ndt - 1) + (l & 15);
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const uint64_t r = k0 + e;
      x[u][e] = (D < ndt && r < avail) ? v[r * ld + uint64_t(kvh) * hd + dim] : 0;
    }
    wl = wl || attn_wide16(x[u]);
  }
  const bool wide = __syncthreads_or(wl) != 0;
  if (threadIdx.x == 0) vwide[uint64_t(kvh) * nks + ks] = wide;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const uint32_t D = (threadIdx.x >> 6) + u * nw;
    if (D >= ndt) break;
    const uint32_t dim = 16 * D + (l & 15);
#pragma unroll
    for (int e = 0; e < 16; ++e)
      if (k0 + e >= avail) x[u][e] = int32_t(wide ? kC4 : kC3);
    v4i limb[4];
    int64_t sm = split4(x[u], wide, limb);
    int8_t* blk = limbs + ((uint64_t(kvh) * ndt + D) * nks + ks) * 4 * kOp + l * 16;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j < 3 || wide) *reinterpret_cast<v4i*>(blk + j * kOp) = limb[j];
    sm += __shfl_xor(sm, 16, 64);
    sm += __shfl_xor(sm, 32, 64);
    if (l < 16) vblk[(uint64_t(kvh) * nks + ks) * hd + dim] = sm;
  }
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
__device__ __forceinline__ void score_tile(const v4i (&q)[NSUB][4], const v4i* kt, uint32_t l, int64_t qpack,
                                           const int64_t* kpack, int32_t* dst, bool on) {
  v4i acc[2 * NL - 1];
#pragma unroll
  for (int s = 0; s < 2 * NL - 1; ++s) acc[s] = v4i{0, 0, 0, 0};
#pragma unroll
  for (int s = 0; s < NSUB; ++s)
#pragma unroll
    for (int j = 0; j < NL; ++j) {
      const v4i k = kt[(s * 4 + j) * 64 + l];
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
// the G heads, span of key tiles). Wave w keeps the limb operands of head
// w % G, query tile w / G in registers and multiplies every key tile of the
// span with them; the key tiles (4 KB per 64 head dims) stream through a ring
// of four LDS stages of KS tiles (about 16 KB), so each is read once per block
// for all its rows, and no wave waits for its own operands. (Key tiles held in
// registers and queries in LDS, each wave loading its own key tiles, left the
// loads exposed: 1643 queries, 8 heads of 256, 65 us.) A tile of 16 x 16 that
// touches the query tile's union window is written whole; the softmax masks
// the positions outside a query's window. grid (kv heads, groups of NW / G
// query tiles, spans), block 64 NW.
constexpr int kScoreStages = 4;
constexpr uint32_t kScoreSpan = 64;  // most key tiles per block
template <int NSUB, int NW>
__global__ __launch_bounds__(64 * NW, NSUB <= 4 ? 4 : 2) void k_attn_scores_mfma(AttnMfmaArgs a, uint32_t span) {
  constexpr int KS = NSUB == 1 ? 4 : (NSUB == 2 ? 2 : 1);  // key tiles per stage
  constexpr int SLOTS = KS * NSUB * 4, LPW = (SLOTS + NW - 1) / NW;
  extern __shared__ __attribute__((aligned(16))) int8_t ring[];  // [stage][key tile][substep][limb][lane]
  __shared__ int64_t kpk[kScoreSpan * 16];
  const uint32_t l = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t kvh = blockIdx.x, G = a.groups, QT = NW / G;
  const uint64_t t_end = a.t0 + a.crow_used;
  // the block's keys: the union window of its queries within its span
  const uint64_t tb = a.t0 + uint64_t(blockIdx.y) * 16 * QT;
  const uint64_t tb_hi = tb + 16 * QT < t_end ? tb + 16 * QT - 1 : t_end - 1;
  uint64_t j0 = attn_range(a, tb).start / 16, j1 = (attn_range(a, tb_hi).end + 15) / 16;
  const uint64_t z0 = uint64_t(blockIdx.z) * span;
  j0 = j0 > z0 ? j0 : z0;
  j1 = j1 < z0 + span ? j1 : z0 + span;
  if (j0 >= j1) return;  // (workgroup-uniform)
  const uint32_t ntile = uint32_t(j1 - j0), nst = (ntile + KS - 1) / KS;
  const int8_t* kb = a.klimbs + uint64_t(kvh) * a.nkt * NSUB * 4 * kOp + l * 16;
  auto copy_stage = [&](uint32_t st) {
#pragma unroll
    for (int u = 0; u < LPW; ++u) {
      uint32_t c = wave * LPW + u;
      if (c >= uint32_t(SLOTS)) c = SLOTS - 1;  // (spare slots copy the last block again)
      uint64_t J = j0 + uint64_t(st) * KS + c / (NSUB * 4);
      if (J >= j1) J = j1 - 1;
      ring_copy(kb + (J * NSUB * 4 + c % (NSUB * 4)) * kOp, ring + ((st % kScoreStages) * SLOTS + c) * kOp);
    }
  };
  for (uint32_t i = threadIdx.x; i < ntile * 16; i += 64 * NW) kpk[i] = a.ksum[(uint64_t(kvh) * a.nkt + j0) * 16 + i];
  // this wave's queries
  const uint32_t h = kvh * G + wave % G;
  const uint64_t t_lo = tb + 16 * (wave / G), t = t_lo + (l & 15);
  const bool q_on = wave < G * QT && t_lo < t_end;  // (wave-uniform)
  const uint64_t tc = q_on ? t_lo : tb;
  const uint64_t T = tc / 16;
  const uint64_t kmin = attn_range(a, tc).start, kmax = attn_range(a, tc + 15 < t_end ? tc + 15 : t_end - 1).end;
  v4i q[NSUB][4];
  const int8_t* qb = a.qlimbs + (uint64_t(q_on ? h : kvh * G) * a.nqt + T) * NSUB * 4 * kOp + l * 16;
#pragma unroll
  for (int s = 0; s < NSUB; ++s)
#pragma unroll
    for (int i = 0; i < 4; ++i) q[s][i] = *reinterpret_cast<const v4i*>(qb + (s * 4 + i) * kOp);
  const int64_t qpack = a.qsum[uint64_t(q_on ? h : kvh * G) * a.nqt * 16 + T * 16 + (l & 15)];
  const bool qwide = __any(qpack & 1);
  int32_t* row = a.scores + (uint64_t(h) * a.crow + (t - a.t0)) * a.srow + 4 * (l >> 4);
  const uint64_t kbase = score_base(a, tc);
  const bool on = q_on && t < t_end;
  __syncthreads();  // the key sums; (no other load is outstanding from here on)
#pragma unroll
  for (int p = 0; p < kScoreStages - 1; ++p)
    if (uint32_t(p) < nst) copy_stage(p);
  for (uint32_t st = 0; st < nst; ++st) {
    ring_barrier<(kScoreStages - 2) * LPW>(st + kScoreStages - 1 <= nst);
    if (st + kScoreStages - 1 < nst) copy_stage(st + kScoreStages - 1);
    const v4i* base = reinterpret_cast<const v4i*>(ring + (st % kScoreStages) * SLOTS * kOp);
#pragma unroll
    for (int u = 0; u < KS; ++u) {
      const uint32_t jl = st * KS + u;
      const uint64_t key0 = (j0 + jl) * 16;
      if (!q_on || jl >= ntile || key0 >= kmax || key0 + 16 <= kmin) continue;  // (wave-uniform)
      const int64_t* kp = kpk + jl * 16;
      const bool wide = qwide || __any(kp[l & 15] & 1);
      int32_t* dst = row + (key0 - kbase);
      if (wide) score_tile<NSUB, 4>(q, base + u * NSUB * 4 * 64, l, qpack, kp, dst, on);
      else score_tile<NSUB, 3>(q, base + u * NSUB * 4 * 64, l, qpack, kp, dst, on);
    }
  }
}

template <int NSUB, int NW>
void launch_scores_nw(const AttnMfmaArgs& m, uint64_t nkv, hipStream_t s) {
  constexpr int KS = NSUB == 1 ? 4 : (NSUB == 2 ? 2 : 1);
  constexpr uint32_t lds = kScoreStages * KS * NSUB * 4 * kOp;
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_attn_scores_mfma<NSUB, NW>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  (void)attr;
  const uint64_t rows = 16 * (NW / m.groups), y = (m.crow_used + rows - 1) / rows;
  // spans short enough for about four blocks per CU (half of them are outside the causal range)
  uint32_t span = kScoreSpan;
  while (span > 8 && nkv * y * ((m.nkt + span - 1) / span) < 1024) span /= 2;
  const dim3 grid(unsigned(nkv), unsigned(y), unsigned((m.nkt + span - 1) / span));
  hipLaunchKernelGGL((k_attn_scores_mfma<NSUB, NW>), grid, dim3(64 * NW), lds, s, m, span);
}
template <int NSUB>
void launch_scores_nsub(const AttnMfmaArgs& m, uint64_t nkv, hipStream_t s) {
  if (m.groups == 3) launch_scores_nw<NSUB, 6>(m, nkv, s);
  else launch_scores_nw<NSUB, 8>(m, nkv, s);
}

// Softmax of every (head, query) row of the chunk, R waves per row (one, or
// the four of a workgroup), four consecutive keys per lane and 256 R keys per
// step: the first argmax, the exp sum, the weights. The weights replace the
// scores in place as 16-bit values w ^ 0x8080 at the start of the row (the
// r-th key at byte 2 r; a step is written after it and, across the waves of a row,
// every cached step is read, and later steps lie past what is written), zero
// outside the window, over the 64-key substeps of the union window of the 32
// queries that share a score row's first key. The first 256 R CR scores and exp
// terms of a row stay in registers; later ones are read and computed a second
// time. Terms 16 or more below the maximum are zero exactly, and a wave's 64
// keys that have only such terms skip the exp series and the weights (rows of
// 256 normalised dims have scores of standard deviation 16).
// wtot: the row's weights' sum; extra: what the first argmax row holds past
// its (clamped) 16-bit weight, the residual included. grid (heads,
// ceil(chunk rows * R / 4)), block 256.
template <int R, int CR>
__global__ __launch_bounds__(256) void k_attn_softmax_rows(AttnMfmaArgs a) {
  __shared__ int64_t red[4][4];
  const uint32_t h = blockIdx.x, l = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint64_t t = a.t0 + (R == 1 ? uint64_t(blockIdx.y) * 4 + wave : uint64_t(blockIdx.y));
  if (t >= a.t0 + a.crow_used) return;  // (workgroup-uniform with R = 4)
  const uint32_t lane = R == 1 ? l : threadIdx.x;  // lane of the row
  // all-reduce over the row's waves (slot: one per use)
  auto row_reduce = [&](int slot, int64_t v, auto op) {
    if constexpr (R == 1) return v;
    if (l == 0) red[slot][wave] = v;
    __syncthreads();
    return op(op(red[slot][0], red[slot][1]), op(red[slot][2], red[slot][3]));
  };
  const AttnRange w = attn_range(a, t);
  const uint64_t p_hi = (t | 31) < a.n_queries ? (t | 31) : a.n_queries - 1;
  const uint64_t K0 = score_base(a, t), K1 = (attn_range(a, p_hi).end + 63) & ~uint64_t(63);
  int32_t* srow = a.scores + (uint64_t(h) * a.crow + (t - a.t0)) * a.srow;
  uint16_t* wrow = reinterpret_cast<uint16_t*>(srow);
  constexpr uint32_t STEP = 256 * R;
  const uint32_t n = uint32_t(K1 - K0), steps = (n + STEP - 1) / STEP;
  const uint32_t w0 = uint32_t(w.start - K0), w1 = uint32_t(w.end - K0);  // the window, relative to K0
  const int32_t* src = srow;
  auto load = [&](uint32_t c, int32_t (&x)[4]) {
    const uint32_t k = STEP * c + 4 * lane;
    const int4 v = *reinterpret_cast<const int4*>(src + (k < n ? k : n - 4));
    x[0] = v.x, x[1] = v.y, x[2] = v.z, x[3] = v.w;
  };
  // positions outside the window take the lowest value (only the steps at its
  // ends hold any)
  auto mask = [&](uint32_t c, int32_t (&x)[4]) {
    if (STEP * c >= w0 && STEP * (c + 1) <= w1) return;  // (wave-uniform)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t k = STEP * c + 4 * lane + e;
      if (k < w0 || k >= w1) x[e] = INT32_MIN;
    }
  };
  int32_t mxl = INT32_MIN;
  auto upd = [&](const int32_t (&x)[4]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) mxl = x[e] > mxl ? x[e] : mxl;
  };
  int32_t sc[CR][4];
#pragma unroll
  for (int c = 0; c < CR; ++c)
    if (uint32_t(c) < steps) load(c, sc[c]);
#pragma unroll
  for (int c = 0; c < CR; ++c)
    if (uint32_t(c) < steps) mask(c, sc[c]), upd(sc[c]);
  for (uint32_t c = CR; c < steps; ++c) {
    int32_t x[4];
    load(c, x);
    mask(c, x);
    upd(x);
  }
  const auto max = [](int64_t x, int64_t y) { return x > y ? x : y; };
  const int32_t mx = int32_t(row_reduce(0, wave_max64(mxl), max));  // the maximum score itself
  // gaps below 2^20 belong to the window, unless the maximum is so low that
  // the masked positions' gaps are below it as well
  const bool low = mx < INT32_MIN + (1 << 20);
  uint32_t first = 0xffffffffu;  // this lane's first position of the maximum
  // exp terms of a step (0 past the window); a term is 2^32 only at gap 0 and
  // below 2^32 - 65000 otherwise, so 32 bits hold it with all ones for 2^32
  int64_t sum_of_terms = 0;  // (below 2^63)
  auto terms = [&](uint32_t c, const int32_t (&x)[4], uint32_t (&e)[4]) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t k = STEP * c + 4 * lane + q;
      const uint32_t gap = uint32_t(mx) - uint32_t(x[q]);  // (mx >= x[q])
      bool in = gap < (1u << 20);
      if (low) in = in && k >= w0 && k < w1;
      e[q] = 0;
      if (__any(in)) {
        if (gap == 0 && in) first = k < first ? k : first;
        const int64_t v = softmax_exp(in ? x[q] : mx, mx);
        e[q] = in ? (v >> 32 ? 0xffffffffu : uint32_t(v)) : 0;
        sum_of_terms += in ? v : 0;
      }
    }
  };
  auto widen = [](uint32_t e) { return int64_t(uint64_t(e) + (e == 0xffffffffu)); };
  const auto add = [](int64_t x, int64_t y) { return int64_t(uint64_t(x) + uint64_t(y)); };
  uint32_t ex[CR][4];
#pragma unroll
  for (int c = 0; c < CR; ++c)
    if (uint32_t(c) < steps) terms(c, sc[c], ex[c]);
  for (uint32_t c = CR; c < steps; ++c) {
    int32_t x[4];
    uint32_t e[4];
    load(c, x);
    mask(c, x);
    terms(c, x, e);
  }
  const int64_t sum = row_reduce(1, wave_sum_wrap64(sum_of_terms), add);
  const uint64_t M = sum > 0 && sum < (int64_t(1) << 61) ? softmax_recip(sum) : 0;
  int64_t ws = 0;  // the weights' sum
  auto put = [&](uint32_t c, const uint32_t (&e)[4]) {
    const uint32_t k0 = STEP * c + 4 * lane;
    int32_t wt[4] = {0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (__any(e[q])) {
        const int64_t v = widen(e[q]);
        wt[q] = M ? softmax_weight_r(v, sum, M) : softmax_weight(v, sum);
        ws += wt[q];
        if (wt[q] > 65535) wt[q] = 65535;  // (the first argmax row: 65536)
      }
    if (k0 < n) {
      const uint32_t lo = (uint32_t(wt[0]) | (uint32_t(wt[1]) << 16)) ^ 0x80808080u;
      const uint32_t hi = (uint32_t(wt[2]) | (uint32_t(wt[3]) << 16)) ^ 0x80808080u;
      *reinterpret_cast<uint2*>(wrow + k0) = make_uint2(lo, hi);
    }
  };
#pragma unroll
  for (int c = 0; c < CR; ++c)
    if (uint32_t(c) < steps) put(c, ex[c]);
  for (uint32_t c = CR; c < steps; ++c) {
    int32_t x[4];
    uint32_t e[4];
    load(c, x);
    mask(c, x);
    terms(c, x, e);
    put(c, e);
  }
  ws = row_reduce(2, wave_sum_wrap64(ws), add);
  const uint32_t mi = ~uint32_t(row_reduce(3, wave_max64(int64_t(~first)), max));  // the first argmax, relative to K0
  if (lane == 0) {
    const uint64_t o = uint64_t(h) * a.n_queries + t;
    const bool on = w.end > w.start;  // (callers keep every window non-empty)
    // the first argmax row's weight (its exp term is that of gap 0) and the
    // residual, added to it with saturation
    const int64_t e0 = int64_t(1) << 32;
    const int32_t wm = !on ? 0 : (M ? softmax_weight_r(e0, sum, M) : softmax_weight(e0, sum));
    const int32_t res = sub_sat(kOneAct, sat32(ws)), kept = wm > 65535 ? 65535 : wm;
    a.extra[o] = on ? add_sat(wm, res) - kept : 0;
    a.argm[o] = on ? uint32_t(K0 + mi) : 0;
    a.wtot[o] = uint32_t(ws - (wm - kept));
  }
}
void launch_softmax(const AttnMfmaArgs& m, uint64_t nh, hipStream_t s) {
  // the chunk's longest row
  uint64_t keys = std::min<uint64_t>(m.t0 + m.crow_used + m.causal_offset, m.avail);
  if (m.window) keys = std::min<uint64_t>(keys, m.window + 127);
  if (keys <= 1024)
    hipLaunchKernelGGL((k_attn_softmax_rows<1, 4>), dim3(unsigned(nh), unsigned((m.crow_used + 3) / 4)), dim3(256), 0, s, m);
  else if (keys <= 4096)
    hipLaunchKernelGGL((k_attn_softmax_rows<4, 4>), dim3(unsigned(nh), unsigned(m.crow_used)), dim3(256), 0, s, m);
  else
    hipLaunchKernelGGL((k_attn_softmax_rows<4, 8>), dim3(unsigned(nh), unsigned(m.crow_used)), dim3(256), 0, s, m);
}

// Weighted sums: block (kv head, 16 queries, group of 8 dim tiles), wave w on
// dim tile 8 dg + w for the weight tiles of the GB (group size) heads. A 64-key
// substep's weights (two bytes each, 2 KB per head) and the waves' V limbs
// (3 KB each) come through a ring of four LDS stages; the two limbs of a weight
// operand are taken apart in registers. The fourth limb of a wide V substep is
// read from global memory when it comes. Loads into registers one substep
// ahead left their latency exposed (1.5 us per substep; 0.9 with the ring,
// 72 queries x 79 substeps). 32 queries per block halve the V traffic but
// leave half the blocks: 1643 queries 172 us for the whole attention against
// 158, 5000 queries the same. Lane l holds, in component r, query
// 4 (l >> 4) + r and dim 16 D + (l & 15). Blocks of the longest windows come
// first. grid (kv heads, query tiles, ceil(dim tiles / 8)), block 512.
template <int GB>
struct WsumShape {
  static constexpr int NA = GB;                 // weight tiles, one per head
  static constexpr int RPW = (2 * NA + 7) / 8;  // weight copies per wave and stage
  static constexpr int STAGE = 8 * RPW + 24;    // 1 KB slots
  static constexpr int NB = 4;                  // stages
};
template <int GB>
__global__ __launch_bounds__(512) void k_attn_wsum_mfma(AttnMfmaArgs a) {
  using S = WsumShape<GB>;
  constexpr int NA = S::NA, RPW = S::RPW, STAGE = S::STAGE, NB = S::NB, LPW = RPW + 3;
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
  const uint32_t ksb = uint32_t(score_base(a, t_lo) / 64);  // substep at the start of the score rows
  const uint32_t ks0 = uint32_t(kmin / 64), ks1 = uint32_t((kmax + 63) / 64);  // key substeps of the union window
  const uint32_t* vw = a.vwide + uint64_t(kvh) * a.nks;
  // this wave's copies: weight slot c is half c & 1 (keys 16 g + 8 half .., g
  // the lane group) of tile c >> 1, lane l its query l & 15
  const int8_t* wsrc[RPW];
#pragma unroll
  for (int u = 0; u < RPW; ++u) {
    uint32_t c = wave * RPW + u;
    if (c >= 2 * NA) c = 2 * NA - 1;
    const uint32_t ai = c >> 1;
    const uint64_t t = t_lo + (l & 15);
    const uint64_t row = uint64_t(kvh * G + ai) * a.crow + ((t < t_end ? t : t_end - 1) - a.t0);
    wsrc[u] = reinterpret_cast<const int8_t*>(a.scores + row * a.srow) + 32 * (l >> 4) + 16 * (c & 1);
  }
  const uint32_t Dc = d_on ? D : ndt - 1, dim = 16 * Dc + (l & 15);
  const int8_t* vb = a.vlimbs + (uint64_t(kvh) * ndt + Dc) * a.nks * 4 * kOp + l * 16;
  auto copy_stage = [&](uint32_t ks) {
    int8_t* st = ring + ((ks - ks0) % NB) * STAGE * kOp;
#pragma unroll
    for (int u = 0; u < RPW; ++u) {
      uint32_t c = wave * RPW + u;
      if (c >= 2 * NA) c = 2 * NA - 1;  // (spare slots copy the last half again)
      ring_copy(wsrc[u] + uint64_t(ks - ksb) * 128, st + c * kOp);
    }
#pragma unroll
    for (int j = 0; j < 3; ++j) ring_copy(vb + (uint64_t(ks) * 4 + j) * kOp, st + (8 * RPW + wave * 3 + j) * kOp);
  };
  // sum of v' over the window's substeps: lane group g takes every fourth one,
  // eight loads at a time (one after the other they cost more than the products)
  int64_t vs = 0;
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
  vs += __shfl_xor(vs, 16, 64);
  vs += __shfl_xor(vs, 32, 64);
  // the window's four-limb V substeps (bit st % 64 of word st / 64; at most
  // 16000 keys), read here and not one by one in the loop
  uint64_t vbits[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const uint32_t k = ks0 + 64 * c + l;
    vbits[c] = __ballot(k < ks1 && vw[k < ks1 ? k : ks0]);
  }
  v4i acc[NA][5];
#pragma unroll
  for (int g = 0; g < NA; ++g)
#pragma unroll
    for (int s = 0; s < 5; ++s) acc[g][s] = v4i{0, 0, 0, 0};
  int32_t wide_sum = 0;  // of weight tile `wave`, this lane's query and keys
  const uint32_t nst = ks1 - ks0;
#pragma unroll
  for (int p = 0; p < NB - 1; ++p)
    if (uint32_t(p) < nst) copy_stage(ks0 + p);
  for (uint32_t ks = ks0; ks < ks1; ++ks) {
    const uint32_t st = ks - ks0;
    ring_barrier<(NB - 2) * LPW>(st + NB - 1 <= nst);
    if (st + NB - 1 < nst) copy_stage(ks + NB - 1);
    const int8_t* base = ring + (st % NB) * STAGE * kOp + l * 16;
    v4i b[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) b[j] = *reinterpret_cast<const v4i*>(base + (8 * RPW + wave * 3 + j) * kOp);
    auto operands = [&](int g, v4i (&w)[2]) {
      const v4i x = *reinterpret_cast<const v4i*>(base + 2 * g * kOp);
      const v4i y = *reinterpret_cast<const v4i*>(base + (2 * g + 1) * kOp);
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        w[0][q] = int(__builtin_amdgcn_perm(uint32_t(x[2 * q + 1]), uint32_t(x[2 * q]), 0x06040200u));
        w[1][q] = int(__builtin_amdgcn_perm(uint32_t(x[2 * q + 1]), uint32_t(x[2 * q]), 0x07050301u));
        w[0][q + 2] = int(__builtin_amdgcn_perm(uint32_t(y[2 * q + 1]), uint32_t(y[2 * q]), 0x06040200u));
        w[1][q + 2] = int(__builtin_amdgcn_perm(uint32_t(y[2 * q + 1]), uint32_t(y[2 * q]), 0x07050301u));
      }
    };
#pragma unroll
    for (int g = 0; g < NA; ++g) {
      v4i w[2];
      operands(g, w);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j)
          acc[g][i + j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[i], b[j], acc[g][i + j], 0, 0, 0);
    }
    const uint64_t vword = st < 128 ? (st < 64 ? vbits[0] : vbits[1]) : (st < 192 ? vbits[2] : vbits[3]);
    if ((vword >> (st & 63)) & 1) {  // (workgroup-uniform)
      const v4i b3 = *reinterpret_cast<const v4i*>(vb + (uint64_t(ks) * 4 + 3) * kOp);
#pragma unroll
      for (int g = 0; g < NA; ++g) {
        v4i w[2];
        operands(g, w);
#pragma unroll
        for (int i = 0; i < 2; ++i)
          acc[g][i + 3] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[i], b3, acc[g][i + 3], 0, 0, 0);
      }
      if (wave < NA)
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
      const uint64_t o = uint64_t(h) * a.n_queries + t;
      uint64_t dot = 0;
#pragma unroll
      for (int s = 0; s < 5; ++s) dot += uint64_t(int64_t(acc[g][s][r])) << (8 * s);
      dot += uint64_t(kC3) * uint64_t(vs) + uint64_t(kC3) * uint64_t(a.wtot[o]) +
             uint64_t(kC4 - kC3) * uint64_t(int64_t(wsw[g][qi]));
      const int32_t vm = a.v[uint64_t(a.argm[o]) * a.kv_ld + uint64_t(kvh) * a.hd + dim];
      dot += uint64_t(int64_t(a.extra[o]) * int64_t(vm));
      a.out[t * a.out_ld + uint64_t(h) * a.hd + dim] = requant(int64_t(dot));
    }
  }
}
template <int GB>
void launch_wsum(const AttnMfmaArgs& m, uint64_t nkv, hipStream_t s) {
  using S = WsumShape<GB>;
  constexpr uint32_t lds = S::NB * S::STAGE * kOp;
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_attn_wsum_mfma<GB>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  (void)attr;
  const dim3 grid(unsigned(nkv), unsigned((m.crow_used + 15) / 16), unsigned((m.hd / 16 + 7) / 8));
  hipLaunchKernelGGL((k_attn_wsum_mfma<GB>), grid, dim3(512), lds, s, m);
}
// Score rows (int32) of one chunk of queries. At 5000 queries, 8 heads of 256:
// 128 MB 1.03 ms, 256 MB 0.97 ms (four chunks), 384 MB 0.93 ms, 64 MB 1.3 ms
// (each chunk ends on a partly filled device); 256 MB keeps the whole work
// area within its bound up to 16000 rows of that shape.
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
  b += nh * nqt * 16 * 8 + nkv * nkt * 16 * 8 + nkv * nks * a.hd * 8 + nkv * nks * 4;  // offset sums, V widths
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
  m.vwide = reinterpret_cast<uint32_t*>(carve(nkv * m.nks * 4));
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
  if (!(a.split_done & 1))
    hipLaunchKernelGGL(k_attn_split_rows, dim3(unsigned(nh), unsigned(m.nqt)), dim3(th), 0, s, a.q, a.q_ld,
                       uint64_t(a.n_queries), a.hd, m.nqt, m.qlimbs, m.qsum);
  if (!(a.split_done & 2))
    hipLaunchKernelGGL(k_attn_split_rows, dim3(unsigned(nkv), unsigned(m.nkt)), dim3(th), 0, s, a.k, a.kv_ld,
                       a.avail, a.hd, m.nkt, m.klimbs, m.ksum);
  const unsigned vth = unsigned(64 * std::min<uint64_t>(a.hd / 16, 16));
  hipLaunchKernelGGL(k_attn_split_v, dim3(unsigned(nkv), unsigned(m.nks)), dim3(vth), 0, s, a.v, a.kv_ld, a.avail,
                     a.hd, m.nks, m.vlimbs, m.vblk, m.vwide);
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
