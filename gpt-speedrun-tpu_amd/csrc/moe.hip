// Top-k expert routing (recipes/reference_moe/train.py:1259-1273).
//
// route_topk: one thread per token.  softmax over the fp32 router logits,
//   jax.lax.top_k selection (largest value first; on equal values the lower
//   expert index first), softmax over the chosen logits.
// route_hist / route_place build the dropless bucket layout over blocks of
//   1024 slots: counts[e], and order = stable argsort(chosen.reshape(-1)) by
//   counting sort (per-block counts in the workspace, per-expert bases from
//   the totals and the blocks before, stable ranks within a block from wave
//   ballots in slot order), rows = order / top_k, position = order^-1.
//
// The routed MLP around it (:1275-1293):
//   router_logits   fp32 x @ router_w (split weights on the matrix cores);
//   moe_gather_rows grouped = flat[rows] (token rows in bucket order);
//   moe_gmm         grouped GEMM over the expert buckets on the MFMA GEMM core,
//                   epilogue bias (+ GELU, or x GELU' for the backward);
//   moe_combine     combined[t] = sum over the token's slots, in bucket order,
//                   of bf16(out * bf16(gate)) -- the .at[rows].add rounding;
//   moe_stats       mean probability, load, (entropy, top-1 gate, logit RMS);
// and their backward: combine_bwd, moe_gmm_dw (per-expert weight + bias
// gradients, split-K fp32 atomics) and router_bwd (gate / probability softmax
// VJPs, dx and d router_w, with the VJP of flat[rows] fused in or, for the
// separate entry points, after gather_bwd).
#include "common.h"
#include "epilogue.h"

#include <math.h>

namespace {

constexpr int kMaxExperts = 64;
constexpr int kFewTopK = 4;

// EP: E rounded up to 4, 8, 16 or 64; the row is held in registers, loaded
// once (re-reading it for each of the passes cost a memory latency per value:
// 9.0 -> 4.6 us at 200 tokens, 9.4 -> 5.5 at 32768, 8 experts).
template <int EP>
__global__ void route_topk_kernel(const float* __restrict__ logits, float* __restrict__ probs,
                                  int32_t* __restrict__ chosen, float* __restrict__ gate, int T, int E, int k) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= T) return;
  float row[EP];
#pragma unroll
  for (int e = 0; e < EP; ++e) row[e] = logits[(size_t)t * E + min(e, E - 1)];
  float mx = -INFINITY;
#pragma unroll
  for (int e = 0; e < EP; ++e)
    if (e < E) mx = fmaxf(mx, row[e]);
  if (probs) {
    float ex[EP], s = 0.f;
#pragma unroll
    for (int e = 0; e < EP; ++e) {
      ex[e] = expf(row[e] - mx);
      if (e < E) s += ex[e];
    }
#pragma unroll
    for (int e = 0; e < EP; ++e)
      if (e < E) probs[(size_t)t * E + e] = ex[e] / s;
  }
  // One pass per chosen expert.
  uint64_t taken = 0;
  auto pick = [&](float& bv) {
    int best = -1;
    bv = 0.f;
#pragma unroll
    for (int e = 0; e < EP; ++e) {
      // Strictly greater keeps the lower index on ties; NaN never wins.
      if (e < E && !(taken >> e & 1) && (best < 0 || row[e] > bv)) {
        best = e;
        bv = row[e];
      }
    }
    taken |= 1ull << best;
    return best;
  };
  int32_t* const ch = chosen + (size_t)t * k;
  float* const gt = gate + (size_t)t * k;
  if (k <= kFewTopK) {  // the chosen logits stay in registers
    float vals[kFewTopK], gm = 0.f, gs = 0.f;
#pragma unroll
    for (int j = 0; j < kFewTopK; ++j) {
      if (j >= k) break;
      ch[j] = pick(vals[j]);
      gm = j == 0 ? vals[0] : fmaxf(gm, vals[j]);
    }
#pragma unroll
    for (int j = 0; j < kFewTopK; ++j) {
      if (j >= k) break;
      vals[j] = expf(vals[j] - gm);
      gs += vals[j];
    }
#pragma unroll
    for (int j = 0; j < kFewTopK; ++j) {
      if (j >= k) break;
      gt[j] = vals[j] / gs;
    }
  } else {  // ... or wait in the gate row
    float gm = 0.f, gs = 0.f;
    for (int j = 0; j < k; ++j) {
      float v;
      ch[j] = pick(v);
      gt[j] = v;
      gm = j == 0 ? v : fmaxf(gm, v);
    }
    for (int j = 0; j < k; ++j) gs += expf(gt[j] - gm);
    for (int j = 0; j < k; ++j) gt[j] = expf(gt[j] - gm) / gs;
  }
}

// Stable bucket order over blocks of kSortBlock slots, in two launches.
// route_hist: each block's per-expert counts into hist[block][e].  route_place:
// each block finds its experts' bases (all experts' totals before e, plus
// the counts of e in the blocks before it) and places its slots at base +
// rank, the rank within the block from wave ballots in slot order; block 0
// also writes counts.
constexpr int kSortBlock = 1024;

__global__ void __launch_bounds__(kSortBlock) route_hist_kernel(const int32_t* __restrict__ chosen, int n_slots,
                                                                int E, int32_t* __restrict__ hist) {
  __shared__ int cnt[kMaxExperts];
  const int tid = threadIdx.x;
  if (tid < E) cnt[tid] = 0;
  __syncthreads();
  const int s = blockIdx.x * kSortBlock + tid;
  if (s < n_slots) atomicAdd(&cnt[chosen[s]], 1);
  __syncthreads();
  if (tid < E) hist[(size_t)blockIdx.x * E + tid] = cnt[tid];
}

__global__ void __launch_bounds__(kSortBlock) route_place_kernel(const int32_t* __restrict__ chosen, int n_slots,
                                                                 int E, int k, const int32_t* __restrict__ hist,
                                                                 int nblocks, int32_t* __restrict__ counts,
                                                                 int32_t* __restrict__ order, int32_t* __restrict__ rows,
                                                                 int32_t* __restrict__ position) {
  __shared__ int total[kMaxExperts], before[kMaxExperts], base[kMaxExperts];
  __shared__ int wave_cnt[kSortBlock / 64][kMaxExperts];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int blk = blockIdx.x;
  if (tid < E) {
    int tot = 0, bef = 0;
    for (int b = 0; b < nblocks; ++b) {
      const int h = hist[(size_t)b * E + tid];
      tot += h;
      bef += b < blk ? h : 0;
    }
    total[tid] = tot;
    before[tid] = bef;
    if (blk == 0) counts[tid] = tot;
  }
  __syncthreads();
  if (tid == 0) {
    int acc = 0;
    for (int e = 0; e < E; ++e) {
      base[e] = acc + before[e];
      acc += total[e];
    }
  }
  const int s = blk * kSortBlock + tid;
  const int my_e = s < n_slots ? chosen[s] : -1;
  const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  int rank = 0;
  for (int e = 0; e < E; ++e) {
    const uint64_t m = __ballot(my_e == e);
    if (my_e == e) rank = __popcll(m & lt_mask);
    if (lane == 0) wave_cnt[wave][e] = __popcll(m);
  }
  __syncthreads();
  if (my_e >= 0) {
    int bw = 0;
    for (int w = 0; w < wave; ++w) bw += wave_cnt[w][my_e];
    const int pos = base[my_e] + bw + rank;
    order[pos] = s;
    rows[pos] = s / k;
    if (position) position[s] = pos;
  }
}

// ---------------------------------------------------------------------------
// Router logits (:1259-1264): logits[t][e] = sum_d f32(x[t][d]) * w[d][e] on
// the bf16 matrix cores without losing a bit of an operand: x is bf16 already
// and each float32 weight is split exactly into three bf16 pieces (8
// significant bits each, by truncation), so a logit is a float32 sum of exact
// products, three MFMAs per 32 columns.  A wave takes 16 tokens
// (v_mfma_f32_16x16x32_bf16, columns = experts, the columns past E unused);
// each lane reads 16 bytes of its token per step straight from memory and the
// weight pieces from LDS.  Bound by reading x once.
// Measured: 32768 tokens x 768, 8 experts 20 us (50 MB of x) against 57 us
// with float32 multiply-adds and 8 lanes per token; 200 x 512 9 against 25.
// ---------------------------------------------------------------------------
constexpr int kMaxRouterExperts = 16;
constexpr int kRouterWaves = 4;

// Elements per LDS row of one expert's weight pieces: whole steps of 32 and 8
// more, so 16 rows read at one column cover all banks.
__host__ __device__ inline int router_row(int D) { return (D + 31) / 32 * 32 + 8; }

// 8 bf16 of row x from column d, zeros past D.
template <bool kVec>
__device__ __forceinline__ bf16x8 load_x8(const bf16* __restrict__ row, int d, int D) {
  if constexpr (kVec) {
    return d < D ? *reinterpret_cast<const bf16x8*>(row + d) : bf16x8{};
  } else {
    bf16x8 v;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = d + j < D ? row[d + j] : (bf16)0.f;
    return v;
  }
}

template <bool kVec>
__global__ void __launch_bounds__(64 * kRouterWaves)
    router_logits_kernel(const bf16* __restrict__ x, const float* __restrict__ w, float* __restrict__ logits, int T,
                         int D, int E) {
  extern __shared__ __attribute__((aligned(16))) bf16 wsh[];  // [3][E][router_row(D)]
  const int R = router_row(D);
  for (int i = threadIdx.x; i < E * R; i += blockDim.x) {
    const int d = i / E, e = i % E;  // (consecutive threads read consecutive weights)
    const float v = d < D ? w[(size_t)d * E + e] : 0.f;
    const uint32_t b0 = __builtin_bit_cast(uint32_t, v) & 0xFFFF0000u;
    const float r1 = v - __builtin_bit_cast(float, b0);  // exact
    const uint32_t b1 = __builtin_bit_cast(uint32_t, r1) & 0xFFFF0000u;
    const float r2 = r1 - __builtin_bit_cast(float, b1);  // exact, 8 bits
    wsh[e * R + d] = (bf16)__builtin_bit_cast(float, b0);
    wsh[(E + e) * R + d] = (bf16)__builtin_bit_cast(float, b1);
    wsh[(2 * E + e) * R + d] = (bf16)r2;
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int l16 = lane & 15, q = lane >> 4;
  const int t0 = (blockIdx.x * kRouterWaves + wave) * 16;
  const bf16* row = x + (size_t)min(t0 + l16, T - 1) * D;
  const bf16* wr = wsh + min(l16, E - 1) * R + 8 * q;
  f32x4 acc[3] = {f32x4{}, f32x4{}, f32x4{}};
  constexpr int kAhead = 8;  // steps whose loads are in flight together
  for (int d0 = 0; d0 < D; d0 += 32 * kAhead) {
    bf16x8 xv[kAhead];
#pragma unroll
    for (int j = 0; j < kAhead; ++j) xv[j] = load_x8<kVec>(row, d0 + 32 * j + 8 * q, D);
#pragma unroll
    for (int j = 0; j < kAhead; ++j) {
      const int d = d0 + 32 * j;
      if (d >= D) break;  // uniform
#pragma unroll
      for (int p = 0; p < 3; ++p)
        acc[p] = mfma16(xv[j], *reinterpret_cast<const bf16x8*>(wr + p * E * R + d), acc[p]);
    }
  }
  if (l16 < E) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = t0 + 4 * q + i;  // lane: expert l16, tokens 4 q .. 4 q + 3
      if (t >= T) continue;
      float s = acc[2][i] + acc[1][i] + acc[0][i];
      // An infinity or NaN: again as plain multiply-adds (the pieces of an
      // infinite weight are not its parts, inf - inf, and an infinite x makes a
      // NaN of a weight's zero pieces).
      if (!(fabsf(s) < INFINITY)) {
        s = 0.f;
        for (int d = 0; d < D; ++d) s = fmaf((float)x[(size_t)t * D + d], w[(size_t)d * E + l16], s);
      }
      logits[(size_t)t * E + l16] = s;
    }
  }
}

// ---------------------------------------------------------------------------
// Grouped GEMM over the expert buckets (megablox.gmm contract):
//   out[off_e + r][n] = sum_k A[off_e + r][k] * B_e(k, n),  r < counts[e],
// A K-major [R][K] (rows in bucket order), B_e either [K][N]
// (kBT = false: rhs + e*K*N) or [N][K] (kBT = true: the transpose, for dX).
// Grid: (ceil(R/256) + E) M-tile slots x ceil(N/256); surplus slots exit.
// Each 256 x 256 tile is computed transposed (features x bucket rows) and
// written through LDS in whole rows by the shared epilogue (epilogue.h),
// which also reads pre in whole rows for kMode 2.
// kMode 0: out = bf16(acc) (+ bias)
//       1: pre = bf16(bf16(acc) + bias), out = bf16(gelu(pre))
//       2: out = bf16(bf16(acc) * gelu'(pre))   (pre read, same layout as out)
// ---------------------------------------------------------------------------
template <bool kBT, int kMode>
__device__ __forceinline__ void moe_gmm_tile(int pid, const bf16* __restrict__ lhs, int64_t lda,
                                             const bf16* __restrict__ rhs, const int32_t* __restrict__ counts, int E,
                                             int K, int N, const bf16* __restrict__ bias, bf16* __restrict__ out,
                                             bf16* __restrict__ pre, int64_t ldo, float* bias_s) {
  const int ntn = (N + gemm::BN - 1) / gemm::BN;
  const int tn = pid % ntn;  // feature tile
  int tm = pid / ntn;        // bucket-row tile of expert e
  int e = 0, off = 0;
  for (; e < E; ++e) {
    const int c = counts[e];
    const int nt = (c + gemm::BM - 1) / gemm::BM;
    if (tm < nt) break;
    tm -= nt;
    off += c;
  }
  if (e >= E) return;  // uniform: surplus slot
  const int cnt = counts[e];
  // The tile is computed transposed (rows = output features, columns =
  // bucket rows), so it leaves through the shared token-row epilogue:
  // A = the expert's weight (K-major [N][K] when transposed, else MN-major
  // [K][N]), B = the bucket's rows (K-major).
  const gemm::Operand Wop = kBT ? gemm::Operand{rhs + (int64_t)e * N * K, K} : gemm::Operand{rhs + (int64_t)e * K * N, N};
  const gemm::Operand Xop{lhs + (int64_t)off * lda, lda};
  constexpr int kEpi = kMode == 0 ? gemm_epi::kBias : kMode == 1 ? gemm_epi::kGelu : gemm_epi::kDGelu;
  if constexpr (gemm_epi::has_bias(kEpi)) gemm_epi::stage_bias(bias_s, bias ? bias + (int64_t)e * N : nullptr, tn * gemm::BM, N);
  f32x16 acc[4][2];
  gemm::mainloop_pp<kBT, true>(acc, Wop, Xop, N, cnt, 0, K, tn * gemm::BM, tm * gemm::BN);
  gemm_epi::EpiArgs ea{};
  const int64_t base = (int64_t)off * ldo;
  if (kMode == 1) {
    ea.y = pre + base;  // h = bf16(bf16(acc) + b)
    ea.act = out + base;  // gelu(h)
  } else {
    ea.y = out + base;
  }
  ea.ldy = ldo;
  ea.aux = kMode == 2 ? pre + base : nullptr;
  ea.ldaux = ldo;
  gemm_epi::linear_epilogue<kEpi>(acc, tn, tm, N, cnt, ea, bias_s);
}

template <bool kBT, int kMode>
__global__ void __launch_bounds__(gemm::THREADS)
    moe_gmm_kernel(const bf16* __restrict__ lhs, int64_t lda,
                   const bf16* __restrict__ rhs, const int32_t* __restrict__ counts, int E, int K, int N,
                   const bf16* __restrict__ bias, bf16* __restrict__ out, bf16* __restrict__ pre, int64_t ldo) {
  __shared__ __attribute__((aligned(16))) float bias_s[gemm::BM];
  moe_gmm_tile<kBT, kMode>(blockIdx.x, lhs, lda, rhs, counts, E, K, N, bias, out, pre, ldo, bias_s);
}

// One tile of an expert's weight (+ bias) gradient over the rows [k_begin,
// k_end) of its bucket, which starts at row `off`:
//   dwe (f32 [K][N]) += sum_r A[r][k] * dy[r][n],  dbe (f32 [N], nullable) += sum_r dy[r][n],
// A [R][K] and dy [R][N] in bucket order; fp32 atomics, or, with store, dwe's
// tile overwritten (also by an empty row range).
__device__ __forceinline__ void moe_dw_tile(const bf16* __restrict__ lhs, int64_t lda, const bf16* __restrict__ dy,
                                            int64_t ldy, int off, int cnt, int k_begin, int k_end, int tile, int K,
                                            int N, float* __restrict__ dwe, float* __restrict__ dbe, bool store) {
  int tm, tn;
  gemm::tile_coords(tile, K, N, tm, tn);
  // A(m = k-index, k = bucket row) MN-major; B(k = bucket row, n) MN-major.
  gemm::Operand A{lhs + (int64_t)off * lda, lda};
  gemm::Operand B{dy + (int64_t)off * ldy, ldy};
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  f32x16 acc[4][2];
  float csum[2] = {0.f, 0.f};
  const bool do_colsum = dbe != nullptr;  // shared out over the M tiles
  gemm::mainloop_pp<false, false, true>(acc, A, B, K, N, k_begin, k_end, tm * gemm::BM, tn * gemm::BN, csum,
                                        do_colsum ? (K + gemm::BM - 1) / gemm::BM : 0, tm);
  const int hl = lane >> 5, l32 = lane & 31;
  const int wm = wave & 1, wn = wave >> 1;
#pragma unroll
  for (int nb = 0; nb < 2; ++nb) {
    const int n = tn * gemm::BN + 64 * wn + 32 * nb + l32;
    if (n >= N) continue;
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int m = tm * gemm::BM + 128 * wm + 32 * mb + 8 * (i >> 2) + 4 * hl + (i & 3);
        if (m >= K) continue;
        if (store)
          dwe[(int64_t)m * N + n] = acc[mb][nb][i];
        else
          atomicAdd(dwe + (int64_t)m * N + n, acc[mb][nb][i]);
      }
  }
  if (do_colsum && wm == 0) {
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
      const float t = csum[nb] + __shfl_xor(csum[nb], 32);
      const int n = tn * gemm::BN + 64 * wn + 32 * nb + l32;
      if (hl == 0 && n < N) atomicAdd(dbe + n, t);
    }
  }
}

// dw[e] += ..., db[e] += ... for every expert.  Grid: E x tiles(K, N) x split;
// bucket e's rows are split into `split` slices, whose partial tiles are added
// with fp32 atomics (measured no slower than a read-modify-write when a tile
// has one writer).
__global__ void __launch_bounds__(gemm::THREADS)
    moe_gmm_dw_kernel(const bf16* __restrict__ lhs, int64_t lda,
                      const bf16* __restrict__ dy, int64_t ldy, const int32_t* __restrict__ counts, int K, int N,
                      int split, float* __restrict__ dw, float* __restrict__ db) {
  const int tiles = ((K + gemm::BM - 1) / gemm::BM) * ((N + gemm::BN - 1) / gemm::BN);
  const int e = blockIdx.x / (tiles * split);
  const int rem = blockIdx.x % (tiles * split);
  const int sp = rem / tiles;
  int off = 0;
  for (int i = 0; i < e; ++i) off += counts[i];
  const int cnt = counts[e];
  const int kslice = ((cnt + split - 1) / split + gemm::BK - 1) / gemm::BK * gemm::BK;
  const int k_begin = sp * kslice;
  const int k_end = min(cnt, k_begin + kslice);
  if (k_begin >= k_end) return;  // uniform
  moe_dw_tile(lhs, lda, dy, ldy, off, cnt, k_begin, k_end, rem % tiles, K, N, dw + (int64_t)e * K * N,
              db ? db + (int64_t)e * N : nullptr, false);
}

// The three backward GEMMs that need only the pre-activation gradient dpre and
// what the forward kept, in one launch:
//   down_dw, down_db from (hidden, dout); up_dw, up_db from (grouped, dpre);
//   dgrouped = dpre up_w^T.
// Alone, each weight gradient leaves CUs idle (8 experts of 768 x 1536: 144
// tiles of 256-stage reductions for 256 CUs, 269 us) and so does the end of
// the input gradient's grid (201 us).  The weight-gradient items come first
// (the longest, handed out first), the short input-gradient tiles fill the CUs
// that are free: 32768 tokens x 768, top 2: 473 us for the three against 739.
// A bucket is cut into slices of `slice` rows (a multiple of BK): its tiles are
// stored when one slice holds it and added with atomics, to gradients that
// moe_zero_kernel cleared, when it takes more (an expert with many times its
// even share must not leave its tiles to a few workgroups).  The slots of a
// weight are experts + rows / slice slices, the most that any counts need;
// surplus ones exit.
struct MoeBwdGemms {
  const bf16 *grouped, *dpre, *hidden, *dout, *up_w;
  const int32_t* counts;
  float *up_dw, *up_db, *down_dw, *down_db;
  bf16* dgrouped;
  int width, hidden_width, experts, slice, n_slots, tiles;  // workgroups: n_slots x tiles down, as many up, dgrouped
};

__global__ void __launch_bounds__(gemm::THREADS) moe_bwd_gemms_kernel(MoeBwdGemms g) {
  __shared__ __attribute__((aligned(16))) float bias_s[gemm::BM];
  const int n_dw = g.n_slots * g.tiles;
  const int b = blockIdx.x;
  if (b < 2 * n_dw) {
    const bool down = b < n_dw;  // uniform
    const int item = down ? b : b - n_dw;
    int slot = item / g.tiles, e = 0, off = 0;
    for (; e < g.experts; ++e) {
      const int c = g.counts[e];
      const int n = c <= g.slice ? 1 : (c + g.slice - 1) / g.slice;  // (an empty bucket stores zeros)
      if (slot < n) break;
      slot -= n;
      off += c;
    }
    if (e >= g.experts) return;  // uniform: surplus slot
    const int cnt = g.counts[e];
    const int K = down ? g.hidden_width : g.width, N = down ? g.width : g.hidden_width;
    moe_dw_tile(down ? g.hidden : g.grouped, K, down ? g.dout : g.dpre, N, off, cnt, slot * g.slice,
                min(cnt, (slot + 1) * g.slice), item % g.tiles, K, N,
                (down ? g.down_dw : g.up_dw) + (int64_t)e * K * N, (down ? g.down_db : g.up_db) + (int64_t)e * N,
                cnt <= g.slice);
  } else {
    moe_gmm_tile<true, 0>(b - 2 * n_dw, g.dpre, g.hidden_width, g.up_w, g.counts, g.experts, g.hidden_width, g.width,
                          nullptr, g.dgrouped, nullptr, g.width, bias_s);
  }
}

// Clears what moe_bwd_gemms_kernel adds to: the bias gradients, and the weight
// gradients of the experts with more than one slice; with d_router (f32
// [width, experts]) that too, an even share per expert.  Grid: (x, experts).
__global__ void __launch_bounds__(256) moe_zero_kernel(MoeBwdGemms g, float* __restrict__ d_router) {
  const int e = blockIdx.y;
  const int i0 = (blockIdx.x * blockDim.x + threadIdx.x) * 4, step = gridDim.x * blockDim.x * 4;
  auto clear = [&](float* p, int64_t n) {
    for (int64_t i = i0; i < n; i += step) *reinterpret_cast<f32x4*>(p + i) = f32x4{};
  };
  clear(g.up_db + (int64_t)e * g.hidden_width, g.hidden_width);
  clear(g.down_db + (int64_t)e * g.width, g.width);
  if (d_router) clear(d_router + (int64_t)e * g.width, g.width);
  if (g.counts[e] <= g.slice) return;
  const int64_t nw = (int64_t)g.width * g.hidden_width;
  clear(g.up_dw + e * nw, nw);
  clear(g.down_dw + e * nw, nw);
}

// grouped[p] = x[rows[p]] (flat[rows], :1278): one wave per bucket row.
__global__ void __launch_bounds__(256) moe_gather_rows_kernel(const bf16* __restrict__ x, const int32_t* __restrict__ rows,
                                                              bf16* __restrict__ grouped, int R, int D) {
  const int p = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (p >= R) return;
  const int lane = threadIdx.x & 63;
  const bf16* src = x + (size_t)rows[p] * D;
  bf16* dst = grouped + (size_t)p * D;
  for (int c = lane * 8; c < D; c += 512) *reinterpret_cast<bf16x8*>(dst + c) = *reinterpret_cast<const bf16x8*>(src + c);
}

// Sort the (at most kMaxTopK) bucket positions of one token ascending.
constexpr int kMaxTopK = 8;
__device__ __forceinline__ void token_slots(const int32_t* __restrict__ position, const float* __restrict__ gate,
                                            int t, int k, int (&p)[kMaxTopK], float (&g)[kMaxTopK]) {
  for (int j = 0; j < k; ++j) {
    p[j] = position[(size_t)t * k + j];
    g[j] = gate ? (float)(bf16)gate[(size_t)t * k + j] : 0.f;
  }
  for (int a = 1; a < k; ++a)
    for (int b = a; b > 0 && p[b - 1] > p[b]; --b) {
      const int tp = p[b];
      p[b] = p[b - 1];
      p[b - 1] = tp;
      const float tg = g[b];
      g[b] = g[b - 1];
      g[b - 1] = tg;
    }
}

// combined[t] = bf16 sum, in bucket order, of bf16(out[p] * bf16(gate)):
// weighted = out * gate[order].astype(bf16); zeros.at[rows].add(weighted).
// K = top_k where it is 1 or 2 (0: any): every row of a token is then loaded
// before the first is used (32768 tokens x 768, top 2: 41 -> 27 us).
template <int K>
__global__ void __launch_bounds__(256) moe_combine_kernel(const bf16* __restrict__ out, const int32_t* __restrict__ position,
                                                          const float* __restrict__ gate, bf16* __restrict__ combined,
                                                          int T, int D, int k_any) {
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= T) return;
  const int lane = threadIdx.x & 63;
  const int k = K ? K : k_any;
  int p[kMaxTopK];
  float g[kMaxTopK];
  token_slots(position, gate, t, k, p, g);
  constexpr int kU = K ? 4 : 1;  // chunks of 4 columns per lane in flight
  for (int c0 = lane * 4; c0 < D; c0 += 256 * kU) {
    float acc[kU][4] = {};
    if constexpr (K > 0) {
      bf16x4 v[K][kU];
#pragma unroll
      for (int j = 0; j < K; ++j)
#pragma unroll
        for (int u = 0; u < kU; ++u)
          v[j][u] = c0 + 256 * u < D ? *reinterpret_cast<const bf16x4*>(out + (size_t)p[j] * D + c0 + 256 * u) : bf16x4{};
#pragma unroll
      for (int j = 0; j < K; ++j)
#pragma unroll
        for (int u = 0; u < kU; ++u)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            acc[u][q] = (float)(bf16)(acc[u][q] + (float)(bf16)((float)v[j][u][q] * g[j]));
    } else {
      for (int j = 0; j < k; ++j) {
        const bf16x4 v = *reinterpret_cast<const bf16x4*>(out + (size_t)p[j] * D + c0);
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[0][q] = (float)(bf16)(acc[0][q] + (float)(bf16)((float)v[q] * g[j]));
      }
    }
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      if (c0 + 256 * u >= D) break;
      bf16x4 o = {(bf16)acc[u][0], (bf16)acc[u][1], (bf16)acc[u][2], (bf16)acc[u][3]};
      *reinterpret_cast<bf16x4*>(combined + (size_t)t * D + c0 + 256 * u) = o;
    }
  }
}

// Backward of the combine: dout[p] = bf16(dcombined[t] * bf16(gate[a])),
// dgate[a] = sum_n dcombined[t][n] * out[p][n] (fp32), a = t*k + j, p = position[a].
__global__ void __launch_bounds__(256) moe_combine_bwd_kernel(const bf16* __restrict__ dcombined,
                                                              const bf16* __restrict__ out,
                                                              const int32_t* __restrict__ position,
                                                              const float* __restrict__ gate, bf16* __restrict__ dout,
                                                              float* __restrict__ dgate, int T, int D, int k) {
  const int a = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (a >= T * k) return;
  const int lane = threadIdx.x & 63;
  const int t = a / k, p = position[a];
  const float g = (float)(bf16)gate[a];
  float dot = 0.f;
  for (int c = lane * 4; c < D; c += 256) {
    const bf16x4 dc = *reinterpret_cast<const bf16x4*>(dcombined + (size_t)t * D + c);
    const bf16x4 ov = *reinterpret_cast<const bf16x4*>(out + (size_t)p * D + c);
    bf16x4 o;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      o[q] = (bf16)((float)dc[q] * g);
      dot = fmaf((float)dc[q], (float)ov[q], dot);
    }
    *reinterpret_cast<bf16x4*>(dout + (size_t)p * D + c) = o;
  }
  dot = wave_sum(dot);
  if (lane == 0) dgate[a] = dot;
}

// VJP of grouped = flat[rows]: dx[t] = bf16 sum, in bucket order, of dgrouped[p].
__global__ void __launch_bounds__(256) moe_gather_bwd_kernel(const bf16* __restrict__ dgrouped,
                                                             const int32_t* __restrict__ position,
                                                             bf16* __restrict__ dx, int T, int D, int k) {
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= T) return;
  const int lane = threadIdx.x & 63;
  int p[kMaxTopK];
  float g[kMaxTopK];
  token_slots(position, nullptr, t, k, p, g);
  for (int c = lane * 4; c < D; c += 256) {
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (int j = 0; j < k; ++j) {
      const bf16x4 v = *reinterpret_cast<const bf16x4*>(dgrouped + (size_t)p[j] * D + c);
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[q] = (float)(bf16)(acc[q] + (float)v[q]);
    }
    bf16x4 o = {(bf16)acc[0], (bf16)acc[1], (bf16)acc[2], (bf16)acc[3]};
    *reinterpret_cast<bf16x4*>(dx + (size_t)t * D + c) = o;
  }
}

// Router statistics (:1295-1306): the sums of probabilities, entropies,
// top-1 gates and squared logits over the tokens, in three launches:
// stats_zero clears the outputs, moe_stats_kernel (one thread per token)
// adds each workgroup's sums into them with atomics, stats_finalize divides
// (and takes the root of the mean square) and writes the load.
__global__ void stats_zero_kernel(float* __restrict__ mean_probability, float* __restrict__ summary, int E) {
  const int i = threadIdx.x;
  if (i < E) mean_probability[i] = 0.f;
  if (i < 3) summary[i] = 0.f;
}

template <int EP>
__global__ void __launch_bounds__(256) moe_stats_kernel(const float* __restrict__ logits, const float* __restrict__ probs,
                                                        const float* __restrict__ gate, int T, int E, int k,
                                                        float* __restrict__ mean_probability,
                                                        float* __restrict__ summary) {
  __shared__ float red[3 + EP][4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int t = blockIdx.x * blockDim.x + tid;
  float pe[EP], ent = 0.f, top = 0.f, sq = 0.f;
#pragma unroll
  for (int e = 0; e < EP; ++e) pe[e] = 0.f;
  if (t < T) {
#pragma unroll
    for (int e = 0; e < EP; ++e) {
      if (e < E) {
        const float pv = probs[(size_t)t * E + e];
        const float lv = logits[(size_t)t * E + e];
        pe[e] = pv;
        ent -= pv * logf(pv + 1.0e-9f);
        sq = fmaf(lv, lv, sq);
      }
    }
    float gm = gate[(size_t)t * k];
    for (int j = 1; j < k; ++j) gm = fmaxf(gm, gate[(size_t)t * k + j]);
    top = gm;
  }
  float vals[3] = {ent, top, sq};
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    const float v = wave_sum(vals[q]);
    if (lane == 0) red[q][wave] = v;
  }
#pragma unroll
  for (int e = 0; e < EP; ++e) {
    if (e < E) {
      const float v = wave_sum(pe[e]);
      if (lane == 0) red[3 + e][wave] = v;
    }
  }
  __syncthreads();
  if (tid < 3 + E) {
    const float v = red[tid][0] + red[tid][1] + red[tid][2] + red[tid][3];
    atomicAdd(tid < 3 ? summary + tid : mean_probability + (tid - 3), v);
  }
}

__global__ void stats_finalize_kernel(const int32_t* __restrict__ counts, int T, int E, int k,
                                      float* __restrict__ mean_probability, float* __restrict__ load,
                                      float* __restrict__ summary) {
  const int i = threadIdx.x;
  if (i < E) {
    mean_probability[i] = mean_probability[i] / T;
    load[i] = (float)counts[i] / (float)((long long)T * k);
  }
  if (i == 0) {
    summary[0] = summary[0] / T;
    summary[1] = summary[1] / T;
    summary[2] = sqrtf(summary[2] / ((float)T * E));
  }
}

// Router backward, per token t:
//   dchosen[j] = gate[j] * (dgate[j] - sum_i gate[i] dgate[i])        (gate softmax)
//   dprobs[e]  = dmean_probability[e] / T                              (mean over tokens)
//   dlogits[e] = probs[e] * (dprobs[e] - sum_i probs[i] dprobs[i]) + sum_{j: chosen[j]=e} dchosen[j]
//   dx[t][d]   = bf16(dx[t][d] + bf16(sum_e dlogits[e] w[d][e]))       (in place)
//   dw[d][e]  += sum_t f32(x[t][d]) dlogits[e]
// A workgroup takes kRouterBwdCols width columns and a run of tokens, in
// tiles of kRouterBwdTokens.  Its threads first turn each token's gate and
// probability cotangents into dlogits (LDS); then thread (token lane tl,
// chunk c) walks tokens tl, tl + 32, ... of the tile for the 8 columns 8 c ..
// 8 c + 7: dx[t][chunk] gets bf16(dlogits[t] @ w[chunk]^T) added and the
// chunk's dw partial f32 [8][EP] grows in registers.  After the last tile the
// 32 token lanes' partials are summed with xor exchanges and through LDS, and
// the workgroup adds one value per (column, expert) to dw with an atomic.  The
// grid is one or two workgroups per CU: every workgroup of a column tile adds to
// the same few cache lines, and those adds run one after the other (32768 tokens
// x 768, inputs past the caches: 84 workgroups per column tile 84 us, 42 72, 21 81).
// kGather >= 0: the row the router's part is added to is not read from dx but
// is the VJP of grouped = flat[rows], the bf16 sum of the token's rows of
// dgrouped in bucket order (moe_gather_bwd_kernel's), so dx is written once and
// never read: at 32768 tokens x 768, top 2, 72 us against 36 + 62 us for the
// two passes.  kGather is top_k where it is 1 or 2 (0: any), so the loops over
// a token's slots unroll and their loads go out together; four tokens' loads
// are in flight per thread.
constexpr int kRouterBwdTokens = 256;
constexpr int kRouterBwdCols = 64;

template <int EP, int kGather>
__global__ void __launch_bounds__(256) router_bwd_kernel(const bf16* __restrict__ x, const float* __restrict__ w,
                                                         const float* __restrict__ probs, const int32_t* __restrict__ chosen,
                                                         const float* __restrict__ gate, const float* __restrict__ dgate,
                                                         const float* __restrict__ dmean_probability,
                                                         const bf16* __restrict__ dgrouped,
                                                         const int32_t* __restrict__ position, bf16* __restrict__ dx,
                                                         float* __restrict__ dw, int T, int D, int E, int k_any,
                                                         int run) {
  constexpr bool kFused = kGather >= 0;
  const int k = kGather > 0 ? kGather : k_any;
  __shared__ __attribute__((aligned(16))) float dl_s[kRouterBwdTokens][EP];
  __shared__ int pos_s[kFused ? kRouterBwdTokens : 1][kMaxTopK];
  __shared__ float red[4][kRouterBwdCols][EP];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // Column tiles fastest: the workgroups of one run of tokens run together and
  // share its rows' cache lines.
  const int ncol = (D + kRouterBwdCols - 1) / kRouterBwdCols;
  const int col0 = blockIdx.x % ncol * kRouterBwdCols;
  const int t_begin = (int)(blockIdx.x / ncol) * run, t_end = min(T, t_begin + run);
  const int c = tid & 7, tl = tid >> 3;  // chunk of the tile, token lane (0 .. 31)
  const int d0 = col0 + 8 * c;
  const bool vec = (D & 7) == 0 && d0 + 8 <= D;  // (kFused: D is a multiple of 8)
  float wc[8][EP], dwp[8][EP];
#pragma unroll
  for (int j = 0; j < 8; ++j)
#pragma unroll
    for (int e = 0; e < EP; ++e) {
      wc[j][e] = (d0 + j < D && e < E) ? w[(size_t)(d0 + j) * E + e] : 0.f;
      dwp[j][e] = 0.f;
    }
  for (int tb = t_begin; tb < t_end; tb += kRouterBwdTokens) {
    __syncthreads();  // the previous tile's dlogits are read
    {
      static_assert(kRouterBwdTokens == 256, "one token per thread");
      const int t = tb + tid;
      float dl[EP];
#pragma unroll
      for (int e = 0; e < EP; ++e) dl[e] = 0.f;
      if (t < t_end) {
        if (dmean_probability) {
          float pd = 0.f;
#pragma unroll
          for (int e = 0; e < EP; ++e)
            if (e < E) pd += probs[(size_t)t * E + e] * (dmean_probability[e] / T);
#pragma unroll
          for (int e = 0; e < EP; ++e)
            if (e < E) dl[e] = probs[(size_t)t * E + e] * (dmean_probability[e] / T - pd);
        }
        float gd = 0.f;
        for (int j = 0; j < k; ++j) gd += gate[(size_t)t * k + j] * dgate[(size_t)t * k + j];
        for (int j = 0; j < k; ++j) {
          const float dc = gate[(size_t)t * k + j] * (dgate[(size_t)t * k + j] - gd);
          const int ce = chosen[(size_t)t * k + j];
#pragma unroll
          for (int e = 0; e < EP; ++e)
            if (e == ce) dl[e] += dc;
        }
        if constexpr (kFused) {
          int p[kMaxTopK];
          float g[kMaxTopK];
          token_slots(position, nullptr, t, k, p, g);
          for (int j = 0; j < k; ++j) pos_s[tid][j] = p[j];
        }
      }
#pragma unroll
      for (int e = 0; e < EP; ++e) dl_s[tid][e] = dl[e];
    }
    __syncthreads();
    constexpr int kU = EP <= 8 ? 4 : 2;  // tokens in flight
    if (d0 < D) {
      for (int i0 = tl; i0 < kRouterBwdTokens; i0 += 32 * kU) {
        if (tb + i0 >= t_end) break;
        bf16x8 xx[kU], old[kU];
        // (Tokens past the run read its last token's rows; their dlogits are zero and
        // nothing of them is stored.)
        int ts[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) ts[u] = min(tb + i0 + 32 * u, t_end - 1);
        if (kFused || vec) {
#pragma unroll
          for (int u = 0; u < kU; ++u) xx[u] = *reinterpret_cast<const bf16x8*>(x + (size_t)ts[u] * D + d0);
        } else {
#pragma unroll
          for (int u = 0; u < kU; ++u)
#pragma unroll
            for (int j = 0; j < 8; ++j) {
              xx[u][j] = d0 + j < D ? x[(size_t)ts[u] * D + d0 + j] : (bf16)0.f;
              old[u][j] = d0 + j < D ? dx[(size_t)ts[u] * D + d0 + j] : (bf16)0.f;
            }
        }
        if constexpr (kGather == 1 || kGather == 2) {
          bf16x8 gv[kU][kGather];
#pragma unroll
          for (int u = 0; u < kU; ++u)
#pragma unroll
            for (int j = 0; j < kGather; ++j)
              gv[u][j] = *reinterpret_cast<const bf16x8*>(dgrouped + (size_t)pos_s[ts[u] - tb][j] * D + d0);
#pragma unroll
          for (int u = 0; u < kU; ++u)
#pragma unroll
            for (int q = 0; q < 8; ++q)
              old[u][q] = kGather == 1 ? gv[u][0][q] : (bf16)((float)gv[u][0][q] + (float)gv[u][kGather - 1][q]);
        } else if constexpr (kFused) {
#pragma unroll
          for (int u = 0; u < kU; ++u) {
            float acc[8] = {};
            for (int j = 0; j < k; ++j) {
              const bf16x8 v = *reinterpret_cast<const bf16x8*>(dgrouped + (size_t)pos_s[ts[u] - tb][j] * D + d0);
#pragma unroll
              for (int q = 0; q < 8; ++q) acc[q] = (float)(bf16)(acc[q] + (float)v[q]);
            }
            old[u] = pack8(acc);
          }
        } else if (vec) {
#pragma unroll
          for (int u = 0; u < kU; ++u) old[u] = *reinterpret_cast<const bf16x8*>(dx + (size_t)ts[u] * D + d0);
        }
#pragma unroll
        for (int u = 0; u < kU; ++u) {
          const int i = i0 + 32 * u;
          float dl[EP];
#pragma unroll
          for (int e4 = 0; e4 < EP; e4 += 4) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(&dl_s[i][e4]);
#pragma unroll
            for (int r = 0; r < 4; ++r) dl[e4 + r] = v[r];
          }
          bf16x8 o;
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            float sj = 0.f;
#pragma unroll
            for (int e = 0; e < EP; ++e) {
              sj = fmaf(dl[e], wc[j][e], sj);
              dwp[j][e] = fmaf((float)xx[u][j], dl[e], dwp[j][e]);
            }
            o[j] = (bf16)((float)old[u][j] + (float)(bf16)sj);
          }
          if (tb + i >= t_end) continue;
          bf16* drow = dx + (size_t)(tb + i) * D + d0;
          if (kFused || vec) {
            *reinterpret_cast<bf16x8*>(drow) = o;
          } else {
#pragma unroll
            for (int j = 0; j < 8; ++j)
              if (d0 + j < D) drow[j] = o[j];
          }
        }
      }
    }
  }
  // Sum the token lanes: lanes 8 m + c of a wave (m = 0..7) by xor over
  // lane bits 3..5, then the 4 waves through LDS.
#pragma unroll
  for (int j = 0; j < 8; ++j)
#pragma unroll
    for (int e = 0; e < EP; ++e) {
      float v = dwp[j][e];
      v += __shfl_xor(v, 8);
      v += __shfl_xor(v, 16);
      v += __shfl_xor(v, 32);
      if (lane < 8) red[wave][8 * c + j][e] = v;
    }
  __syncthreads();
  for (int i = tid; i < kRouterBwdCols * EP; i += blockDim.x) {
    const int col = i / EP, e = i % EP;
    const float v = red[0][col][e] + red[1][col][e] + red[2][col][e] + red[3][col][e];
    if (col0 + col < D && e < E) atomicAdd(dw + (size_t)(col0 + col) * E + e, v);
  }
}

template <int EP>
void launch_router_bwd(unsigned grid, int run, hipStream_t s, const bf16* x, const float* w, const float* probs,
                       const int32_t* chosen, const float* gate, const float* dgate, const float* dmean,
                       const bf16* dgrouped, const int32_t* position, bf16* dx, float* dw, int T, int D, int E, int k) {
  auto* kernel = !dgrouped ? router_bwd_kernel<EP, -1>
                 : k == 1  ? router_bwd_kernel<EP, 1>
                 : k == 2  ? router_bwd_kernel<EP, 2>
                           : router_bwd_kernel<EP, 0>;
  kernel<<<grid, 256, 0, s>>>(x, w, probs, chosen, gate, dgate, dmean, dgrouped, position, dx, dw, T, D, E, k, run);
}

int router_bwd(const void* x, const float* router_w, const float* probs, const int32_t* chosen, const float* gate,
               const float* dgate, const float* dmean_probability, const void* dgrouped, const int32_t* position,
               void* dx, float* dw_router, int tokens, int width, int experts, int top_k, void* stream) {
  if (!x || !router_w || !probs || !chosen || !gate || !dgate || !dx || !dw_router) return GPTRIG_E_NULL;
  if (tokens <= 0 || width <= 0 || experts <= 0 || top_k <= 0 || top_k > experts) return GPTRIG_E_SHAPE;
  if (experts > kMaxRouterExperts || (size_t)width * experts * sizeof(float) > 32768) return GPTRIG_E_UNSUPPORTED;
  const int ncol = ceil_div(width, kRouterBwdCols);
  int runs = gemm::device_cus() / ncol > 1 ? gemm::device_cus() / ncol : 1;
  // Two workgroups fit a CU up to 8 experts; where each still has a whole tile of
  // tokens they are worth the second round of adds (gathered / two-pass form, one and
  // two per CU, 32768 tokens, inputs past the caches: 2048 columns 148 -> 138 / 124 ->
  // 106 us, 1024 99 -> 88 / 86 -> 73, 768 81 -> 72 / 74 -> 62, 512 58 -> 57 / 51 -> 50;
  // 8192 x 1024 35 -> 35; but 4096 x 512 18 -> 21, and 16 experts of 512 90 -> 111).
  if (experts <= 8 && tokens / (2 * runs) >= kRouterBwdTokens) runs *= 2;
  // Tokens per workgroup: an even share, in whole sweeps of the 32 token lanes.
  const int run = ceil_div(ceil_div(tokens, runs), 32) * 32;
  const unsigned grid = (unsigned)ncol * (unsigned)ceil_div(tokens, run);
  (experts <= 4   ? launch_router_bwd<4>
   : experts <= 8 ? launch_router_bwd<8>
                  : launch_router_bwd<16>)(grid, run, (hipStream_t)stream, (const bf16*)x, router_w, probs, chosen, gate,
                                           dgate, dmean_probability, (const bf16*)dgrouped, position, (bf16*)dx,
                                           dw_router, tokens, width, experts, top_k);
  GPTRIG_CHECK_LAUNCH();
  return GPTRIG_OK;
}

// gptrig_moe_bwd_gemms; d_router (nullable, f32 [width, experts]) is cleared too.
int moe_bwd_gemms(const void* grouped, const void* dpre, const void* hidden, const void* dout, const void* up_w,
                         const int32_t* counts, float* up_dw, float* up_db, float* down_dw, float* down_db,
                         void* dgrouped, int rows, int width, int hidden_width, int experts, float* d_router, void* stream) {
  if (!grouped || !dpre || !hidden || !dout || !up_w || !counts || !up_dw || !up_db || !down_dw || !down_db || !dgrouped)
    return GPTRIG_E_NULL;
  if (rows <= 0 || width <= 0 || hidden_width <= 0 || experts <= 0 || width % 8 || hidden_width % 8)
    return GPTRIG_E_SHAPE;
  if (((uintptr_t)grouped | (uintptr_t)dpre | (uintptr_t)hidden | (uintptr_t)dout | (uintptr_t)up_w |
       (uintptr_t)dgrouped | (uintptr_t)up_dw | (uintptr_t)up_db | (uintptr_t)down_dw | (uintptr_t)down_db) & 15)
    return GPTRIG_E_SHAPE;
  if (experts > kMaxExperts) return GPTRIG_E_UNSUPPORTED;
  hipStream_t s = (hipStream_t)stream;
  const int cus = gemm::device_cus();
  // Both weights have the same number of 256 x 256 tiles.
  const int tiles = ceil_div(hidden_width, gemm::BM) * ceil_div(width, gemm::BN);
  const int n_dx = (ceil_div(rows, gemm::BM) + experts) * ceil_div(width, gemm::BN);
  // Slices per evenly filled bucket, from the estimated makespan: stages of 32
  // rows plus an epilogue (10 for a plain store, 60 for the atomic add of a
  // tile, measured in the FLCE gradient launches), the longest items first.
  const int stages = ceil_div(ceil_div(rows, experts), gemm::BK);
  const double dx_cost = (double)ceil_div(rows, gemm::BM) * ceil_div(width, gemm::BN) *
                         ((double)ceil_div(hidden_width, gemm::BK) + 10.0);
  int split = 1;
  double best = 1e300;
  for (int k = 1; k <= 64 && (k == 1 || stages / k >= 8); ++k) {
    const double item = ceil_div(stages, k) + (k > 1 ? 60.0 : 10.0);
    const int64_t items = 2ll * tiles * experts * k;
    const double rounds = (double)ceil_div(items, (int64_t)cus) * item;
    const double even = ((double)items * item + dx_cost) / cus;
    const double cost = rounds > even ? rounds : even;
    if (cost < best * 0.999) {
      best = cost;
      split = k;
    }
  }
  // One slice holds a bucket of up to twice the even share.
  const int64_t slice = split == 1 ? 2ll * stages * gemm::BK : (int64_t)ceil_div(stages, split) * gemm::BK;
  const int slots = experts + (int)(rows / slice);
  MoeBwdGemms g{(const bf16*)grouped, (const bf16*)dpre, (const bf16*)hidden, (const bf16*)dout, (const bf16*)up_w,
                counts, up_dw, up_db, down_dw, down_db, (bf16*)dgrouped, width, hidden_width, experts,
                (int)(slice < (1 << 30) ? slice : (1 << 30)), slots, tiles};
  moe_zero_kernel<<<dim3(32, (unsigned)experts), 256, 0, s>>>(g, d_router);
  GPTRIG_CHECK_LAUNCH();
  moe_bwd_gemms_kernel<<<2u * (unsigned)slots * (unsigned)tiles + (unsigned)n_dx, gemm::THREADS, 0, s>>>(g);
  GPTRIG_CHECK_LAUNCH();
  return GPTRIG_OK;
}

}  // namespace

extern "C" {

size_t gptrig_moe_route_workspace_bytes(int tokens, int experts, int top_k) {
  if (tokens <= 0 || experts <= 0 || top_k <= 0) return 0;
  const size_t blocks = (size_t)ceil_div((int64_t)tokens * top_k, kSortBlock);
  return (blocks * experts * sizeof(int32_t) + 255) & ~(size_t)255;
}

int gptrig_moe_route(const float* logits, float* probs, int32_t* chosen, float* gate, int32_t* counts,
                     int32_t* order, int32_t* rows, int32_t* position, void* workspace, size_t workspace_bytes,
                     int tokens, int experts, int top_k, void* stream) {
  if (!logits || !chosen || !gate || !counts || !order || !rows) return GPTRIG_E_NULL;
  if (tokens <= 0 || experts <= 0 || top_k <= 0) return GPTRIG_E_SHAPE;
  if (experts > kMaxExperts || top_k > experts) return GPTRIG_E_UNSUPPORTED;
  if ((int64_t)tokens * top_k >= (1ll << 31)) return GPTRIG_E_SHAPE;
  if (!workspace || workspace_bytes < gptrig_moe_route_workspace_bytes(tokens, experts, top_k))
    return GPTRIG_E_WORKSPACE;
  hipStream_t s = (hipStream_t)stream;
  (experts <= 4    ? route_topk_kernel<4>
   : experts <= 8  ? route_topk_kernel<8>
   : experts <= 16 ? route_topk_kernel<16>
                   : route_topk_kernel<kMaxExperts>)<<<ceil_div(tokens, 128), 128, 0, s>>>(logits, probs, chosen, gate,
                                                                                           tokens, experts, top_k);
  GPTRIG_CHECK_LAUNCH();
  const int n_slots = tokens * top_k, nblocks = ceil_div(n_slots, kSortBlock);
  int32_t* hist = (int32_t*)workspace;
  route_hist_kernel<<<nblocks, kSortBlock, 0, s>>>(chosen, n_slots, experts, hist);
  GPTRIG_CHECK_LAUNCH();
  route_place_kernel<<<nblocks, kSortBlock, 0, s>>>(chosen, n_slots, experts, top_k, hist, nblocks, counts, order,
                                                    rows, position);
  GPTRIG_CHECK_LAUNCH();
  return GPTRIG_OK;
}


int gptrig_moe_router_logits(const void* x, const float* router_w, float* logits, int tokens, int width, int experts,
                             void* stream) {
  if (!x || !router_w || !logits) return GPTRIG_E_NULL;
  if (tokens <= 0 || width <= 0 || experts <= 0) return GPTRIG_E_SHAPE;
  if (experts > kMaxRouterExperts || (size_t)width * experts * sizeof(float) > 32768) return GPTRIG_E_UNSUPPORTED;
  const size_t smem = (size_t)3 * experts * router_row(width) * sizeof(bf16);  // at most 54 KB
  const unsigned grid = (unsigned)ceil_div(tokens, 16 * kRouterWaves);
  // 16-byte loads of token rows.
  (width % 8 == 0 && ((uintptr_t)x & 15) == 0 ? router_logits_kernel<true> : router_logits_kernel<false>)<<<
      grid, 64 * kRouterWaves, smem, (hipStream_t)stream>>>((const bf16*)x, router_w, logits, tokens, width, experts);
  GPTRIG_CHECK_LAUNCH();
  return GPTRIG_OK;
}

int gptrig_moe_gather_rows(const void* x, const int32_t* rows, void* grouped, int n_rows, int width, void* stream) {
  if (!x || !rows || !grouped) return GPTRIG_E_NULL;
  if (n_rows <= 0 || width <= 0 || width % 8) return GPTRIG_E_SHAPE;
  if (((uintptr_t)x | (uintptr_t)grouped) & 15) return GPTRIG_E_SHAPE;
  moe_gather_rows_kernel<<<ceil_div(n_rows, 4), 256, 0, (hipStream_t)stream>>>((const bf16*)x, rows, (bf16*)grouped,
                                                                               n_rows, width);
  GPTRIG_CHECK_LAUNCH();
  return GPTRIG_OK;
}

int gptrig_moe_gmm(const void* lhs, int64_t lda, const void* rhs, int rhs_transposed, const int32_t* counts,
                   const void* bias, int mode, void* out, void* pre, int64_t ldo, int rows, int k, int n, int experts,
                   void* stream) {
  if (!lhs || !rhs || !counts || !out) return GPTRIG_E_NULL;
  if ((mode == 1 || mode == 2) && !pre) return GPTRIG_E_NULL;
  if (rows <= 0 || k <= 0 || n <= 0 || experts <= 0 || mode < 0 || mode > 2) return GPTRIG_E_SHAPE;
  if (k % 8 || n % 8 || lda % 8 || lda < k || ldo < n || ldo % 8) return GPTRIG_E_SHAPE;
  if (((uintptr_t)lhs | (uintptr_t)rhs | (uintptr_t)out | (uintptr_t)pre) & 15) return GPTRIG_E_SHAPE;
  if (experts > kMaxExperts) return GPTRIG_E_UNSUPPORTED;
  const unsigned grid = (unsigned)((ceil_div(rows, gemm::BM) + experts) * ceil_div(n, gemm::BN));
  hipStream_t s = (hipStream_t)stream;
  const bf16* L = (const bf16*)lhs;
  const bf16* Rh = (const bf16*)rhs;
  const bf16* Bi = (const bf16*)bias;
  bf16* O = (bf16*)out;
  bf16* P = (bf16*)pre;
#define GPTRIG_GMM(BT, MODE)                                                                                     \
  moe_gmm_kernel<BT, MODE><<<grid, gemm::THREADS, 0, s>>>(L, lda, Rh, counts, experts, k, n, Bi, O, P, ldo)
  if (rhs_transposed) {
    if (mode == 0) GPTRIG_GMM(true, 0);
    else if (mode == 1) GPTRIG_GMM(true, 1);
    else GPTRIG_GMM(true, 2);
  } else {
    if (mode == 0) GPTRIG_GMM(false, 0);
    else if (mode == 1) GPTRIG_GMM(false, 1);
    else GPTRIG_GMM(false, 2);
  }
#undef GPTRIG_GMM
  GPTRIG_CHECK_LAUNCH();
  return GPTRIG_OK;
}

int gptrig_moe_gmm_dw(const void* lhs, int64_t lda, const void* dy, int64_t ldy, const int32_t* counts, float* dw,
                      float* db, int rows, int k, int n, int experts, void* stream) {
  if (!lhs || !dy || !counts || !dw) return GPTRIG_E_NULL;
  if (rows <= 0 || k <= 0 || n <= 0 || experts <= 0) return GPTRIG_E_SHAPE;
  if (k % 8 || n % 8 || lda % 8 || ldy % 8 || lda < k || ldy < n) return GPTRIG_E_SHAPE;
  if (((uintptr_t)lhs | (uintptr_t)dy) & 15) return GPTRIG_E_SHAPE;
  if (experts > kMaxExperts) return GPTRIG_E_UNSUPPORTED;
  const unsigned tiles = (unsigned)(ceil_div(k, gemm::BM) * ceil_div(n, gemm::BN));
  // No split once E x tiles fills the GPU (every split adds an atomic
  // epilogue per tile); below that, short split blocks, which in the training
  // step also leave room for the main stream's kernels beside this one (on
  // the weight-gradient stream): config E measured 46.6 ms/step with them
  // against 49.2 ms with 144 unsplit blocks, and 60.7 against 62.5 ms with
  // 288 unsplit blocks instead of split ones.
  const int64_t cells = (int64_t)tiles * experts;
  const int split = cells >= gemm::device_cus() ? 1 : gemm::choose_split(tiles * experts,
                                                                         ceil_div(ceil_div(rows, experts), gemm::BK));
  moe_gmm_dw_kernel<<<tiles * experts * split, gemm::THREADS, 0, (hipStream_t)stream>>>(
      (const bf16*)lhs, lda, (const bf16*)dy, ldy, counts, k, n, split, dw, db);
  GPTRIG_CHECK_LAUNCH();
  return GPTRIG_OK;
}

int gptrig_moe_bwd_gemms(const void* grouped, const void* dpre, const void* hidden, const void* dout, const void* up_w,
                         const int32_t* counts, float* up_dw, float* up_db, float* down_dw, float* down_db,
                         void* dgrouped, int rows, int width, int hidden_width, int experts, void* stream) {
  return moe_bwd_gemms(grouped, dpre, hidden, dout, up_w, counts, up_dw, up_db, down_dw, down_db, dgrouped, rows, width,
                       hidden_width, experts, nullptr, stream);
}

int gptrig_moe_combine(const void* out, const int32_t* position, const float* gate, void* combined, int tokens,
                       int width, int top_k, void* stream) {
  if (!out || !position || !gate || !combined) return GPTRIG_E_NULL;
  if (tokens <= 0 || width <= 0 || top_k <= 0 || width % 8) return GPTRIG_E_SHAPE;
  if (top_k > kMaxTopK) return GPTRIG_E_UNSUPPORTED;
  (top_k == 1   ? moe_combine_kernel<1>
   : top_k == 2 ? moe_combine_kernel<2>
                : moe_combine_kernel<0>)<<<ceil_div(tokens, 4), 256, 0, (hipStream_t)stream>>>(
      (const bf16*)out, position, gate, (bf16*)combined, tokens, width, top_k);
  GPTRIG_CHECK_LAUNCH();
  return GPTRIG_OK;
}

int gptrig_moe_combine_bwd(const void* dcombined, const void* out, const int32_t* position, const float* gate,
                           void* dout, float* dgate, int tokens, int width, int top_k, void* stream) {
  if (!dcombined || !out || !position || !gate || !dout || !dgate) return GPTRIG_E_NULL;
  if (tokens <= 0 || width <= 0 || top_k <= 0 || width % 8) return GPTRIG_E_SHAPE;
  if (top_k > kMaxTopK) return GPTRIG_E_UNSUPPORTED;
  moe_combine_bwd_kernel<<<ceil_div((long long)tokens * top_k, 4), 256, 0, (hipStream_t)stream>>>(
      (const bf16*)dcombined, (const bf16*)out, position, gate, (bf16*)dout, dgate, tokens, width, top_k);
  GPTRIG_CHECK_LAUNCH();
  return GPTRIG_OK;
}

int gptrig_moe_gather_bwd(const void* dgrouped, const int32_t* position, void* dx, int tokens, int width, int top_k,
                          void* stream) {
  if (!dgrouped || !position || !dx) return GPTRIG_E_NULL;
  if (tokens <= 0 || width <= 0 || top_k <= 0 || width % 8) return GPTRIG_E_SHAPE;
  if (top_k > kMaxTopK) return GPTRIG_E_UNSUPPORTED;
  moe_gather_bwd_kernel<<<ceil_div(tokens, 4), 256, 0, (hipStream_t)stream>>>((const bf16*)dgrouped, position,
                                                                             (bf16*)dx, tokens, width, top_k);
  GPTRIG_CHECK_LAUNCH();
  return GPTRIG_OK;
}

int gptrig_moe_stats(const float* logits, const float* probs, const float* gate, const int32_t* counts, int tokens,
                     int experts, int top_k, float* mean_probability, float* load, float* summary, void* stream) {
  if (!logits || !probs || !gate || !counts || !mean_probability || !load || !summary) return GPTRIG_E_NULL;
  if (tokens <= 0 || experts <= 0 || top_k <= 0 || top_k > experts) return GPTRIG_E_SHAPE;
  if (experts > kMaxRouterExperts) return GPTRIG_E_UNSUPPORTED;
  hipStream_t s = (hipStream_t)stream;
  stats_zero_kernel<<<1, 64, 0, s>>>(mean_probability, summary, experts);
  GPTRIG_CHECK_LAUNCH();
  const unsigned grid = (unsigned)ceil_div(tokens, 256);
  if (experts <= 4)
    moe_stats_kernel<4><<<grid, 256, 0, s>>>(logits, probs, gate, tokens, experts, top_k, mean_probability, summary);
  else if (experts <= 8)
    moe_stats_kernel<8><<<grid, 256, 0, s>>>(logits, probs, gate, tokens, experts, top_k, mean_probability, summary);
  else
    moe_stats_kernel<16><<<grid, 256, 0, s>>>(logits, probs, gate, tokens, experts, top_k, mean_probability, summary);
  GPTRIG_CHECK_LAUNCH();
  stats_finalize_kernel<<<1, 64, 0, s>>>(counts, tokens, experts, top_k, mean_probability, load, summary);
  GPTRIG_CHECK_LAUNCH();
  return GPTRIG_OK;
}

int gptrig_moe_router_bwd(const void* x, const float* router_w, const float* probs, const int32_t* chosen,
                          const float* gate, const float* dgate, const float* dmean_probability, void* dx,
                          float* dw_router, int tokens, int width, int experts, int top_k, void* stream) {
  return router_bwd(x, router_w, probs, chosen, gate, dgate, dmean_probability, nullptr, nullptr, dx, dw_router,
                    tokens, width, experts, top_k, stream);
}

int gptrig_moe_input_bwd(const void* dgrouped, const int32_t* position, const void* x, const float* router_w,
                         const float* probs, const int32_t* chosen, const float* gate, const float* dgate,
                         const float* dmean_probability, void* dx, float* dw_router, int tokens, int width,
                         int experts, int top_k, void* stream) {
  if (!dgrouped || !position) return GPTRIG_E_NULL;
  if (width % 8 || (((uintptr_t)dgrouped | (uintptr_t)x | (uintptr_t)dx) & 15)) return GPTRIG_E_SHAPE;
  if (top_k > kMaxTopK) return GPTRIG_E_UNSUPPORTED;
  return router_bwd(x, router_w, probs, chosen, gate, dgate, dmean_probability, dgrouped, position, dx, dw_router,
                    tokens, width, experts, top_k, stream);
}

}  // extern "C"

// ---------------------------------------------------------------------------
// The whole routed MLP behind one call per direction: the launches above in
// order, over two buffers of the caller's (what the backward needs, and
// scratch), so a caller's program pays for one call and a few allocations
// instead of a dozen each (200 tokens x 512, 8 experts of 1024, forward +
// backward from Python: 402 -> 262 us with the weight casts in one launch).
// ---------------------------------------------------------------------------
namespace {

struct RoutedLayout {
  // byte offsets; saved: from the forward for the backward
  size_t probs, chosen, gate, counts, position, grouped, pre, hidden, out, saved;
  size_t logits, order, rows, route, fwd_scratch;
  size_t dout, dgate, dpre, dgrouped, bwd_scratch;
};

RoutedLayout routed_layout(int tokens, int width, int hidden, int experts, int top_k) {
  RoutedLayout l;
  const size_t T = (size_t)tokens, R = T * top_k;
  auto take = [](size_t& at, size_t bytes) {
    const size_t here = at;
    at += (bytes + 255) & ~(size_t)255;
    return here;
  };
  size_t at = 0;
  l.probs = take(at, T * experts * 4);
  l.chosen = take(at, R * 4);
  l.gate = take(at, R * 4);
  l.counts = take(at, (size_t)experts * 4);
  l.position = take(at, R * 4);
  l.grouped = take(at, R * width * 2);
  l.pre = take(at, R * hidden * 2);
  l.hidden = take(at, R * hidden * 2);
  l.out = take(at, R * width * 2);
  l.saved = at;
  at = 0;
  l.logits = take(at, T * experts * 4);
  l.order = take(at, R * 4);
  l.rows = take(at, R * 4);
  l.route = take(at, gptrig_moe_route_workspace_bytes(tokens, experts, top_k));
  l.fwd_scratch = at;
  at = 0;
  l.dout = take(at, R * width * 2);
  l.dgate = take(at, R * 4);
  l.dpre = take(at, R * hidden * 2);
  l.dgrouped = take(at, R * width * 2);
  l.bwd_scratch = at;
  return l;
}

bool routed_sizes_ok(int tokens, int width, int hidden, int experts, int top_k) {
  return tokens > 0 && width > 0 && hidden > 0 && experts > 0 && top_k > 0 && top_k <= experts &&
         (int64_t)tokens * top_k < (1ll << 31);
}

#define GPTRIG_TRY(call)                        \
  do {                                          \
    const int status_ = (call);                 \
    if (status_ != GPTRIG_OK) return status_;   \
  } while (0)

}  // namespace

extern "C" {

size_t gptrig_routed_saved_bytes(int tokens, int width, int hidden, int experts, int top_k) {
  return routed_sizes_ok(tokens, width, hidden, experts, top_k) ? routed_layout(tokens, width, hidden, experts, top_k).saved : 0;
}

size_t gptrig_routed_scratch_bytes(int tokens, int width, int hidden, int experts, int top_k, int backward) {
  if (!routed_sizes_ok(tokens, width, hidden, experts, top_k)) return 0;
  const RoutedLayout l = routed_layout(tokens, width, hidden, experts, top_k);
  return backward ? l.bwd_scratch : l.fwd_scratch;
}

int gptrig_routed_fwd(const void* x, const float* router_w, const void* up_w, const void* up_b, const void* down_w,
                      const void* down_b, void* combined, float* mean_probability, float* load, float* summary,
                      void* saved, size_t saved_bytes, void* scratch, size_t scratch_bytes, int tokens, int width,
                      int hidden, int experts, int top_k, void* stream) {
  if (!saved || !scratch) return GPTRIG_E_NULL;
  if (!routed_sizes_ok(tokens, width, hidden, experts, top_k)) return GPTRIG_E_SHAPE;
  const RoutedLayout l = routed_layout(tokens, width, hidden, experts, top_k);
  if (saved_bytes < l.saved || scratch_bytes < l.fwd_scratch) return GPTRIG_E_WORKSPACE;
  char *sv = (char*)saved, *sc = (char*)scratch;
  const int R = tokens * top_k;
  float *logits = (float*)(sc + l.logits), *probs = (float*)(sv + l.probs), *gate = (float*)(sv + l.gate);
  int32_t *chosen = (int32_t*)(sv + l.chosen), *counts = (int32_t*)(sv + l.counts),
          *position = (int32_t*)(sv + l.position), *rows = (int32_t*)(sc + l.rows);
  GPTRIG_TRY(gptrig_moe_router_logits(x, router_w, logits, tokens, width, experts, stream));
  GPTRIG_TRY(gptrig_moe_route(logits, probs, chosen, gate, counts, (int32_t*)(sc + l.order), rows, position,
                              sc + l.route, l.fwd_scratch - l.route, tokens, experts, top_k, stream));
  GPTRIG_TRY(gptrig_moe_gather_rows(x, rows, sv + l.grouped, R, width, stream));
  GPTRIG_TRY(gptrig_moe_gmm(sv + l.grouped, width, up_w, 0, counts, up_b, 1, sv + l.hidden, sv + l.pre, hidden, R,
                            width, hidden, experts, stream));
  GPTRIG_TRY(gptrig_moe_gmm(sv + l.hidden, hidden, down_w, 0, counts, down_b, 0, sv + l.out, nullptr, width, R, hidden,
                            width, experts, stream));
  GPTRIG_TRY(gptrig_moe_combine(sv + l.out, position, gate, combined, tokens, width, top_k, stream));
  return gptrig_moe_stats(logits, probs, gate, counts, tokens, experts, top_k, mean_probability, load, summary, stream);
}

int gptrig_routed_bwd(const void* dcombined, const float* dmean_probability, const void* x, const float* router_w,
                      const void* up_w, const void* down_w, void* saved, size_t saved_bytes, void* dx, float* d_router,
                      float* d_up_w, float* d_up_b, float* d_down_w, float* d_down_b, void* scratch,
                      size_t scratch_bytes, int tokens, int width, int hidden, int experts, int top_k, void* stream) {
  if (!saved || !scratch || !d_router) return GPTRIG_E_NULL;
  if (!routed_sizes_ok(tokens, width, hidden, experts, top_k)) return GPTRIG_E_SHAPE;
  const RoutedLayout l = routed_layout(tokens, width, hidden, experts, top_k);
  if (saved_bytes < l.saved || scratch_bytes < l.bwd_scratch) return GPTRIG_E_WORKSPACE;
  char *sv = (char*)saved, *sc = (char*)scratch;
  const int R = tokens * top_k;
  const float *probs = (const float*)(sv + l.probs), *gate = (const float*)(sv + l.gate);
  const int32_t *chosen = (const int32_t*)(sv + l.chosen), *counts = (const int32_t*)(sv + l.counts),
                *position = (const int32_t*)(sv + l.position);
  float* dgate = (float*)(sc + l.dgate);
  GPTRIG_TRY(gptrig_moe_combine_bwd(dcombined, sv + l.out, position, gate, sc + l.dout, dgate, tokens, width, top_k,
                                    stream));
  // d(pre) = (dout W_down^T) * gelu'(pre); then the weight gradients of both
  // projections and d(grouped) = dpre W_up^T.
  GPTRIG_TRY(gptrig_moe_gmm(sc + l.dout, width, down_w, 1, counts, nullptr, 2, sc + l.dpre, sv + l.pre, hidden, R, width,
                            hidden, experts, stream));
  GPTRIG_TRY(moe_bwd_gemms(sv + l.grouped, sc + l.dpre, sv + l.hidden, sc + l.dout, up_w, counts, d_up_w, d_up_b,
                           d_down_w, d_down_b, sc + l.dgrouped, R, width, hidden, experts, d_router, stream));
  return gptrig_moe_input_bwd(sc + l.dgrouped, position, x, router_w, probs, chosen, gate, dgate, dmean_probability, dx,
                              d_router, tokens, width, experts, top_k, stream);
}

}  // extern "C"
