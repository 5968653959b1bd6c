// Fused linear cross-entropy with float32 compute (compute_dtype=float32 of
// rig/kernels/linear_cross_entropy.py:38-41): the same algorithm as the bf16
// kernels of flce.hip -- tiled logits with a per-tile (max, sum exp) in the
// forward, the logits recomputed one vocabulary chunk at a time in the
// backward -- with float32 operands, products and sums, as the reference's
// einsums with compute_dtype float32 (`_tile_logits`, :92-112; the backward,
// :220-302).  The [n, vocab] logits never exist; the backward's working set is
// one float32 [n, chunk] logit gradient, the reference's own [n,
// vocab_tile_size] bound, plus, from the default tile up, partial sums of at
// most the same size each for the two gradient products (below).
//
// Float32 products on the bf16 matrix cores: every float32 operand element is
// split exactly into three bf16 pieces (x = hi + mid + lo, 8 significant bits
// each, by truncation), and a product keeps the six terms of weight 2^-16 and
// above (lo*hi, hi*lo, mid*mid, mid*hi, hi*mid, hi*hi).  What is dropped is
// below 2^-21 of a product (mid*lo + lo*mid, each below 2^-7 2^-15).  hi*hi has
// an accumulator of its own and the five smaller terms, smallest first, another,
// added at the end: with one for all, six roundings of the whole sum per 16
// products cost up to twice the error over products of one sign.
// Short sums take more: up to 64 products also the two dropped terms, up to 16
// plain float32 multiply-adds (there a dropped term, or one rounding more, shows
// against the few roundings of a chain).
// Error against 64 bits, relative to one float32 multiply-add chain per output
// on the vector ALU, operands of random signs, 1..200 tokens, d 1..512, V 1000:
// dW 0.35 to 1.0, dh 0.2 to 0.4; of one sign: dW 0.35 to 1.1, dh 0.5 to 0.9 (the
// six terms alone: dW up to 2.2 at one token).
// A bf16 MFMA has 16 times the float32 MFMA's rate, so six of them are 2.7
// times cheaper than one float32 MFMA and 5 times cheaper than the vector
// ALU's multiply-adds.
//
// Tile kernel: 128 x 128 outputs per 256-thread workgroup, four waves of 64 x
// 64 (2 x 2 blocks of v_mfma_f32_32x32x16_bf16), k in stages of 16.  A stage's
// float32 elements go global -> registers one stage ahead, are split there and
// written as three bf16 planes per operand into a double-buffered LDS stage
// (24 KB): splitting on the way costs 5.5 vector operations per element, far
// below the 24 MFMAs per wave and stage, and needs neither a pre-pass over the
// weight nor a buffer for its planes.  The two accumulators leave registers for
// two workgroups per CU, so one's loads, splits and epilogue run under another's
// MFMAs (one accumulator and three workgroups: 2% faster).
// Measured at 2048 tokens, d 512, V 50304, against 64 x 64 vector-ALU tiles:
// logits 606 us (174 TFLOP/s, 1.04 PFLOP/s of MFMA) against 1430, forward +
// backward 2.57 ms in the 6288-row chunks the front end takes, against 23.0.  What bounds it now: a chunk of 2048 rows (37 us logit gradient,
// 55 us the two products) holds one or two workgroups per CU at this size, so a
// stage's serial parts (fragment reads, 24 MFMAs, split, barrier) overlap only
// partly; larger ones run at the logits' rate.
#include "gemm_core.h"

#include <math.h>

namespace {

constexpr int kT = 128;      // tile edge
constexpr int kK = 16;       // k per LDS stage
constexpr int kThreads = 256;
constexpr int kPlane = kT * kK;          // bf16 elements of one plane of one operand
constexpr int kStage = 6 * kPlane;       // A's three planes, then B's
constexpr int kFewTerms = kK;            // sums of so many products run as multiply-adds
constexpr int kFewStages = 4;            // sums of so many stages take eight terms of a product
constexpr int kChunkRows = 64;           // granularity of the vocabulary chunk
constexpr int kDefaultChunk = 2048;      // the reference's default vocab_tile_size

using gemm::lds_t;
using gemm::lds_x8;

__shared__ __attribute__((aligned(1024))) bf16 s32_stage0[kStage];
__shared__ __attribute__((aligned(1024))) bf16 s32_stage1[kStage];

// Operand X(mn, k): element (mn, k) at p[mn * ld + k] (K-major) or
// p[k * ld + mn] (MN-major); extents: mn < mn_end, k < k_end.
struct Mat {
  const float* p;
  int64_t ld;
};

// Where the 16-byte half `c` (8 values) of an operand plane's row sits.
// K-major plane: 128 rows (mn) of 16 k, 32 bytes each; the half is swapped in
// every other group of 8 rows, so the 16 rows a quarter-wave reads at one half
// cover all 64 banks.
__device__ __forceinline__ int kpos(int row, int c) { return row * 16 + 8 * (c ^ ((row >> 3) & 1)); }
// MN-major plane: 8 blocks of 16 k-rows x 16 mn, 32 bytes per k-row.  Row k of
// block b sits at k ^ f(b), f(b) = (b & 1) << 2 | (b >> 1): the 8 blocks one
// k-row spans (a write) then cover all banks, and so do the two neighbouring
// blocks of a transposed read.
__device__ __forceinline__ int mpos(int b, int k) { return b * 256 + (k ^ (((b & 1) << 2) | ((b >> 1) & 3))) * 16; }

// One thread's 8 consecutive elements of a stage: K-major, row tid / 2 and k
// 8 (tid % 2) ..; MN-major, k-row tid / 16 and mn 8 (tid % 16) ... kVec: 16-byte
// loads (base, ld and the contiguous extent multiples of 4 elements).
template <bool KMAJOR, bool kVec>
struct Loader {
  const float* p;    // this thread's first element at the tile's first stage
  const float* safe; // a readable address for masked-out loads
  int64_t step;      // elements per stage
  int inner;         // contiguous elements left from this thread's first one (K-major: shrinks by stage)
  int outer;         // K-major: row inside the extent (> 0); MN-major: k-rows left
  f32x4 lo, hi;

  __device__ __forceinline__ void init(Mat m, int mn0, int k0, int mn_end, int k_end, int tid) {
    safe = m.p;
    if (KMAJOR) {
      const int row = mn0 + (tid >> 1), k = k0 + 8 * (tid & 1);
      p = m.p + (int64_t)row * m.ld + k;
      inner = k_end - k;
      outer = mn_end - row;
      step = kK;
    } else {
      const int k = k0 + (tid >> 4), mn = mn0 + 8 * (tid & 15);
      p = m.p + (int64_t)k * m.ld + mn;
      inner = mn_end - mn;
      outer = k_end - k;
      step = (int64_t)kK * m.ld;
    }
  }
  // Elements past an extent come from `safe` and are replaced by zeros when split.
  __device__ __forceinline__ void load(int kt) {
    const float* q = p + kt * step;
    const int in = KMAJOR ? inner - kK * kt : inner;
    const bool ok = KMAJOR ? outer > 0 : outer > kK * kt;
    if constexpr (kVec) {
      lo = *reinterpret_cast<const f32x4*>(ok && in > 0 ? q : safe);
      hi = *reinterpret_cast<const f32x4*>(ok && in > 4 ? q + 4 : safe);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        lo[j] = *(ok && in > j ? q + j : safe);
        hi[j] = *(ok && in > 4 + j ? q + 4 + j : safe);
      }
    }
  }
  // Split the loaded stage kt and write its planes (plane q at dst + q * kPlane).
  __device__ __forceinline__ void store(lds_t* dst, int kt, int tid) const {
    const int in = KMAJOR ? inner - kK * kt : inner;
    const bool ok = KMAJOR ? outer > 0 : outer > kK * kt;
    uint32_t w[3][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint32_t piece[3][2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int i = 2 * j + u;
        const float raw = i < 4 ? lo[i] : hi[i - 4];
        const float x = ok && in > (kVec ? i & 4 : i) ? raw : 0.f;
        const uint32_t b0 = __builtin_bit_cast(uint32_t, x);
        const float r1 = x - __builtin_bit_cast(float, b0 & 0xFFFF0000u);   // exact
        const uint32_t b1 = __builtin_bit_cast(uint32_t, r1);
        const float r2 = r1 - __builtin_bit_cast(float, b1 & 0xFFFF0000u);  // exact, 8 bits
        piece[0][u] = b0;
        piece[1][u] = b1;
        piece[2][u] = __builtin_bit_cast(uint32_t, r2);
      }
#pragma unroll
      for (int q = 0; q < 3; ++q)  // the upper halves of the two words
        w[q][j] = __builtin_amdgcn_perm(piece[q][1], piece[q][0], 0x07060302u);
    }
    const int pos = KMAJOR ? kpos(tid >> 1, tid & 1) : mpos((tid & 15) >> 1, tid >> 4) + 8 * (tid & 1);
#pragma unroll
    for (int q = 0; q < 3; ++q)
      *(lds_x8*)(dst + q * kPlane + pos) = __builtin_bit_cast(bf16x8, u32x4{w[q][0], w[q][1], w[q][2], w[q][3]});
  }
};

// MFMA operand (8 k of this lane's half) of rows / columns r0 + lane % 32 of a plane.
template <bool KMAJOR>
__device__ __forceinline__ bf16x8 frag32(const lds_t* plane, int r0, int lane) {
  if (KMAJOR) return *(const lds_x8*)(plane + kpos(r0 + (lane & 31), lane >> 5));
  // Transposed read: lane 4j + q of a 16-lane group supplies row k0 + j,
  // columns 4q .. +3 of its block and receives rows k0 .. k0 + 3 of one column.
  const int c = lane & 15, b = (r0 >> 4) + ((lane >> 4) & 1), k = 8 * (lane >> 5) + (c >> 2);
  const bf16x4 lo = gemm::read_tr(plane + mpos(b, k) + 4 * (c & 3));
  const bf16x4 hi = gemm::read_tr(plane + mpos(b, k + 4) + 4 * (c & 3));
  return bf16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
}

// One stage: hi*hi into acc, the smaller terms into small.  all (uniform): also
// the two terms of weight 2^-21 and below (lo*mid, mid*lo).
template <bool AK, bool BKM>
__device__ __forceinline__ void mma_stage32(f32x16 (&acc)[2][2], f32x16 (&small)[2][2], const lds_t* st, int wm0,
                                            int wn0, int lane, bool all) {
  bf16x8 a[2][3], b[2][3];
#pragma unroll
  for (int q = 0; q < 3; ++q)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      a[i][q] = frag32<AK>(st + q * kPlane, wm0 + 32 * i, lane);
      b[i][q] = frag32<BKM>(st + (3 + q) * kPlane, wn0 + 32 * i, lane);
    }
  // Smallest terms first; the accumulators alternate, so no MFMA waits for the
  // one before it.
  constexpr int kTerm[8][2] = {{2, 1}, {1, 2}, {2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}, {0, 0}};
  auto term = [&](int t) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        f32x16& c = t == 7 ? acc[i][j] : small[i][j];
        c = mfma32(a[i][kTerm[t][0]], b[j][kTerm[t][1]], c);
      }
  };
  if (all) {
    term(0);
    term(1);
  }
#pragma unroll
  for (int t = 2; t < 8; ++t) term(t);
}

// tile32's product as plain float32 multiply-adds, one chain per output: all of
// it (`all`, the shortest sums), or the elements that came out infinite or NaN,
// while the others keep their bits (an infinite operand has no finite remainders
// to split off, inf - inf, and the pieces of an overflowing product may differ
// in sign).  Both operands' stages are staged as [k][row] floats, rows padded to
// 132; one column block at a time, for the registers.
template <bool AK, bool BKM>
__device__ __forceinline__ void tile32_plain(f32x16 (&acc)[2][2], Mat A, Mat B, int m_end, int n_end, int k0,
                                             int k_end, int m0, int n0, bool all) {
  typedef __attribute__((address_space(3))) float lds_f;
  typedef __attribute__((address_space(3))) f32x4 lds_f4;
  constexpr int kRow = kT + 4;
  static_assert(kK * kRow * sizeof(float) <= kStage * sizeof(bf16), "one operand per stage array");
  lds_f* const as = (lds_f*)gemm::lds_cast(s32_stage0);
  lds_f* const bs = (lds_f*)gemm::lds_cast(s32_stage1);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm0 = 64 * (wave & 1), wn0 = 64 * (wave >> 1);
  auto fill = [&](lds_f* dst, Mat m, bool kmajor, int mn0, int mn_end, int kb) {
    for (int idx = tid; idx < kT * kK; idx += kThreads) {
      const int r = kmajor ? idx / kK : idx % kT, kk = kmajor ? idx % kK : idx / kT;
      const int mn = mn0 + r, k = kb + kk;
      dst[kk * kRow + r] = mn < mn_end && k < k_end ? m.p[kmajor ? mn * m.ld + k : k * m.ld + mn] : 0.f;
    }
  };
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    f32x16 sum[2] = {};
    for (int kb = k0; kb < k_end; kb += kK) {
      if (j == 0 || k_end - k0 > kK) {  // (one stage stays for the second column block)
        __syncthreads();
        fill(as, A, AK, m0, m_end, kb);
        fill(bs, B, BKM, n0, n_end, kb);
        __syncthreads();
      }
      for (int kk = 0; kk < min(kK, k_end - kb); ++kk) {
        const float b = bs[kk * kRow + wn0 + 32 * j + (lane & 31)];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const f32x4 a = *(const lds_f4*)(as + kk * kRow + wm0 + 32 * i + 8 * q + 4 * (lane >> 5));
#pragma unroll
            for (int u = 0; u < 4; ++u) sum[i][4 * q + u] = fmaf(a[u], b, sum[i][4 * q + u]);
          }
      }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        acc[i][j][r] = !all && fabsf(acc[i][j][r]) < INFINITY ? acc[i][j][r] : sum[i][r];
  }
  __syncthreads();
}

// acc[i][j][r] = C[m0 + wm0 + 32 i + 8 (r / 4) + 4 (lane / 32) + r % 4][n0 + wn0 + 32 j + lane % 32],
// wm0 = 64 (wave % 2), wn0 = 64 (wave / 2), over k in [k0, k_end).  Ends on a barrier:
// the stage arrays may be reused.
// kShort: the sum may be short enough for more terms or plain multiply-adds
// (a template parameter: the test of every stage costs a long sum 1.6%).
template <bool AK, bool BKM, bool kVec, bool kShort>
__device__ __forceinline__ void tile32(f32x16 (&acc)[2][2], Mat A, Mat B, int m_end, int n_end, int k0, int k_end,
                                       int m0, int n0) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm0 = 64 * (wave & 1), wn0 = 64 * (wave >> 1);
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x16{};
  f32x16 small[2][2] = {};
  const bool few = kShort && k_end - k0 <= kFewTerms;  // uniform
  __shared__ int plain_s;
  if (!few) {
    lds_t* const st0 = gemm::lds_cast(s32_stage0);
    lds_t* const st1 = gemm::lds_cast(s32_stage1);
    if (tid == 0) plain_s = 0;
    Loader<AK, kVec> la;
    Loader<BKM, kVec> lb;
    la.init(A, m0, k0, m_end, k_end, tid);
    lb.init(B, n0, k0, n_end, k_end, tid);
    const int nk = (k_end - k0 + kK - 1) / kK;
    la.load(0);
    lb.load(0);
    la.store(st0, 0, tid);
    lb.store(st0 + 3 * kPlane, 0, tid);
    la.load(1);
    lb.load(1);
    __syncthreads();
    // Stage kt + 1 (already in registers) is written into the other buffer, whose
    // readers passed the last barrier, while stage kt is multiplied.
    auto step = [&](const lds_t* cur, lds_t* nxt, int kt) __attribute__((always_inline)) {
      mma_stage32<AK, BKM>(acc, small, cur, wm0, wn0, lane, kShort && nk <= kFewStages);
      la.store(nxt, kt + 1, tid);
      lb.store(nxt + 3 * kPlane, kt + 1, tid);
      la.load(kt + 2);
      lb.load(kt + 2);
      GPTRIG_WAIT_LGKM0();  // this wave's LDS writes (the global loads stay in flight)
      wg_barrier();
    };
    for (int kt = 0; kt < nk; kt += 2) {
      step(st0, st1, kt);
      if (kt + 1 < nk) step(st1, st0, kt + 1);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] += small[i][j];
    // A sum of zeros unless an element is an infinity or NaN.
    float zero[4] = {};
#pragma unroll
    for (int r = 0; r < 16; ++r)
#pragma unroll
      for (int q = 0; q < 4; ++q) zero[q] = fmaf(acc[q >> 1][q & 1][r], 0.f, zero[q]);
    const float z = (zero[0] + zero[1]) + (zero[2] + zero[3]);
    if (__any(z != z) && lane == 0) plain_s = 1;
    __syncthreads();
  }
  if (few || plain_s) tile32_plain<AK, BKM>(acc, A, B, m_end, n_end, k0, k_end, m0, n0, few);  // uniform
}

// Bytes of the rows of a tile that exist (at most kT of `ld` floats), and a
// lane offset past any of them even with a row's offset added: such accesses
// read zeros or are dropped.  That takes a resource of at most 2^31 bytes: rows
// of at most kMaxRow32 floats, which the host's token blocks (block32) and its
// check of d see to.
constexpr uint32_t kOff32Drop = 0x80000000u;
constexpr int kMaxRow32 = 1 << 22;
static_assert((int64_t)kT * kMaxRow32 * 4 <= (int64_t)kOff32Drop, "");
__device__ __forceinline__ uint32_t row_bytes32(int rows, int ld) {
  return 4u * (uint32_t)((rows < kT ? rows : kT) * ld);
}

// Workgroup -> (row tile, column tile) with the column tile fastest inside one
// XCD's contiguous share, so the workgroups that run together on an XCD share
// rows of A.
__device__ __forceinline__ void tile_of(int pid, int total, int col_tiles, int& tr, int& tc) {
  const int id = gemm::xcd_swizzle(pid, total);
  tr = id / col_tiles;
  tc = id % col_tiles;
}

// Logits of 128 vocabulary rows x 128 tokens (rows = vocabulary) and their
// per-token (max, sum exp(logit - max)) over the tile's classes.
template <bool kVec, bool kShort>
__global__ void __launch_bounds__(kThreads, 2)
    stats32_kernel(const float* __restrict__ w, const float* __restrict__ h, int V, int N, int D, int sem_v,
                   float2* __restrict__ partial) {
  __shared__ float2 half_s[kT];
  const int tok_tiles = (N + kT - 1) / kT;
  int tv, tn;
  tile_of(blockIdx.x, gridDim.x, tok_tiles, tv, tn);
  f32x16 acc[2][2];
  tile32<true, true, kVec, kShort>(acc, Mat{w, D}, Mat{h, D}, V, N, 0, D, tv * kT, tn * kT);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, hl = lane >> 5;
  const int wm0 = 64 * (wave & 1), wn0 = 64 * (wave >> 1);
  const int left = sem_v - (tv * kT + wm0 + 4 * hl);  // classes from this lane's first row on
  float mx[2], sum[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    mx[j] = -INFINITY;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) mx[j] = fmaxf(mx[j], 32 * i + 8 * (r >> 2) + (r & 3) < left ? acc[i][j][r] : -INFINITY);
    mx[j] = fmaxf(mx[j], __shfl_xor(mx[j], 32));
    sum[j] = 0.f;
    // (max ignores NaN logits; the sum must not, also when nothing else is there.)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float x = acc[i][j][r];
        if (32 * i + 8 * (r >> 2) + (r & 3) < left) sum[j] += mx[j] == -INFINITY && x == x ? 0.f : expf(x - mx[j]);
      }
    sum[j] += __shfl_xor(sum[j], 32);
  }
  // The two 64-row halves of a token, merged through LDS.
  if ((wave & 1) && hl == 0) {
#pragma unroll
    for (int j = 0; j < 2; ++j) half_s[wn0 + 32 * j + lane] = make_float2(mx[j], sum[j]);
  }
  __syncthreads();
  if (!(wave & 1) && hl == 0) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int n = tn * kT + wn0 + 32 * j + lane;
      const float2 o = half_s[wn0 + 32 * j + lane];
      const float m = fmaxf(mx[j], o.x);
      // (A half without classes, or with -inf logits only, adds its sum as it is: 0, or NaN.)
      const float s = (mx[j] == -INFINITY ? sum[j] : sum[j] * expf(mx[j] - m)) +
                      (o.x == -INFINITY ? o.y : o.y * expf(o.x - m));
      if (n < N) partial[(size_t)tv * N + n] = make_float2(m, s);
    }
  }
}

// G^T of one vocabulary chunk: gt[v][n] = (exp(logit - lse) - [v == target]) ct,
// zero for rows that are no classes (linear_cross_entropy.py:255-266) and for
// the padding columns N .. ld - 1.
template <bool kVec, bool kShort>
__global__ void __launch_bounds__(kThreads, 2)
    grad32_kernel(const float* __restrict__ w, const float* __restrict__ h, int C, int N, int D, int v0, int sem_v,
                  const int32_t* __restrict__ targets, const float* __restrict__ lse, const float* __restrict__ cot,
                  float cot_scale, float* __restrict__ gt, int ld) {
  const int tok_tiles = (N + kT - 1) / kT;
  int tv, tn;
  tile_of(blockIdx.x, gridDim.x, tok_tiles, tv, tn);
  f32x16 acc[2][2];
  tile32<true, true, kVec, kShort>(acc, Mat{w, D}, Mat{h, D}, C, N, 0, D, tv * kT, tn * kT);
  // Branch-free, through a buffer resource over the tile's rows: stores past
  // the chunk or the row are dropped.  (With a branch per element the 64
  // elements of a lane ran one after the other: 44 against 37 us per chunk of
  // 2048 rows x 2048 tokens, and 71 against 55 us for the two products below.)
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, hl = lane >> 5;
  const int wm0 = 64 * (wave & 1), wn0 = 64 * (wave >> 1);
  const __amdgpu_buffer_rsrc_t rs = make_rsrc(gt + (int64_t)tv * kT * ld, row_bytes32(C - tv * kT, ld));
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int n = tn * kT + wn0 + 32 * j + (lane & 31);
    const bool in = n < N;
    const int t = in ? targets[n] : -1;
    const float ct = t >= 0 && t < sem_v ? (cot ? cot[n] : cot_scale) : 0.f;
    const float l = in ? lse[n] : 0.f;
    const int row0 = wm0 + 4 * hl;             // this lane's first row of the tile
    const int left = sem_v - v0 - tv * kT - row0;  // classes from there on
    const int hit = t - v0 - tv * kT - row0;       // the target's row from there
    const uint32_t off = n < ld ? 4u * (uint32_t)(row0 * ld + n) : kOff32Drop;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int dr = 32 * i + 8 * (r >> 2) + (r & 3);
        const float g = (expf(acc[i][j][r] - l) - (dr == hit ? 1.f : 0.f)) * ct;
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, in && dr < left ? g : 0.f), rs,
                                              off + 4u * (uint32_t)(dr * ld), 0, 0);
      }
  }
}

// The two gradient products of one chunk in one launch: workgroups [0, n_dw)
// compute dW[chunk] = G^T h (k = tokens), the others dh = G W[chunk] (k = the
// chunk's rows).  Neither product has enough 128 x 128 tiles for 256 CUs at a
// few thousand tokens, so each k range is cut into slices and every slice
// writes a plain partial sum of its own: no atomics, so the results do not
// depend on the order of the workgroups.  dh's slices accumulate over the
// chunks in place; sum32_kernel adds the slices.
struct Out32 {
  float* p;        // [slices][rows][D]
  int slices;
  int64_t stride;  // elements between slices
  bool add;        // += (the slice holds earlier sums) instead of =
};

template <bool kVec, bool kShort>
__global__ void __launch_bounds__(kThreads, 2)
    grads32_kernel(const float* __restrict__ gt, int ld, const float* __restrict__ w, const float* __restrict__ h, int C,
                   int N, int D, Out32 dw, Out32 dh, int n_dw) {
  const int col_tiles = (D + kT - 1) / kT;
  f32x16 acc[2][2];
  const bool is_dw = (int)blockIdx.x < n_dw;  // uniform
  const Out32 o = is_dw ? dw : dh;
  const int pid = is_dw ? blockIdx.x : blockIdx.x - n_dw;
  const int rows = is_dw ? C : N, depth = is_dw ? N : C;
  const int tiles = ((rows + kT - 1) / kT) * col_tiles;
  const int slice = pid / tiles, id = pid % tiles;
  const int tr = id / col_tiles, tc = id % col_tiles;
  const int per = ((depth + o.slices - 1) / o.slices + kK - 1) / kK * kK;
  const int k0 = slice * per, k1 = min(depth, k0 + per);  // (an empty slice writes zeros)
  if (is_dw)
    tile32<true, false, kVec, kShort>(acc, Mat{gt, ld}, Mat{h, D}, C, D, k0, k1, tr * kT, tc * kT);
  else
    tile32<false, false, kVec, kShort>(acc, Mat{gt, ld}, Mat{w, D}, ld, D, k0, k1, tr * kT, tc * kT);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, hl = lane >> 5;
  const int wm0 = 64 * (wave & 1), wn0 = 64 * (wave >> 1);
  const __amdgpu_buffer_rsrc_t rs =
      make_rsrc(o.p + slice * o.stride + (int64_t)tr * kT * D, row_bytes32(rows - tr * kT, D));
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int c = tc * kT + wn0 + 32 * j + (lane & 31);
    const uint32_t off = c < D ? 4u * (uint32_t)((wm0 + 4 * hl) * D + c) : kOff32Drop;
    // All loads of earlier sums first, then the stores.
    if (o.add) {  // uniform
      float old[2][16];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          old[i][r] = __builtin_bit_cast(
              float, __builtin_amdgcn_raw_buffer_load_b32(rs, off + 4u * (uint32_t)((32 * i + 8 * (r >> 2) + (r & 3)) * D), 0, 0));
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] += old[i][r];
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float x = acc[i][j][r];  // (a bit cast straight from a vector element reads element 0 of its quad)
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, x), rs,
                                              off + 4u * (uint32_t)((32 * i + 8 * (r >> 2) + (r & 3)) * D), 0, 0);
      }
  }
}

// out (+)= the sum of `slices` arrays of n elements.
__global__ void __launch_bounds__(256) sum32_kernel(const float* __restrict__ parts, int slices, int64_t n,
                                                    float* __restrict__ out, int add) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float s = parts[i];
  for (int k = 1; k < slices; ++k) s += parts[k * n + i];
  out[i] = add ? out[i] + s : s;
}

// Target logit h[n] . W[t[n]] in float32 (0 for an invalid target): one wave per token.
__global__ void __launch_bounds__(256) target32_kernel(const float* __restrict__ h, const float* __restrict__ w,
                                                       const int32_t* __restrict__ targets, int N, int D, int sem_v,
                                                       float* __restrict__ tlogit) {
  const int n = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (n >= N) return;
  const int t = targets[n];
  float acc = 0.f;
  if (t >= 0 && t < sem_v)
    for (int c = lane; c < D; c += 64) acc = fmaf(h[(size_t)n * D + c], w[(size_t)t * D + c], acc);
  acc = wave_sum(acc);
  if (lane == 0) tlogit[n] = acc;
}

// lse = max + log(sum) over the vocabulary tiles' partials; loss = lse - target
// logit, +inf for an invalid target.  64 tokens per workgroup, each of its 16
// waves folding every 16th tile: one thread per token ran 365 us at 2048
// tokens and V 50304 (8 workgroups, one dependent pass after the other), this
// form 13 us.
constexpr int kCombineWaves = 16;
__global__ void __launch_bounds__(64 * kCombineWaves)
    combine32_kernel(const float2* __restrict__ partial, int ntiles, int N, int sem_v,
                     const int32_t* __restrict__ targets, const float* __restrict__ tlogit, float* __restrict__ lse,
                     float* __restrict__ losses) {
  __shared__ float m_s[kCombineWaves][64], s_s[kCombineWaves][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n = blockIdx.x * 64 + lane;
  float m = -INFINITY, s = 0.f;
  if (n < N) {
    for (int t = wave; t < ntiles; t += kCombineWaves) m = fmaxf(m, partial[(size_t)t * N + n].x);
    for (int t = wave; t < ntiles; t += kCombineWaves) {
      const float2 p = partial[(size_t)t * N + n];
      s += p.x == -INFINITY ? p.y : p.y * expf(p.x - m);  // (p.y is 0, or NaN, without a maximum)
    }
  }
  m_s[wave][lane] = m;
  s_s[wave][lane] = s;
  __syncthreads();
  if (wave || n >= N) return;
  float mt = -INFINITY;
#pragma unroll
  for (int k = 0; k < kCombineWaves; ++k) mt = fmaxf(mt, m_s[k][lane]);
  float st = 0.f;
#pragma unroll
  for (int k = 0; k < kCombineWaves; ++k)
    st += m_s[k][lane] == -INFINITY ? s_s[k][lane] : s_s[k][lane] * expf(m_s[k][lane] - mt);
  const float l = mt + logf(st);
  lse[n] = l;
  const int t = targets[n];
  losses[n] = (t >= 0 && t < sem_v) ? l - tlogit[n] : INFINITY;
}

size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

int chunk32(int vocab, int vocab_chunk) {
  const int64_t c = vocab_chunk <= 0 ? kDefaultChunk : ((int64_t)vocab_chunk + kChunkRows - 1) / kChunkRows * kChunkRows;
  return (int)(c < vocab ? c : ((int64_t)vocab + kChunkRows - 1) / kChunkRows * kChunkRows);
}

// Columns of the G^T rows: n rounded up to whole 16-byte groups.
int64_t gt_ld(int n) { return ((int64_t)n + 3) & ~(int64_t)3; }

int64_t tiles32(int64_t rows, int64_t cols) { return ((rows + kT - 1) / kT) * ((cols + kT - 1) / kT); }

// Tokens a launch takes: at most kMaxRow32 (the rows of G^T stay addressable by
// 32-bit byte offsets) and fewer than 2^24 tiles with `rows` vocabulary rows (a
// grid has fewer than 2^32 threads).  Both directions walk the tokens in such
// blocks; up to 4 million tokens are one block for 65,000 rows.
int block32(int n, int64_t rows) {
  const int64_t most = ((1ll << 24) - 1) / tiles32(rows, 1) * kT;
  const int64_t b = most < kT ? kT : most < kMaxRow32 ? most : kMaxRow32;
  return (int)(b < n ? b : n);
}

// Slices of a gradient product of rows x d outputs over `depth`: enough
// workgroups for one per CU (256 are assumed; a fixed number keeps the
// workspace query independent of the device), slices at least 8 stages deep,
// and all partial sums together no larger than `budget` values: the [n, chunk]
// gradient, or none for a chunk below the default, which asks for a small working
// set (the backward at 2048 tokens, d 512, V 50304 in chunks of 1024: 3.3 ms with
// partial sums, 6.0 without, 32.5 on the vector ALU in the same bytes).
int slices32(int64_t rows, int d, int depth, int64_t budget) {
  const int64_t tiles = tiles32(rows, d);
  int64_t s = (256 + tiles / 2) / tiles;
  const int64_t deep = depth / (8 * kK), fit = budget / (rows * d);
  if (s > deep) s = deep;
  if (s > fit) s = fit;
  return s < 1 ? 1 : (int)s;
}

struct Plan32 {
  int block, chunk, dh_slices, dw_slices;
  int64_t ld;
  size_t gt_bytes, dh_bytes, dw_bytes;  // workspace: G^T, dh partials, dW partials (0: written in place)
};

Plan32 plan32(int n, int d, int vocab, int vocab_chunk) {
  Plan32 p;
  p.chunk = chunk32(vocab, vocab_chunk);
  p.block = n = block32(n, p.chunk);
  p.ld = gt_ld(n);
  const int64_t gt = (int64_t)p.chunk * p.ld;
  const int64_t budget = vocab_chunk > 0 && vocab_chunk < kDefaultChunk ? 0 : gt;
  p.dh_slices = slices32(n, d, p.chunk, budget);
  p.dw_slices = slices32(p.chunk, d, n, budget);
  p.gt_bytes = align256((size_t)gt * sizeof(float));
  p.dh_bytes = p.dh_slices > 1 ? align256((size_t)p.dh_slices * n * d * sizeof(float)) : 0;
  p.dw_bytes = p.dw_slices > 1 ? align256((size_t)p.dw_slices * p.chunk * d * sizeof(float)) : 0;
  return p;
}

// A kernel's form for 16-byte loads or not, for short sums or not.
constexpr int kShort32 = kFewStages * kK;
template <class Kernel>
Kernel* pick32(bool vec, bool is_short, Kernel* v, Kernel* e, Kernel* v_short, Kernel* e_short) {
  return is_short ? (vec ? v_short : e_short) : (vec ? v : e);
}

// 16-byte loads of rows of d floats.
bool vec32(const float* a, const float* b, int d) {
  return d % 4 == 0 && (((uintptr_t)a | (uintptr_t)b) & 15) == 0;
}

}  // namespace

extern "C" {

size_t gptrig_flce32_fwd_workspace_bytes(int n, int d, int vocab) {
  (void)d;
  if (n <= 0 || vocab <= 0) return 0;
  n = block32(n, vocab);
  const size_t ntiles = (size_t)((vocab + kT - 1) / kT);
  return align256(ntiles * n * sizeof(float2)) + align256((size_t)n * sizeof(float));
}

int gptrig_flce32_fwd(const float* hidden, const float* weight, const int32_t* targets, float* losses, float* lse,
                      void* workspace, size_t workspace_bytes, int n, int d, int vocab, int semantic_vocab,
                      void* stream) {
  if (!hidden || !weight || !targets || !losses || !lse || !workspace) return GPTRIG_E_NULL;
  if (n <= 0 || d <= 0 || vocab <= 0) return GPTRIG_E_SHAPE;
  if (semantic_vocab <= 0 || semantic_vocab > vocab) return GPTRIG_E_SHAPE;
  if (workspace_bytes < gptrig_flce32_fwd_workspace_bytes(n, d, vocab)) return GPTRIG_E_WORKSPACE;
  if ((int64_t)n * d >= (1ll << 31) || (int64_t)vocab * d >= (1ll << 31)) return GPTRIG_E_SHAPE;
  hipStream_t s = (hipStream_t)stream;
  const int ntiles = (vocab + kT - 1) / kT, block = block32(n, vocab);
  float2* partial = (float2*)workspace;
  float* tlogit = (float*)((char*)workspace + align256((size_t)ntiles * block * sizeof(float2)));
  for (int64_t t0 = 0; t0 < n; t0 += block) {
    const int nb = (int)(n - t0 < block ? n - t0 : block);
    const float* hb = hidden + t0 * d;
    // logits[v][token] = sum_d W[v][d] h[token][d]
    const unsigned grid = (unsigned)tiles32(vocab, nb);
    pick32(vec32(hb, weight, d), d <= kShort32, stats32_kernel<true, false>, stats32_kernel<false, false>,
           stats32_kernel<true, true>, stats32_kernel<false, true>)<<<grid, kThreads, 0, s>>>(
        weight, hb, vocab, nb, d, semantic_vocab, partial);
    GPTRIG_CHECK_LAUNCH();
    target32_kernel<<<(unsigned)((nb + 3) / 4), 256, 0, s>>>(hb, weight, targets + t0, nb, d, semantic_vocab, tlogit);
    GPTRIG_CHECK_LAUNCH();
    combine32_kernel<<<(unsigned)((nb + 63) / 64), 64 * kCombineWaves, 0, s>>>(
        partial, ntiles, nb, semantic_vocab, targets + t0, tlogit, lse + t0, losses + t0);
    GPTRIG_CHECK_LAUNCH();
  }
  return GPTRIG_OK;
}

size_t gptrig_flce32_bwd_workspace_bytes(int n, int d, int vocab, int vocab_chunk) {
  if (n <= 0 || d <= 0 || vocab <= 0) return 0;
  const Plan32 p = plan32(n, d, vocab, vocab_chunk);
  return p.gt_bytes + p.dh_bytes + p.dw_bytes;
}

int gptrig_flce32_bwd(const float* hidden, const float* weight, const int32_t* targets, const float* lse,
                      const float* cotangent, float cotangent_scale, float* dhidden, float* dweight,
                      int accumulate_dweight, void* workspace, size_t workspace_bytes, int n, int d, int vocab,
                      int semantic_vocab, int vocab_chunk, void* stream) {
  if (!hidden || !weight || !targets || !lse || !dhidden || !dweight || !workspace) return GPTRIG_E_NULL;
  if (n <= 0 || d <= 0 || vocab <= 0 || vocab_chunk < 0) return GPTRIG_E_SHAPE;
  if (semantic_vocab <= 0 || semantic_vocab > vocab) return GPTRIG_E_SHAPE;
  if (workspace_bytes < gptrig_flce32_bwd_workspace_bytes(n, d, vocab, vocab_chunk)) return GPTRIG_E_WORKSPACE;
  if ((int64_t)n * d >= (1ll << 31) || (int64_t)vocab * d >= (1ll << 31)) return GPTRIG_E_SHAPE;
  if (d > kMaxRow32) return GPTRIG_E_SHAPE;
  hipStream_t s = (hipStream_t)stream;
  const Plan32 p = plan32(n, d, vocab, vocab_chunk);
  float* G = (float*)workspace;
  float* dh_parts = (float*)((char*)workspace + p.gt_bytes);
  float* dw_parts = (float*)((char*)workspace + p.gt_bytes + p.dh_bytes);
  for (int64_t t0 = 0; t0 < n; t0 += p.block) {
    const int nb = (int)(n - t0 < p.block ? n - t0 : p.block);
    const float* hb = hidden + t0 * d;
    float* dhb = dhidden + t0 * d;
    const float* cot = cotangent ? cotangent + t0 : nullptr;
    const int ld = (int)gt_ld(nb);
    const int64_t nd = (int64_t)nb * d;
    const bool add = accumulate_dweight || t0 > 0;
    const bool vec = vec32(hb, weight, d) && ((uintptr_t)workspace & 15) == 0;
    for (int v0 = 0; v0 < vocab; v0 += p.chunk) {
      const int c = vocab - v0 < p.chunk ? vocab - v0 : p.chunk;
      const float* Wc = weight + (int64_t)v0 * d;
      float* dWc = dweight + (int64_t)v0 * d;
      const int64_t cd = (int64_t)c * d;
      pick32(vec, d <= kShort32, grad32_kernel<true, false>, grad32_kernel<false, false>, grad32_kernel<true, true>,
             grad32_kernel<false, true>)<<<(unsigned)tiles32(c, nb), kThreads, 0, s>>>(
          Wc, hb, c, nb, d, v0, semantic_vocab, targets + t0, lse + t0, cot, cotangent_scale, G, ld);
      GPTRIG_CHECK_LAUNCH();
      // dW[chunk] (+)= G^T h (the dynamic_update_slice of :279-283) and
      // dh += G W[chunk] (the reference's grad_hidden carry, :247).
      const Out32 dw{p.dw_bytes ? dw_parts : dWc, p.dw_slices, cd, !p.dw_bytes && add};
      const Out32 dh{p.dh_bytes ? dh_parts : dhb, p.dh_slices, nd, v0 > 0};
      const int64_t n_dw = tiles32(c, d) * p.dw_slices, n_dh = tiles32(nb, d) * p.dh_slices;
      pick32(vec, nb <= kShort32 || c <= kShort32, grads32_kernel<true, false>, grads32_kernel<false, false>,
             grads32_kernel<true, true>, grads32_kernel<false, true>)<<<(unsigned)(n_dw + n_dh), kThreads, 0, s>>>(
          G, ld, Wc, hb, c, nb, d, dw, dh, (int)n_dw);
      GPTRIG_CHECK_LAUNCH();
      if (p.dw_bytes) {
        sum32_kernel<<<(unsigned)((cd + 255) / 256), 256, 0, s>>>(dw_parts, p.dw_slices, cd, dWc, add);
        GPTRIG_CHECK_LAUNCH();
      }
    }
    if (p.dh_bytes) {
      sum32_kernel<<<(unsigned)((nd + 255) / 256), 256, 0, s>>>(dh_parts, p.dh_slices, nd, dhb, 0);
      GPTRIG_CHECK_LAUNCH();
    }
  }
  return GPTRIG_OK;
}

}  // extern "C"
