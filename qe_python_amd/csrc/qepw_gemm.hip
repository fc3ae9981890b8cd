// Complex GEMM on CDNA4 matrix cores: C = alpha op(A) op(B) + beta C.
//
// Every complex product is four real MFMA products accumulated into separate
// real / imaginary accumulators (no 3M trick, which loses accuracy):
//   op N : re += Ar Br - Ai Bi ;  im += Ar Bi + Ai Br
//   op C : re += Ar Br + Ai Bi ;  im += Ar Bi - Ai Br
// (op(B) = B^H is conjugated as it is staged into LDS).
// using v_mfma_f64_16x16x4f64 (FP64) or v_mfma_f32_16x16x4f32 (FP32, FP32
// accumulation).  A 256-thread workgroup owns a TM x TN output tile (kVariants:
// eight shapes from 32 x 32 to 128 x 64); each of its four waves owns a part of
// 16x16 MFMA blocks and walks K in steps of 8 or 16 staged through LDS.  Products
// with few tiles (A^H B over K = npw above all) are split over K: every split
// writes its partial tile to the workspace and a second kernel sums the splits in
// fixed order, so results are bitwise reproducible run to run, and the plan depends
// on the shape alone (a workspace below the quoted one: gemm_t).
//
// MFMA 16x16x4 operand layout (lane l of a wave64): A element (row l%16,
// k l/16); B element (k l/16, col l%16).  Accumulator v of lane l holds
// column l%16 and row 4*(l/16)+v for the f32 instruction but row l/16+4v
// for the f64 one (measured on gfx950 with an in-bounds probe).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "qepw_internal.h"

namespace qepw {

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef double v2d __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));

template <typename T> struct Mfma;
template <> struct Mfma<double> {
  using acc = v4d;
  using pair = v2d;
  static __device__ __forceinline__ acc op(double a, double b, acc c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int v) { return (lane >> 4) + 4 * v; }
};
template <> struct Mfma<float> {
  using acc = v4f;
  using pair = v2f;
  static __device__ __forceinline__ acc op(float a, float b, acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int v) { return 4 * (lane >> 4) + v; }
};

constexpr int kGemmThreads = 256;
constexpr int kPad = 1;
// K depth of one LDS step: 16 columns, eight of the larger FP64 tiles (whose
// steps are long enough, and whose LDS would halve the workgroups of a CU).
template <typename T, int TM, int TN> constexpr int gemm_bk() {
  return sizeof(T) == 8 && TM * TN > 1024 ? 8 : 16;
}
// LDS buffers: two (one barrier a step), one for the smallest FP32 tile, which
// more workgroups of a CU serve better than fewer barriers.
template <typename T, int TM, int TN> constexpr int gemm_buffers() {
  return sizeof(T) == 4 && TM * TN <= 1024 ? 1 : 2;
}

// The tile of linear block id ``b`` of an (mt, nt, splits) grid.  Consecutive
// blocks go to different XCDs, each with an L2 of its own: the tiles that read
// the same operand rows -- all tiles of one K split, or, unsplit, the column
// tiles of one row tile -- are given ids a multiple of eight apart.
__device__ __forceinline__ void gemm_tile(unsigned b, unsigned mt, unsigned nt, unsigned splits,
                                          unsigned& tm, unsigned& tn, unsigned& ts) {
  const unsigned group = splits > 1 ? mt * nt : nt;     // tiles that share operands
  const unsigned groups = splits > 1 ? splits : mt;
  const unsigned whole = groups & ~7u;                  // groups dealt out to the XCDs
  unsigned gi, in;
  if (b < whole * group) {
    const unsigned x = b & 7u, j = b >> 3;
    gi = (j / group) * 8u + x;
    in = j % group;
  } else {
    const unsigned j = b - whole * group;
    gi = whole + j / group;
    in = j % group;
  }
  if (splits > 1) {
    ts = gi;
    tn = in / mt;
    tm = in - tn * mt;
  } else {
    ts = 0;
    tm = gi;
    tn = in;
  }
}

// TM x TN output tile per 256-thread workgroup; its four waves form a
// WAVES_M x (4 / WAVES_M) grid, each owning a (TM / WAVES_M) x (TN * WAVES_M / 4)
// block of 16x16 MFMA tiles.  Rectangular tiles let a tall-skinny product
// (npw x 128 outputs) cover all its columns in one workgroup, so the tall
// operand is streamed from HBM once.
//
// The K loop is double-buffered in LDS with one barrier a step: the next step's
// operands are fetched into registers before the MFMAs of the current one and
// stored to the other buffer after them.  Rows and columns past the edge are
// read from the last one (their outputs are not stored) and a short last step
// is fetched by a checked path, so that a full step costs one address addition
// a load: the FP64 MFMA rate (64 cycles each) leaves little time for more.
// The second launch bound keeps the accumulators out of the AGPRs, whose
// copies cost a fifth of the rate.  Measured, against a single buffer with
// every load checked: FP64 78 805 x 192 x 512 1114 -> 983 us (63 TFLOP/s, at
// the power limit), 512 x 192 x 78 805 (A^H B) 1136 -> 1010; FP32 695 -> 548
// (113 TFLOP/s) and 740 -> 560; FP64 23 847 x 13 x 256 35 -> 28.
template <typename T, int TM, int TN, int WAVES_M> struct GemmTile {
  static constexpr int BK = gemm_bk<T, TM, TN>();
  static constexpr int NBUF = gemm_buffers<T, TM, TN>();
  static constexpr int WAVES_N = 4 / WAVES_M;
  static constexpr int WTM = TM / WAVES_M;  // wave tile
  static constexpr int WTN = TN / WAVES_N;
  static constexpr int NBM = WTM / 16;      // MFMA blocks per wave and dimension
  static constexpr int NBN = WTN / 16;
  static_assert(NBM >= 1 && NBN >= 1 && WAVES_M * WAVES_N == 4, "tile shape");
  // whether A^H B sums chains of K apart: at the wave tiles whose registers allow it
  static constexpr bool chains = NBM * NBN <= (sizeof(T) == 8 ? 2 : 4);
};

// Columns of K that A^H B adds up in one chain, of a split's k, in a wave tile of
// ``blocks``.  An accumulator's error grows with the square root of its chain, and
// the cost model's splits are longer than those of the table that it replaced:
// single chains were up to 1.8 (FP32) and 1.4 times (FP64) as far from the exact
// product over the projections and subspaces of 2 .. 128 atoms (384 x 150 x 35 769
// in FP32 5.3e-7 with 86 splits, 9.6e-7 with 25, 3.0e-7 with chains; 0.57 times in
// the mean).  Chains cost 0-2% at the tiles chosen; chains of 32 throughout
// 2-4%, and with FP64 wave tiles of four blocks, whose registers then halve the
// waves, 20% (those keep one chain: their splits are as short as they were).
template <int BLOCKS> __device__ __forceinline__ int gemm_chain(int64_t k) {
  return k <= 64 ? 32 : k <= 256 ? 64 : BLOCKS >= 4 ? 256 : 128;
}

// re, im = the wave's part of op(A) op(B) over K in [kbeg, kend), at rows m0,
// columns n0 of the output
template <typename T, bool CONJ_A, bool CONJ_B, int TM, int TN, int WAVES_M, int NBM, int NBN>
__device__ __forceinline__ void gemm_accumulate(
    int64_t M, int64_t N, int64_t m0, int64_t n0, int64_t kbeg, int64_t kend,
    const cplx<T>* __restrict__ A, int64_t lda, const cplx<T>* __restrict__ B, int64_t ldb,
    typename Mfma<T>::acc (&re)[NBM][NBN], typename Mfma<T>::acc (&im)[NBM][NBN]) {
  using Pair = typename Mfma<T>::pair;
  using G = GemmTile<T, TM, TN, WAVES_M>;
  using Acc = typename Mfma<T>::acc;
  constexpr int BK = G::BK, NBUF = G::NBUF;
  __shared__ Pair As[NBUF][BK][TM + kPad];
  __shared__ Pair Bs[NBUF][BK][TN + kPad];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = (wave % WAVES_M) * G::WTM;
  const int wn = (wave / WAVES_M) * G::WTN;
#pragma unroll
  for (int i = 0; i < NBM; ++i)
#pragma unroll
    for (int j = 0; j < NBN; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) { re[i][j][v] = T(0); im[i][j][v] = T(0); }

  // element e of the BK x TM / BK x TN operand tiles: its k and its row / column
  constexpr int kPerA = BK * TM / kGemmThreads;  // elements per thread
  constexpr int kPerB = BK * TN / kGemmThreads;
  static_assert(kPerA >= 1 && kPerB >= 1, "tile too small for the workgroup");
  auto a_k = [](int e) { return CONJ_A ? (e & (BK - 1)) : (e / TM); };
  auto a_m = [](int e) { return CONJ_A ? (e / BK) : (e % TM); };
  auto b_k = [](int e) { return CONJ_B ? (e / TN) : (e & (BK - 1)); };
  auto b_n = [](int e) { return CONJ_B ? (e % TN) : (e / BK); };
  const Pair* const A2 = reinterpret_cast<const Pair*>(A);
  const Pair* const B2 = reinterpret_cast<const Pair*>(B);
  const Pair* pa[kPerA];
  const Pair* pb[kPerB];
#pragma unroll
  for (int p = 0; p < kPerA; ++p) {
    const int e = tid + p * kGemmThreads;
    const int64_t m = m0 + a_m(e) < M ? m0 + a_m(e) : M - 1;
    const int64_t k = kbeg + a_k(e);
    pa[p] = CONJ_A ? A2 + k + m * lda : A2 + m + k * lda;
  }
#pragma unroll
  for (int p = 0; p < kPerB; ++p) {
    const int e = tid + p * kGemmThreads;
    const int64_t n = n0 + b_n(e) < N ? n0 + b_n(e) : N - 1;
    const int64_t k = kbeg + b_k(e);
    pb[p] = CONJ_B ? B2 + n + k * ldb : B2 + k + n * ldb;
  }
  const int64_t step_a = CONJ_A ? BK : BK * lda;
  const int64_t step_b = CONJ_B ? BK * ldb : BK;
  Pair ra[kPerA], rb[kPerB];
  // fetches the step starting at k0 and moves the pointers to the next
  auto fetch = [&](int64_t k0) __attribute__((always_inline)) {
    if (k0 + BK <= kend) {
#pragma unroll
      for (int p = 0; p < kPerA; ++p) ra[p] = *pa[p];
#pragma unroll
      for (int p = 0; p < kPerB; ++p) rb[p] = *pb[p];
    } else {
#pragma unroll
      for (int p = 0; p < kPerA; ++p)
        ra[p] = k0 + a_k(tid + p * kGemmThreads) < kend ? *pa[p] : Pair{T(0), T(0)};
#pragma unroll
      for (int p = 0; p < kPerB; ++p)
        rb[p] = k0 + b_k(tid + p * kGemmThreads) < kend ? *pb[p] : Pair{T(0), T(0)};
    }
#pragma unroll
    for (int p = 0; p < kPerA; ++p) pa[p] += step_a;
#pragma unroll
    for (int p = 0; p < kPerB; ++p) pb[p] += step_b;
  };
  auto store = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < kPerA; ++p) {
      const int e = tid + p * kGemmThreads;
      As[buf][a_k(e)][a_m(e)] = ra[p];
    }
#pragma unroll
    for (int p = 0; p < kPerB; ++p) {
      const int e = tid + p * kGemmThreads;
      Pair v = rb[p];
      if (CONJ_B) v.y = -v.y;  // op(B) = B^H
      Bs[buf][b_k(e)][b_n(e)] = v;
    }
  };
  auto multiply = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int ks = 0; ks < BK; ks += 4) {
      const int kk = ks + (lane >> 4);
      Pair a[NBM], b[NBN];
#pragma unroll
      for (int i = 0; i < NBM; ++i) a[i] = As[buf][kk][wm + 16 * i + (lane & 15)];
#pragma unroll
      for (int j = 0; j < NBN; ++j) b[j] = Bs[buf][kk][wn + 16 * j + (lane & 15)];
      // the two products of an accumulator stand apart: the matrix core does
      // not wait for the first before it takes the second
#pragma unroll
      for (int i = 0; i < NBM; ++i)
#pragma unroll
        for (int j = 0; j < NBN; ++j) {
          re[i][j] = Mfma<T>::op(a[i].x, b[j].x, re[i][j]);
          im[i][j] = Mfma<T>::op(a[i].x, b[j].y, im[i][j]);
        }
#pragma unroll
      for (int i = 0; i < NBM; ++i) {
        const T ai_re = CONJ_A ? a[i].y : -a[i].y;
        const T ai_im = CONJ_A ? -a[i].y : a[i].y;
#pragma unroll
        for (int j = 0; j < NBN; ++j) {
          re[i][j] = Mfma<T>::op(ai_re, b[j].y, re[i][j]);
          im[i][j] = Mfma<T>::op(ai_im, b[j].x, im[i][j]);
        }
      }
    }
  };

  // sums of the chains
  constexpr bool kChains = G::chains && CONJ_A;
  Acc sre[kChains ? NBM : 1][kChains ? NBN : 1], sim[kChains ? NBM : 1][kChains ? NBN : 1];
  if constexpr (kChains) {
#pragma unroll
    for (int i = 0; i < NBM; ++i)
#pragma unroll
      for (int j = 0; j < NBN; ++j) {
        sre[i][j] = re[i][j];
        sim[i][j] = im[i][j];
      }
  }
  if (kbeg < kend) {
    fetch(kbeg);
    store(0);
    __syncthreads();
  }
  int buf = 0;
  const int chain_steps = gemm_chain<NBM * NBN>(kend - kbeg) / BK;
  int chain = chain_steps;  // steps left of this chain
  for (int64_t k0 = kbeg; k0 < kend; k0 += BK) {
    const bool more = k0 + BK < kend;
    if (more) fetch(k0 + BK);
    multiply(buf);
    if (NBUF == 1) __syncthreads();
    else buf ^= 1;
    if (more) store(buf);
    if constexpr (kChains) {
      if (--chain == 0) {
        chain = chain_steps;
#pragma unroll
        for (int i = 0; i < NBM; ++i)
#pragma unroll
          for (int j = 0; j < NBN; ++j) {
            sre[i][j] += re[i][j];
            sim[i][j] += im[i][j];
#pragma unroll
            for (int v = 0; v < 4; ++v) { re[i][j][v] = T(0); im[i][j][v] = T(0); }
          }
      }
    }
    __syncthreads();
  }
  if constexpr (kChains) {
#pragma unroll
    for (int i = 0; i < NBM; ++i)
#pragma unroll
      for (int j = 0; j < NBN; ++j) {
        re[i][j] += sre[i][j];
        im[i][j] += sim[i][j];
      }
  }
}

template <typename T, bool CONJ_A, bool CONJ_B, int TM, int TN, int WAVES_M>
__global__ __launch_bounds__(kGemmThreads, 2) void k_cgemm(
    int64_t M, int64_t N, int64_t K, int64_t kchunk, unsigned mt, unsigned nt, unsigned splits,
    const cplx<T>* __restrict__ A, int64_t lda, const cplx<T>* __restrict__ B, int64_t ldb,
    cplx<T>* __restrict__ C, int64_t ldc, cplx<T>* __restrict__ partial, T alpha_r, T alpha_i,
    T beta_r, T beta_i) {
  using G = GemmTile<T, TM, TN, WAVES_M>;
  constexpr int NBM = G::NBM, NBN = G::NBN;
  unsigned bm, bn, bs;
  gemm_tile(blockIdx.x, mt, nt, splits, bm, bn, bs);
  const int64_t m0 = (int64_t)bm * TM;
  const int64_t n0 = (int64_t)bn * TN;
  const int64_t kbeg = (int64_t)bs * kchunk;
  const int64_t kend = (kbeg + kchunk) < K ? (kbeg + kchunk) : K;
  typename Mfma<T>::acc re[NBM][NBN], im[NBM][NBN];
  gemm_accumulate<T, CONJ_A, CONJ_B, TM, TN, WAVES_M>(M, N, m0, n0, kbeg, kend, A, lda, B, ldb,
                                                      re, im);

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wm = (wave % WAVES_M) * G::WTM;
  const int wn = (wave / WAVES_M) * G::WTN;
  const bool direct = splits == 1;
#pragma unroll
  for (int i = 0; i < NBM; ++i)
#pragma unroll
    for (int j = 0; j < NBN; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int64_t row = m0 + wm + 16 * i + Mfma<T>::row(lane, v);
        const int64_t col = n0 + wn + 16 * j + (lane & 15);
        if (row >= M || col >= N) continue;
        const T sr = re[i][j][v], si = im[i][j][v];
        if (direct) {
          cplx<T> out;
          out.x = alpha_r * sr - alpha_i * si;
          out.y = alpha_r * si + alpha_i * sr;
          if (beta_r != T(0) || beta_i != T(0)) {
            const cplx<T> c = C[row + col * ldc];
            out.x += beta_r * c.x - beta_i * c.y;
            out.y += beta_r * c.y + beta_i * c.x;
          }
          C[row + col * ldc] = out;
        } else {
          partial[((int64_t)bs * N + col) * M + row] = mk<T>(sr, si);
        }
      }
}

// Sums the split-K partial tiles: a block owns 64 consecutive outputs and
// each of its four waves adds every fourth split (eight loads in flight per
// lane); the four partial sums are combined in LDS in wave order, so the
// summation order is fixed and results are reproducible.
template <typename T>
__global__ __launch_bounds__(256) void k_reduce_splits(
    int64_t M, int64_t N, int splits, const cplx<T>* __restrict__ partial,
    cplx<T>* __restrict__ C, int64_t ldc, T alpha_r, T alpha_i, T beta_r, T beta_i) {
  __shared__ T sr_part[4][64], si_part[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t total = M * N;
  const int64_t idx = (int64_t)blockIdx.x * 64 + lane;
  T sr = T(0), si = T(0);
  if (idx < total) {
    const cplx<T>* p = partial + idx;
    int z = wave;
    for (; z + 28 < splits; z += 32) {
      cplx<T> v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = p[(int64_t)(z + 4 * u) * total];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        sr += v[u].x;
        si += v[u].y;
      }
    }
    for (; z < splits; z += 4) {
      const cplx<T> v = p[(int64_t)z * total];
      sr += v.x;
      si += v.y;
    }
  }
  sr_part[wave][lane] = sr;
  si_part[wave][lane] = si;
  __syncthreads();
  if (wave != 0 || idx >= total) return;
  sr = sr_part[0][lane] + sr_part[1][lane] + sr_part[2][lane] + sr_part[3][lane];
  si = si_part[0][lane] + si_part[1][lane] + si_part[2][lane] + si_part[3][lane];
  const int64_t col = idx / M, row = idx - col * M;
  cplx<T> out;
  out.x = alpha_r * sr - alpha_i * si;
  out.y = alpha_r * si + alpha_i * sr;
  if (beta_r != T(0) || beta_i != T(0)) {
    const cplx<T> c = C[row + col * ldc];
    out.x += beta_r * c.x - beta_i * c.y;
    out.y += beta_r * c.y + beta_i * c.x;
  }
  C[row + col * ldc] = out;
}

// One-column products (n = 1: a single band's projections and projector
// sums) as matrix-vector passes instead of MFMA tiles with one live column.
//   k_gemv_n: sum_j A[i + j lda] b_j, one workgroup per 64 rows, a lane a row;
//             its sixteen waves take every sixteenth column, in two chains;
//   k_gemv_c: sum_g conj(A[g + i lda]) b_g, one workgroup per i with a
//             fixed-order tree sum of four chains a thread.
// b_j = B[j bstride], conjugated when CB.  Both finish the sum in the workgroup and
// scale it by alpha, beta.  Deep products (gemv_direct) take k_gemv_n_split or
// SPLIT, 256 wide, whose partials part[s * m + i] k_reduce_splits sums in a fixed
// order.  Bound by launches at a single band, by A's bytes above: an h_psi of 36^3
// takes 82 -> 73 us with the three reductions gone; FP64 23 847 x 256 19.7 -> 17.3
// us, its A^H 18.6 -> 17.2.
template <typename T>
__device__ __forceinline__ void gemv_store(cplx<T>* C, int64_t i, T sr, T si, T alpha_r, T alpha_i,
                                           T beta_r, T beta_i) {
  cplx<T> out;
  out.x = alpha_r * sr - alpha_i * si;
  out.y = alpha_r * si + alpha_i * sr;
  if (beta_r != T(0) || beta_i != T(0)) {
    const cplx<T> c = C[i];
    out.x += beta_r * c.x - beta_i * c.y;
    out.y += beta_r * c.y + beta_i * c.x;
  }
  C[i] = out;
}

constexpr int kGemvWaves = 16;  // k_gemv_n adds them in pairs

template <typename T, bool CB>
__global__ __launch_bounds__(64 * kGemvWaves) void k_gemv_n(
    int64_t m, int64_t k, const cplx<T>* __restrict__ A, int64_t lda,
    const cplx<T>* __restrict__ B, int64_t bstride, cplx<T>* __restrict__ C, T alpha_r, T alpha_i,
    T beta_r, T beta_i) {
  __shared__ T shr[kGemvWaves][64], shi[kGemvWaves][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t i = (int64_t)blockIdx.x * 64 + lane;
  const cplx<T>* row = A + (i < m ? i : m - 1);
  constexpr int W = kGemvWaves;
  T sr = T(0), si = T(0), tr = T(0), ti = T(0);
  auto add = [&](T& pr, T& pi, const cplx<T> x, const cplx<T> y) __attribute__((always_inline)) {
    const T yi = CB ? -y.y : y.y;
    pr += x.x * y.x - x.y * yi;
    pi += x.x * yi + x.y * y.x;
  };
  int64_t j = wave;
  for (; j + 3 * W < k; j += 4 * W) {
    cplx<T> x[4], y[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      x[u] = row[(j + u * W) * lda];
      y[u] = B[(j + u * W) * bstride];
    }
    add(sr, si, x[0], y[0]);
    add(tr, ti, x[1], y[1]);
    add(sr, si, x[2], y[2]);
    add(tr, ti, x[3], y[3]);
  }
  for (; j < k; j += W) add(sr, si, row[j * lda], B[j * bstride]);
  shr[wave][lane] = sr + tr;
  shi[wave][lane] = si + ti;
  __syncthreads();
  if (wave != 0 || i >= m) return;
  T pr[4], pi[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int w = 4 * q;
    pr[q] = (shr[w][lane] + shr[w + 1][lane]) + (shr[w + 2][lane] + shr[w + 3][lane]);
    pi[q] = (shi[w][lane] + shi[w + 1][lane]) + (shi[w + 2][lane] + shi[w + 3][lane]);
  }
  pr[0] = (pr[0] + pr[1]) + (pr[2] + pr[3]);
  pi[0] = (pi[0] + pi[1]) + (pi[2] + pi[3]);
  gemv_store<T>(C, i, pr[0], pi[0], alpha_r, alpha_i, beta_r, beta_i);
}

template <typename T, bool CB>
__global__ __launch_bounds__(256) void k_gemv_n_split(int64_t m, int64_t k, int64_t kchunk,
                                                      const cplx<T>* __restrict__ A, int64_t lda,
                                                      const cplx<T>* __restrict__ B,
                                                      int64_t bstride, cplx<T>* __restrict__ part) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= m) return;
  const int64_t j0 = (int64_t)blockIdx.y * kchunk;
  const int64_t j1 = j0 + kchunk < k ? j0 + kchunk : k;
  T sr = T(0), si = T(0);
#pragma unroll 8
  for (int64_t j = j0; j < j1; ++j) {
    const cplx<T> a = A[i + j * lda];
    const cplx<T> b = B[j * bstride];
    const T bi = CB ? -b.y : b.y;
    sr += a.x * b.x - a.y * bi;
    si += a.x * bi + a.y * b.x;
  }
  part[(int64_t)blockIdx.y * m + i] = mk<T>(sr, si);
}

template <typename T, bool CB, bool SPLIT>
__global__ __launch_bounds__(SPLIT ? 256 : 1024) void k_gemv_c(
    int64_t m, int64_t k, int64_t kchunk, const cplx<T>* __restrict__ A, int64_t lda,
    const cplx<T>* __restrict__ B, int64_t bstride, cplx<T>* __restrict__ part, T alpha_r,
    T alpha_i, T beta_r, T beta_i) {
  constexpr int THREADS = SPLIT ? 256 : 1024;
  __shared__ T shr[THREADS], shi[THREADS];
  const int64_t i = blockIdx.x;
  const int64_t g0 = SPLIT ? (int64_t)blockIdx.y * kchunk : 0;
  const int64_t g1 = SPLIT && g0 + kchunk < k ? g0 + kchunk : k;
  const cplx<T>* col = A + i * lda;
  T cr[4] = {}, ci[4] = {};
  // (512 x 78 805 split: FP64 115 us, 126 unrolled by four; FP32 90 and 72)
  constexpr int U = SPLIT && sizeof(T) == 8 ? 1 : 4;
#pragma unroll U
  for (int64_t g = g0 + threadIdx.x; g < g1; g += THREADS) {
    const cplx<T> a = col[g];
    const cplx<T> b = B[g * bstride];
    const T bi = CB ? -b.y : b.y;
    cr[0] += a.x * b.x + a.y * bi;
    ci[0] += a.x * bi - a.y * b.x;
    if constexpr (!SPLIT) {  // the next chain's turn: register names, unrolled
      const T r = cr[0], i0 = ci[0];
#pragma unroll
      for (int u = 0; u < 3; ++u) {
        cr[u] = cr[u + 1];
        ci[u] = ci[u + 1];
      }
      cr[3] = r;
      ci[3] = i0;
    }
  }
  const T sr = (cr[0] + cr[1]) + (cr[2] + cr[3]);
  const T si = (ci[0] + ci[1]) + (ci[2] + ci[3]);
  const int tid = threadIdx.x;
  shr[tid] = sr;
  shi[tid] = si;
  __syncthreads();
  for (int w = THREADS / 2; w > 0; w >>= 1) {
    if (tid < w) {
      shr[tid] += shr[tid + w];
      shi[tid] += shi[tid + w];
    }
    __syncthreads();
  }
  if (tid != 0) return;
  if (SPLIT) part[(int64_t)blockIdx.y * m + i] = mk<T>(shr[0], shi[0]);
  else gemv_store<T>(part, i, shr[0], shi[0], alpha_r, alpha_i, beta_r, beta_i);
}

// Splits of a one-column product, whose partials the caller's workspace holds:
// about 1024 workgroups in all, each split of K at least 8 columns of A or, of A^H,
// 1024 rows.
struct GemvPlan {
  int64_t splits;
  int64_t kchunk;
};

static GemvPlan gemv_plan(bool ca, int64_t m, int64_t k) {
  const int64_t blocks = ca ? m : (m + 255) / 256;
  const int64_t most = ca ? (k + 1023) / 1024 : (k + 7) / 8;
  int64_t splits = (1024 + blocks - 1) / blocks;
  if (splits > most) splits = most;
  if (splits > 65535) splits = 65535;
  if (splits < 1) splits = 1;
  const int64_t kchunk = (k + splits - 1) / splits;
  return {(k + kchunk - 1) / kchunk, kchunk};
}

// Whether a one-column product runs unsplit: where it fills the chip, or ends sooner
// than a second kernel starts.  Beyond, split and unsplit: FP64 64 x 2000 13.9 and
// 29.1 us, FP32 78 805 x 512 56 and 65; A^H FP64 64 x 100 000 21 and 35, 512 x 78 805
// 115 and 122.  (A launch runs fewer than 2^32 threads, and more wrap without an
// error: the rows beyond take the split kernels, of 256 threads.)
static bool gemv_direct(bool ca, int64_t m, int64_t k) {
  if ((ca ? m : (m + 63) / 64) > kMaxLaunch / (64 * kGemvWaves)) return false;
  return ca ? k <= 8192 || (m >= 64 && k <= 32768) : k <= 384;
}

// The projector force, dE/dtau_a,c = 2 sum_n f_n Re sum_{i in a} conj(dO_c[i,n])
// (D O)[i,n] with dO_c = i B^H (q_c psi), in one product over the bands instead of
// three over the plane waves: with W = psi (f D O)^H (npw x P),
//   dE/dtau_a,c = 2 sum_G q_c(G) sum_{i in a} Im(B[G,i] conj(W[G,i])),
// so W is contracted with B and q in the tile's epilogue and never stored.  Each
// wave writes the sums of its rows, in FP64 for both precisions, to
// partial[(c P + i) parts + part]; k_force_sum adds them in a fixed order.
//
// Bound by the product's FP64 MFMAs (8 npw P nb flops, a third of the former
// ones, which also read psi, scaled, three times).  23 847 x 256 projectors x
// 128 bands: the three scalings and products with their reductions took 430 us
// in FP64, this and its sums 137.
template <typename T, int TM, int TN, int WAVES_M>
__global__ __launch_bounds__(kGemmThreads, 2) void k_force_product(
    int64_t npw, int64_t nproj, int64_t nb, unsigned mt, unsigned nt,
    const cplx<T>* __restrict__ psi, int64_t ldpsi, const cplx<T>* __restrict__ fdo,
    int64_t ldf, const cplx<T>* __restrict__ proj, int64_t ldproj, const double* __restrict__ q,
    double* __restrict__ partial) {
  using G = GemmTile<T, TM, TN, WAVES_M>;
  constexpr int NBM = G::NBM, NBN = G::NBN;
  unsigned bm, bn, bs;
  gemm_tile(blockIdx.x, mt, nt, 1, bm, bn, bs);
  const int64_t m0 = (int64_t)bm * TM;
  const int64_t n0 = (int64_t)bn * TN;
  typename Mfma<T>::acc re[NBM][NBN], im[NBM][NBN];
  gemm_accumulate<T, false, true, TM, TN, WAVES_M>(npw, nproj, m0, n0, 0, nb, psi, ldpsi, fdo,
                                                   ldf, re, im);

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int64_t row0 = m0 + (wave % WAVES_M) * G::WTM;
  const int64_t col0 = n0 + (wave / WAVES_M) * G::WTN + (lane & 15);
  double sum[NBN][3];
#pragma unroll
  for (int j = 0; j < NBN; ++j) sum[j][0] = sum[j][1] = sum[j][2] = 0.0;
#pragma unroll
  for (int i = 0; i < NBM; ++i)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int64_t row = row0 + 16 * i + Mfma<T>::row(lane, v);
      if (row >= npw) continue;
      const double q0 = q[3 * row], q1 = q[3 * row + 1], q2 = q[3 * row + 2];
#pragma unroll
      for (int j = 0; j < NBN; ++j) {
        const int64_t col = col0 + 16 * j;
        if (col >= nproj) continue;
        const cplx<T> b = proj[row + col * ldproj];
        const double z = (double)b.y * re[i][j][v] - (double)b.x * im[i][j][v];
        sum[j][0] += q0 * z;
        sum[j][1] += q1 * z;
        sum[j][2] += q2 * z;
      }
    }
  // the four lanes of a column
  const int64_t parts = (int64_t)mt * WAVES_M;
  const int64_t part = (int64_t)bm * WAVES_M + wave % WAVES_M;
#pragma unroll
  for (int j = 0; j < NBN; ++j) {
    const int64_t col = col0 + 16 * j;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      double s = sum[j][c];
      s += __shfl_xor(s, 16);
      s += __shfl_xor(s, 32);
      if (lane < 16 && col < nproj) partial[(c * nproj + col) * parts + part] = s;
    }
  }
}

// out[a, c] = 2 sum of the partials of atom a's projectors [off[a], off[a+1])
__global__ __launch_bounds__(1024) void k_force_sum(const double* __restrict__ partial,
                                                    int64_t nproj, int64_t parts,
                                                    const int* __restrict__ off,
                                                    double* __restrict__ out) {
  __shared__ double sh[1024];
  const int a = blockIdx.x, c = blockIdx.y, tid = threadIdx.x;
  const int i0 = off[a];
  const int64_t count = (int64_t)(off[a + 1] - i0) * parts;
  const double* p = partial + (c * nproj + i0) * parts;
  double s = 0.0;
  for (int64_t e = tid; e < count; e += 1024) s += p[e];
  sh[tid] = s;
  __syncthreads();
  for (int h = 512; h > 0; h >>= 1) {
    if (tid < h) sh[tid] += sh[tid + h];
    __syncthreads();
  }
  if (tid == 0) out[3 * a + c] = 2.0 * sh[0];
}

// Tile variants of k_cgemm: (TM, TN, WAVES_M).
struct GemmVariant {
  int tm, tn, waves_m;
};
constexpr GemmVariant kVariants[] = {
    {32, 32, 2},    // 0: small outputs (the reduced problem), wave 16x16
    {64, 64, 2},    // 1: square-ish outputs, wave 32x32
    {32, 128, 1},   // 2: tall outputs with up to 128 columns: A streamed once
    {64, 128, 2},   // 3: tall outputs, wave 32x64
    {128, 64, 2},   // 4: tall-row outputs (A^H B with m > n), wave 64x32
    {128, 32, 4},   // 5: tall outputs with 32 columns
    {32, 64, 1},    // 6: tall outputs with up to 64 columns, wave 32x16
    {64, 16, 4},    // 7: at most 16 columns (a solve's last roots), wave 16x16
};
constexpr int kNumVariants = (int)(sizeof(kVariants) / sizeof(kVariants[0]));

struct SplitPlan {
  int64_t splits;
  int64_t kchunk;
  int variant;
};

// Tuned choices (qepw_gemm_set_rule): the first rule whose ranges hold the
// shape wins over the built-in choice.
struct GemmRule {
  int precision, op;
  int64_t m_lo, m_hi, n_lo, n_hi, k_lo, k_hi;
  int variant;
  int64_t splits;
};
constexpr int kMaxRules = 256;
GemmRule g_rules[kMaxRules];
int g_nrules = 0;

static int64_t tiles_of(int variant, int64_t m, int64_t n) {
  const GemmVariant& v = kVariants[variant];
  return ((m + v.tm - 1) / v.tm) * ((n + v.tn - 1) / v.tn);
}

static SplitPlan finish_plan(int variant, int64_t splits, int64_t k) {
  constexpr int kBK = 16;  // a whole number of steps of every kernel
  if (splits < 1) splits = 1;
  int64_t kchunk = (k + splits - 1) / splits;
  kchunk = ((kchunk + kBK - 1) / kBK) * kBK;
  if (kchunk < kBK) kchunk = kBK;
  splits = (k + kchunk - 1) / kchunk;
  if (splits < 1) splits = 1;
  return {splits, kchunk, variant};
}

// The time of one choice in microseconds, as measured on 47 shapes (8 .. 78 805
// rows, 2 .. 512 columns, depths 8 .. 78 805) with every tile and 19 split
// counts: the chosen tile and split are within 3% of the best measured in the
// mean and 8% at products of more than 20 us.  256 CUs run their tiles at a
// rate that depends on the tile shape (the wave tile's ratio of MFMAs to LDS
// reads), or, with few tiles, one K step per latency; a split writes and sums
// partial tiles.
static double plan_cost(int precision, int variant, int64_t m, int64_t n, int64_t splits,
                        int64_t kchunk) {
  const bool fp64 = precision == QEPW_C128;
  // TFLOP/s of each tile, and the workgroups a CU holds
  static constexpr double rate64[] = {53.6, 61.6, 57.0, 57.6, 58.0, 55.4, 56.3, 47.7};
  static constexpr double rate32[] = {111.0, 112.2, 102.8, 102.8, 107.4, 101.6, 110.3, 84.8};
  static constexpr int hold64[] = {4, 4, 3, 2, 2, 3, 5, 5};
  static constexpr int hold32[] = {8, 4, 3, 3, 3, 3, 6, 8};
  const GemmVariant& v = kVariants[variant];
  const double size = fp64 ? 16.0 : 8.0;
  const double q = (double)(tiles_of(variant, m, n) * splits) / 256.0;
  const double waves = std::ceil(q / (fp64 ? hold64 : hold32)[variant]);
  const double tile = 8.0 * v.tm * v.tn * (double)kchunk * 256.0 /
                      ((fp64 ? rate64 : rate32)[variant] * 1e6);
  // a tile alone on its CU does not hide its own loads and barriers (the
  // single-buffered FP32 tile least)
  const double on = std::min(std::ceil(q), (double)(fp64 ? hold64 : hold32)[variant]);
  const double bare = !fp64 && variant == 0 ? 0.6 / on : 0.25 / (on * on);
  const double compute = (q < 6.0 ? std::ceil(q) : q + 0.5) * tile * (1.0 + bare);
  // us per column of K
  const double step = fp64 ? (v.tm * v.tn > 1024 ? 0.166 : 0.050) : 0.039;
  double t = std::max(compute, waves * (double)kchunk * step) + waves * (fp64 ? 0.1 : 1.9);
  if (splits > 1)
    t += (fp64 ? 3.2 : 2.5) + (double)splits * m * n * size / (fp64 ? 4.9e6 : 7.8e6);
  return t;
}

// a plan that needs no search, and no more scratch than callers that size
// theirs by other means than qepw_gemm_workspace provide
static SplitPlan fixed_plan(int op_a, int64_t m, int64_t n, int64_t k) {
  if (m <= 0 || n <= 0 || k <= 0) return finish_plan(0, 1, k);
  const bool ca = (op_a & QEPW_OP_C) != 0;
  const bool tall = ca && k > 2048;
  int variant;
  if (tall) {
    // A^H B over npw: parallelism from splitting K
    variant = 1;
  } else if (!ca && m > 4096 && n <= 128) {
    // npw x n outputs (Ritz vectors, residuals, projector sums): all n
    // columns in one workgroup, so the npw x k operand is read once
    variant = n > 64 ? 2 : (n > 32 ? 6 : 0);
  } else {
    const int64_t tiles64 = ((m + 63) / 64) * ((n + 63) / 64);
    variant = tiles64 < 256 ? 0 : 1;
  }
  const int64_t tiles = tiles_of(variant, m, n);
  int64_t splits = 1;
  // split K when the output tiles alone cannot fill the 256 CUs: the tall
  // A^H B products over npw (about two workgroups per CU and at least 256 of
  // K per split: shorter splits spend more on writing and summing their
  // partial tiles than on the product) and the small square products of the
  // reduced eigensolve (small partial tiles: four workgroups per CU, at
  // least 128 of K per split)
  if (tall || (ca && k > 512) || (tiles < 256 && k >= 256)) {
    const int64_t want = ((tall ? 512 : 1024) + tiles - 1) / tiles;
    const int64_t most = k / (tall ? 256 : 128);
    splits = want < most ? want : most;
  }
  return finish_plan(variant, splits, k);
}

static SplitPlan built_in_plan(int precision, int op_a, int64_t m, int64_t n, int64_t k) {
  const SplitPlan fixed = fixed_plan(op_a, m, n, k);
  if (m <= 0 || n <= 0 || k <= 0) return fixed;
  // partial tiles stay within the static scratch (qepw_gemm_static) where the
  // fixed choice's do, and within four times that where they do not: with the
  // operands of 512 x 192 x 78 805 at 1.2 GB, 21 splits take 1.12 ms, 32 1.02
  const int64_t out_bytes = m * n * (precision == QEPW_C128 ? 16 : 8);
  const int64_t scratch = (int64_t)QEPW_GEMM_STATIC_SCRATCH;
  const bool over = fixed.splits > 1 && fixed.splits > scratch / out_bytes;
  // A^H B of fewer than 256 columns stays unsplit: Gram matrices of small bases
  // keep the order of their sums, which decides the pivot's sign where a basis is
  // singular to the last bit.  A B is split down to chunks of 32 (the D coupling,
  // 168 x 96 x 168 in FP32, with its h_psi: 172 us unsplit, 166 split)
  const int64_t most = (op_a & QEPW_OP_C) && k < 256
                           ? 1
                           : std::min(k / 32, (over ? 4 : 1) * scratch / out_bytes);
  // ... of which one row or column of tiles has to fit the static scratch
  // (split_panel)
  const auto most_of = [&](const GemmVariant& v) {
    const int64_t panel = std::min(std::min<int64_t>(v.tm, m) * n, m * std::min<int64_t>(v.tn, n));
    return over ? std::min(most, scratch * m * n / (panel * out_bytes)) : most;
  };
  SplitPlan best = fixed;
  double cost = plan_cost(precision, fixed.variant, m, n, fixed.splits, fixed.kchunk);
  for (int v = 0; v < kNumVariants; ++v) {
    const int64_t vt = tiles_of(v, m, n);
    int64_t last = 0;
    // unsplit, and the splits that give each CU one, two, ... eight tiles, up
    // to what the scratch holds and to chunks of 32 columns
    for (int per = 0; per <= 8; ++per) {
      const int64_t s = per == 0 ? 1 : std::min(most_of(kVariants[v]), 256 * per / vt);
      if (s <= last) continue;
      last = s;
      const SplitPlan p = finish_plan(v, s, k);
      const double c = plan_cost(precision, v, m, n, p.splits, p.kchunk);
      if (c < cost) {
        cost = c;
        best = p;
      }
    }
  }
  return best;
}

// The plan of a shape: a rule's (qepw_gemm_set_rule), or the cheapest by
// plan_cost, remembered per thread (a search costs about a microsecond).
static SplitPlan split_plan(int precision, int op_a, int64_t m, int64_t n, int64_t k) {
  for (int r = 0; r < g_nrules; ++r) {
    const GemmRule& g = g_rules[r];
    if (g.precision == precision && g.op == op_a && m >= g.m_lo && m <= g.m_hi &&
        n >= g.n_lo && n <= g.n_hi && k >= g.k_lo && k <= g.k_hi)
      return finish_plan(g.variant, g.splits, k);
  }
  struct Known {
    int64_t m = -1, n = 0, k = 0;
    int precision = 0, op = 0;
    SplitPlan plan{};
  };
  constexpr int kKnown = 256;
  static thread_local Known known[kKnown];
  const uint64_t h = (uint64_t)m * 0x9E3779B97F4A7C15ull ^ (uint64_t)n * 0xC2B2AE3D27D4EB4Full ^
                     (uint64_t)k * 0x165667B19E3779F9ull ^ (uint64_t)(op_a * 2 + precision) << 56;
  Known& e = known[(h >> 32) % kKnown];
  if (e.m != m || e.n != n || e.k != k || e.precision != precision || e.op != op_a) {
    e.plan = built_in_plan(precision, op_a, m, n, k);
    e.m = m;
    e.n = n;
    e.k = k;
    e.precision = precision;
    e.op = op_a;
  }
  return e.plan;
}

int gemm_set_rule(int precision, int op_a, const int64_t* ranges, int variant, int64_t splits) {
  if (precision != QEPW_C128 && precision != QEPW_C64) return QEPW_ERR_ARG;
  if (op_a & ~(QEPW_OP_C | QEPW_OP_BC)) return QEPW_ERR_ARG;
  if (variant < 0 || variant >= kNumVariants || splits < 1 || splits > 65535 || !ranges)
    return QEPW_ERR_ARG;
  if (g_nrules >= kMaxRules) return QEPW_ERR_UNSUPPORTED;
  g_rules[g_nrules++] = {precision, op_a,      ranges[0], ranges[1], ranges[2],
                         ranges[3], ranges[4], ranges[5], variant,   splits};
  return QEPW_OK;
}

void gemm_clear_rules() { g_nrules = 0; }

int gemm_variant_count() { return kNumVariants; }

int gemm_plan(int precision, int op_a, int64_t m, int64_t n, int64_t k, int64_t* out) {
  const SplitPlan sp = split_plan(precision, op_a & (QEPW_OP_C | QEPW_OP_BC), m, n, k);
  out[0] = sp.variant;
  out[1] = sp.splits;
  out[2] = kVariants[sp.variant].tm;
  out[3] = kVariants[sp.variant].tn;
  return QEPW_OK;
}

// Of the 32 x 32 and the 64 x 64 tile the cheaper for the product by plan_cost:
// 10 127 x 108 projectors x 60 bands in FP32 20.7 us with the large tile, 1.2 of
// which a CU gets, 14.8 with the small one.
static int force_variant(int precision, int64_t npw, int64_t nproj, int64_t nb) {
  return plan_cost(precision, 0, npw, nproj, 1, nb) < plan_cost(precision, 1, npw, nproj, 1, nb)
             ? 0
             : 1;
}

static int64_t force_parts(int precision, int64_t npw, int64_t nproj, int64_t nb) {
  const GemmVariant& v = kVariants[force_variant(precision, npw, nproj, nb)];
  return (npw + v.tm - 1) / v.tm * v.waves_m;
}

// the weighted couplings (a multiple of 256 bytes), then the partial sums
static size_t force_weighted_bytes(int precision, int64_t nproj, int64_t nb) {
  const size_t elem = precision == QEPW_C128 ? sizeof(double2) : sizeof(float2);
  return ((size_t)nproj * (size_t)nb * elem + 255) & ~(size_t)255;
}

size_t position_gradient_bytes(int precision, int64_t npw, int64_t nproj, int64_t nb) {
  if (npw <= 0 || nproj <= 0 || nb < 0) return 0;
  return force_weighted_bytes(precision, nproj, nb) +
         (size_t)3 * nproj * force_parts(precision, npw, nproj, nb) * sizeof(double);
}

template <typename T>
static int force_product_t(int64_t npw, int64_t nproj, int64_t nb, const void* psi,
                           int64_t ldpsi, const cplx<T>* fdo, const void* proj, int64_t ldproj,
                           const double* q, double* partial, hipStream_t stream) {
  const int variant =
      force_variant(std::is_same<T, double>::value ? QEPW_C128 : QEPW_C64, npw, nproj, nb);
  const GemmVariant& v = kVariants[variant];
  const int64_t mt = (npw + v.tm - 1) / v.tm, nt = (nproj + v.tn - 1) / v.tn;
  if (mt > kMaxLaunch / kGemmThreads / nt) return QEPW_ERR_UNSUPPORTED;
  const dim3 grid((unsigned)(mt * nt));
  const cplx<T>* x = static_cast<const cplx<T>*>(psi);
  const cplx<T>* b = static_cast<const cplx<T>*>(proj);
  if (variant == 0)
    hipLaunchKernelGGL((k_force_product<T, 32, 32, 2>), grid, dim3(kGemmThreads), 0, stream, npw,
                       nproj, nb, (unsigned)mt, (unsigned)nt, x, ldpsi, fdo, nproj, b, ldproj, q,
                       partial);
  else
    hipLaunchKernelGGL((k_force_product<T, 64, 64, 2>), grid, dim3(kGemmThreads), 0, stream, npw,
                       nproj, nb, (unsigned)mt, (unsigned)nt, x, ldpsi, fdo, nproj, b, ldproj, q,
                       partial);
  return hipGetLastError() == hipSuccess ? QEPW_OK : QEPW_ERR_HIP;
}

int position_gradient(int precision, int64_t npw, int64_t nproj, int nb, const void* psi,
                      int64_t ldpsi, const void* coupled, int64_t ldc, const double* f,
                      const void* proj, int64_t ldproj, const double* q, const int* off,
                      int natom, double* out, void* ws, size_t ws_bytes, hipStream_t stream) {
  if (precision != QEPW_C128 && precision != QEPW_C64) return QEPW_ERR_ARG;
  if (natom <= 0) return QEPW_OK;
  if (natom > 0x7fffffff / 3) return QEPW_ERR_UNSUPPORTED;
  if (ws_bytes < position_gradient_bytes(precision, npw, nproj, nb)) return QEPW_ERR_WORKSPACE;
  double* partial = nullptr;
  int64_t parts = 0;
  if (npw > 0 && nproj > 0) {
    parts = force_parts(precision, npw, nproj, nb);
    partial = reinterpret_cast<double*>(static_cast<char*>(ws) +
                                        force_weighted_bytes(precision, nproj, nb));
    int rc = scale_rows(precision, coupled, ldc, nullptr, 0, f, ws, nproj, nproj, nb, stream);
    if (rc != QEPW_OK) return rc;
    rc = precision == QEPW_C128
             ? force_product_t<double>(npw, nproj, nb, psi, ldpsi, static_cast<double2*>(ws),
                                       proj, ldproj, q, partial, stream)
             : force_product_t<float>(npw, nproj, nb, psi, ldpsi, static_cast<float2*>(ws), proj,
                                      ldproj, q, partial, stream);
    if (rc != QEPW_OK) return rc;
  }
  hipLaunchKernelGGL(k_force_sum, dim3((unsigned)natom, 3), dim3(1024), 0, stream, partial, nproj,
                     parts, off, out);
  return hipGetLastError() == hipSuccess ? QEPW_OK : QEPW_ERR_HIP;
}

// Products of commuting Hermitian matrices (the Newton-Schulz steps of the
// reduced eigensolve): C = alpha X Y + beta D with X, Y, D Hermitian
// polynomials of one matrix, so that C is Hermitian.  Only the lower-triangle
// 16x16 tiles are computed, one per workgroup, and each is written together
// with its conjugate transpose (the diagonal made real): C is exactly
// Hermitian, which the conjugated loads of Y below rely on.  Y's element
// (k, j) is read as conj(Y[j, k]), a contiguous run like X's (i, k).  The eight
// waves of a workgroup split K, each fetching its next kHermUnroll MFMA
// steps while the current ones run, and their partial tiles are summed in LDS
// in wave order, so results are reproducible.  Bound by each wave's chain of
// loads up to n ~ 200, by the tiles' L2 reads above.  n = 32 / 128 / 264 / 432 /
// 512 with four, eight and sixteen waves: 4.0 / 5.7 / 9.7 / 16.3 / 23.4, 3.9 /
// 5.0 / 8.0 / 14.6 / 21.4 and 4.8 / 5.7 / 8.6 / 16.3 / 22.5 us a launch.  Two
// steps in flight (with four waves n = 264 / 432 / 512 take 18-23% longer with
// eight; four and six lie in between).
constexpr int kHermUnroll = 2;
constexpr int kHermWaves = 8;

__global__ __launch_bounds__(64 * kHermWaves) void k_herm_product(
    int n, const double2* __restrict__ X, const double2* __restrict__ Y,
    const double2* __restrict__ D, double2* __restrict__ C, int64_t ld, double alpha,
    double beta) {
  constexpr int U = kHermUnroll, W = kHermWaves;
  __shared__ double2 part[W][256];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // tile (ti, tj), ti >= tj, of linear index b = ti (ti + 1) / 2 + tj
  const int b = blockIdx.x;
  int ti = (int)((sqrt(8.0 * b + 1.0) - 1.0) * 0.5);
  while ((ti + 1) * (ti + 2) / 2 <= b) ++ti;
  while (ti * (ti + 1) / 2 > b) --ti;
  const int tj = b - ti * (ti + 1) / 2;
  const int m0 = 16 * ti, n0 = 16 * tj;
  // this wave's K steps (4 columns of K each): [s0, s1)
  const int steps = (n + 3) >> 2;
  const int per = (steps + W - 1) / W;
  const int s0 = min(steps, wave * per);
  const int s1 = min(steps, s0 + per);
  const int r = lane & 15, kq = lane >> 4;
  const int row = m0 + r, col = n0 + r;
  const bool rok = row < n, cok = col < n;
  v4d re = {0.0, 0.0, 0.0, 0.0}, im = {0.0, 0.0, 0.0, 0.0};
  // operands are loaded unconditionally from an in-bounds element (the
  // matrix corner when out of range) and zeroed by register selects, which
  // keeps the loads on the global path and the operands in registers
  const double2* xr = X + (rok ? row : 0);
  const double2* yc = Y + (cok ? col : 0);
  double ar[U], ai[U], wr[U], wi[U], nar[U], nai[U], nwr[U], nwi[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int k = 4 * (s0 + u) + kq;
    const bool ok = s0 + u < s1 && k < n;
    const int64_t off = ok ? (int64_t)k * ld : 0;
    const double2 xa = xr[off], yw = yc[off];
    const bool ua = ok && rok, uw = ok && cok;
    ar[u] = ua ? xa.x : 0.0;
    ai[u] = ua ? xa.y : 0.0;
    wr[u] = uw ? yw.x : 0.0;
    wi[u] = uw ? yw.y : 0.0;
  }
  for (int s = s0; s < s1; s += U) {
    const int sn = s + U;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = 4 * (sn + u) + kq;
      const bool ok = sn + u < s1 && k < n;
      const int64_t off = ok ? (int64_t)k * ld : 0;
      const double2 xa = xr[off], yw = yc[off];
      const bool ua = ok && rok, uw = ok && cok;
      nar[u] = ua ? xa.x : 0.0;
      nai[u] = ua ? xa.y : 0.0;
      nwr[u] = uw ? yw.x : 0.0;
      nwi[u] = uw ? yw.y : 0.0;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      // (X Y)_ij += X_ik conj(Y_jk)
      re = Mfma<double>::op(ar[u], wr[u], re);
      re = Mfma<double>::op(ai[u], wi[u], re);
      im = Mfma<double>::op(ai[u], wr[u], im);
      im = Mfma<double>::op(-ar[u], wi[u], im);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      ar[u] = nar[u];
      ai[u] = nai[u];
      wr[u] = nwr[u];
      wi[u] = nwi[u];
    }
  }
#pragma unroll
  for (int v = 0; v < 4; ++v)
    part[wave][Mfma<double>::row(lane, v) + 16 * r] = make_double2(re[v], im[v]);
  __syncthreads();
  const int er = tid & 15, ec = tid >> 4;
  const int gi = m0 + er, gj = n0 + ec;
  if (ec >= 16 || gi >= n || gj >= n || gi < gj) return;
  double sr = 0.0, si = 0.0;
#pragma unroll
  for (int q = 0; q < W; ++q) {
    sr += part[q][tid].x;
    si += part[q][tid].y;
  }
  double2 out = make_double2(alpha * sr, alpha * si);
  if (beta != 0.0) {
    const double2 d = D[gi + (int64_t)gj * ld];
    out.x += beta * d.x;
    out.y += beta * d.y;
  }
  if (gi == gj) {
    out.y = 0.0;
    C[gi + (int64_t)gj * ld] = out;
  } else {
    C[gi + (int64_t)gj * ld] = out;
    C[gj + (int64_t)gi * ld] = make_double2(out.x, -out.y);
  }
}

int herm_product(int n, const void* x, const void* y, const void* d, void* c, int64_t ld,
                 double alpha, double beta, hipStream_t stream) {
  if (n <= 0) return QEPW_OK;
  if (ld < n) return QEPW_ERR_ARG;
  const int nt = (n + 15) / 16;
  hipLaunchKernelGGL(k_herm_product, dim3((unsigned)(nt * (nt + 1) / 2)), dim3(64 * kHermWaves),
                     0, stream, n, static_cast<const double2*>(x), static_cast<const double2*>(y),
                     static_cast<const double2*>(d), static_cast<double2*>(c), ld, alpha, beta);
  return hipGetLastError() == hipSuccess ? QEPW_OK : QEPW_ERR_HIP;
}

size_t gemm_workspace_bytes(int precision, int op, int64_t m, int64_t n, int64_t k) {
  const size_t elem = precision == QEPW_C128 ? sizeof(double2) : sizeof(float2);
  if (n == 1 && k > 0 && m > 0)
    return (size_t)gemv_plan((op & QEPW_OP_C) != 0, m, k).splits * (size_t)m * elem;
  const SplitPlan sp = split_plan(precision, op & (QEPW_OP_C | QEPW_OP_BC), m, n, k);
  if (sp.splits <= 1) return 0;
  const size_t c = precision == QEPW_C128 ? sizeof(double2) : sizeof(float2);
  return (size_t)sp.splits * (size_t)m * (size_t)n * c;
}

template <typename T>
static int gemv_t(int op, int64_t m, int64_t k, const double* alpha, const void* a, int64_t lda,
                  const void* b, int64_t ldb, const double* beta, void* c, int64_t ldc,
                  void* ws, size_t ws_bytes, hipStream_t stream) {
  const bool ca = (op & QEPW_OP_C) != 0, cb = (op & QEPW_OP_BC) != 0;
  const GemvPlan gp = gemv_plan(ca, m, k);
  if (ws_bytes < (size_t)gp.splits * (size_t)m * sizeof(cplx<T>)) return QEPW_ERR_WORKSPACE;
  // the single column of op(B): B[j] (k x 1), or conj(B[j ldb]) for its (1 x k) adjoint
  const int64_t bstride = cb ? ldb : 1;
  const cplx<T>* pa = static_cast<const cplx<T>*>(a);
  const cplx<T>* pb = static_cast<const cplx<T>*>(b);
  cplx<T>* part = static_cast<cplx<T>*>(ws);
  cplx<T>* pc = static_cast<cplx<T>*>(c);
  const T ar = (T)alpha[0], ai = (T)alpha[1], br = (T)beta[0], bi = (T)beta[1];
  const bool direct = gemv_direct(ca, m, k);
  if (!ca && direct) {
    const dim3 grid((unsigned)((m + 63) / 64));
    if (cb)
      hipLaunchKernelGGL((k_gemv_n<T, true>), grid, dim3(64 * kGemvWaves), 0, stream, m, k, pa,
                         lda, pb, bstride, pc, ar, ai, br, bi);
    else
      hipLaunchKernelGGL((k_gemv_n<T, false>), grid, dim3(64 * kGemvWaves), 0, stream, m, k, pa,
                         lda, pb, bstride, pc, ar, ai, br, bi);
  } else if (!direct) {
    const dim3 grid((unsigned)(ca ? m : (m + 255) / 256), (unsigned)gp.splits);
    if (ca && cb)
      hipLaunchKernelGGL((k_gemv_c<T, true, true>), grid, dim3(256), 0, stream, m, k, gp.kchunk,
                         pa, lda, pb, bstride, part, ar, ai, br, bi);
    else if (ca)
      hipLaunchKernelGGL((k_gemv_c<T, false, true>), grid, dim3(256), 0, stream, m, k, gp.kchunk,
                         pa, lda, pb, bstride, part, ar, ai, br, bi);
    else if (cb)
      hipLaunchKernelGGL((k_gemv_n_split<T, true>), grid, dim3(256), 0, stream, m, k, gp.kchunk,
                         pa, lda, pb, bstride, part);
    else
      hipLaunchKernelGGL((k_gemv_n_split<T, false>), grid, dim3(256), 0, stream, m, k, gp.kchunk,
                         pa, lda, pb, bstride, part);
    hipLaunchKernelGGL(k_reduce_splits<T>, dim3((unsigned)((m + 63) / 64)), dim3(256), 0, stream,
                       m, (int64_t)1, (int)gp.splits, part, pc, ldc, ar, ai, br, bi);
  } else {
    if (cb)
      hipLaunchKernelGGL((k_gemv_c<T, true, false>), dim3((unsigned)m), dim3(1024), 0, stream, m,
                         k, k, pa, lda, pb, bstride, pc, ar, ai, br, bi);
    else
      hipLaunchKernelGGL((k_gemv_c<T, false, false>), dim3((unsigned)m), dim3(1024), 0, stream, m,
                         k, k, pa, lda, pb, bstride, pc, ar, ai, br, bi);
  }
  return hipGetLastError() == hipSuccess ? QEPW_OK : QEPW_ERR_HIP;
}

static size_t split_bytes(const SplitPlan& p, int64_t m, int64_t n, size_t elem) {
  return p.splits > 1 ? (size_t)p.splits * m * n * elem : 0;
}

// A product whose partials exceed its workspace runs in panels of whole tiles, of
// mp rows or np columns, one after the other with the same plan: the bits of the
// result do not depend on the workspace.  False where the workspace is refused:
// short of the fixed choice's partials, or of the static scratch where those
// exceed it, unless two partial outputs already do.
static bool split_panel(const SplitPlan& sp, const SplitPlan& fixed, int64_t m, int64_t n,
                        size_t elem, size_t ws_bytes, int64_t* mp, int64_t* np) {
  const size_t least = std::min(split_bytes(fixed, m, n, elem),
                                std::max(QEPW_GEMM_STATIC_SCRATCH, 2 * (size_t)m * n * elem));
  if (ws_bytes < least) return false;
  const GemmVariant& v = kVariants[sp.variant];
  const int64_t held = (int64_t)(ws_bytes / ((size_t)sp.splits * elem));
  const int64_t rows = held / n / v.tm * v.tm, cols = held / m / v.tn * v.tn;
  if (rows > 0) *mp = rows;
  else if (cols > 0) *np = cols;
  else return false;
  return true;
}

template <typename T>
static int gemm_t(int op, int64_t m, int64_t n, int64_t k, const double* alpha,
                  const void* a, int64_t lda, const void* b, int64_t ldb, const double* beta,
                  void* c, int64_t ldc, void* ws, size_t ws_bytes, hipStream_t stream) {
  if (n == 1 && k > 0)
    return gemv_t<T>(op, m, k, alpha, a, lda, b, ldb, beta, c, ldc, ws, ws_bytes, stream);
  SplitPlan sp = split_plan(std::is_same<T, double>::value ? QEPW_C128 : QEPW_C64,
                                  op & (QEPW_OP_C | QEPW_OP_BC), m, n, k);
  int64_t mp = m, np = n;
  if (ws_bytes < split_bytes(sp, m, n, sizeof(cplx<T>))) {
    const SplitPlan fixed = fixed_plan(op, m, n, k);
    if (fixed.splits == 1 ||
        !split_panel(sp, fixed, m, n, sizeof(cplx<T>), ws_bytes, &mp, &np)) {
      if (ws_bytes < split_bytes(fixed, m, n, sizeof(cplx<T>))) return QEPW_ERR_WORKSPACE;
      sp = fixed;
    }
  }
  if (sp.splits > 65535) return QEPW_ERR_UNSUPPORTED;
  const GemmVariant gv = kVariants[sp.variant];
  const T ar = (T)alpha[0], ai = (T)alpha[1], br = (T)beta[0], bi = (T)beta[1];
  const bool ca = (op & QEPW_OP_C) != 0, cb = (op & QEPW_OP_BC) != 0;
  cplx<T>* part = static_cast<cplx<T>*>(ws);
  for (int64_t m0 = 0; m0 < m; m0 += mp)
    for (int64_t n0 = 0; n0 < n; n0 += np) {
      const int64_t mm = std::min(mp, m - m0), nn = std::min(np, n - n0);
      const int64_t mt = (mm + gv.tm - 1) / gv.tm, nt = (nn + gv.tn - 1) / gv.tn;
      if (mt > 0x7fffffff || nt > 65535 || mt * nt > kMaxLaunch / kGemmThreads / sp.splits)
        return QEPW_ERR_UNSUPPORTED;
      const dim3 grid((unsigned)(mt * nt * sp.splits));
      const cplx<T>* pa = static_cast<const cplx<T>*>(a) + (ca ? m0 * lda : m0);
      const cplx<T>* pb = static_cast<const cplx<T>*>(b) + (cb ? n0 : n0 * ldb);
      cplx<T>* pc = static_cast<cplx<T>*>(c) + m0 + n0 * ldc;
#define QEPW_GEMM_TILE(CA, CB, TM, TN, WM)                                                \
  hipLaunchKernelGGL((k_cgemm<T, CA, CB, TM, TN, WM>), grid, dim3(kGemmThreads), 0, stream, \
                     mm, nn, k, sp.kchunk, (unsigned)mt, (unsigned)nt, (unsigned)sp.splits, pa, \
                     lda, pb, ldb, pc, ldc, part, ar, ai, br, bi)
#define QEPW_GEMM_LAUNCH(CA, CB)                                   \
  do {                                                             \
    switch (sp.variant) {                                          \
      case 0: QEPW_GEMM_TILE(CA, CB, 32, 32, 2); break;            \
      case 1: QEPW_GEMM_TILE(CA, CB, 64, 64, 2); break;            \
      case 2: QEPW_GEMM_TILE(CA, CB, 32, 128, 1); break;           \
      case 3: QEPW_GEMM_TILE(CA, CB, 64, 128, 2); break;           \
      case 4: QEPW_GEMM_TILE(CA, CB, 128, 64, 2); break;           \
      case 5: QEPW_GEMM_TILE(CA, CB, 128, 32, 4); break;           \
      case 6: QEPW_GEMM_TILE(CA, CB, 32, 64, 1); break;            \
      default: QEPW_GEMM_TILE(CA, CB, 64, 16, 4); break;           \
    }                                                              \
  } while (0)
      if (ca && cb) QEPW_GEMM_LAUNCH(true, true);
      else if (ca) QEPW_GEMM_LAUNCH(true, false);
      else if (cb) QEPW_GEMM_LAUNCH(false, true);
      else QEPW_GEMM_LAUNCH(false, false);
#undef QEPW_GEMM_LAUNCH
#undef QEPW_GEMM_TILE
      if (sp.splits > 1)
        hipLaunchKernelGGL(k_reduce_splits<T>, dim3((unsigned)((mm * nn + 63) / 64)), dim3(256),
                           0, stream, mm, nn, (int)sp.splits, part, pc, ldc, ar, ai, br, bi);
    }
  return hipGetLastError() == hipSuccess ? QEPW_OK : QEPW_ERR_HIP;
}

int gemm(int precision, int op, int64_t m, int64_t n, int64_t k, const double* alpha,
         const void* a, int64_t lda, const void* b, int64_t ldb, const double* beta,
         void* c, int64_t ldc, void* ws, size_t ws_bytes, hipStream_t stream) {
  if (m < 0 || n < 0 || k < 0) return QEPW_ERR_ARG;
  if (op & ~(QEPW_OP_C | QEPW_OP_BC)) return QEPW_ERR_ARG;
  if (m == 0 || n == 0) return QEPW_OK;
  const bool ca = (op & QEPW_OP_C) != 0, cb = (op & QEPW_OP_BC) != 0;
  if (ldc < m || ldb < (cb ? n : (k > 0 ? k : 1))) return QEPW_ERR_ARG;
  if (!ca ? lda < m : lda < (k > 0 ? k : 1)) return QEPW_ERR_ARG;
  if (precision == QEPW_C128)
    return gemm_t<double>(op, m, n, k, alpha, a, lda, b, ldb, beta, c, ldc, ws, ws_bytes,
                          stream);
  if (precision == QEPW_C64)
    return gemm_t<float>(op, m, n, k, alpha, a, lda, b, ldb, beta, c, ldc, ws, ws_bytes,
                         stream);
  return QEPW_ERR_ARG;
}

}  // namespace qepw
