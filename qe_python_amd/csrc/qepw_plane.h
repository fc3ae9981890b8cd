// The xy-plane stage on register "team" FFTs (qepw_regfft.h): one workgroup
// per (z-plane, band), any pair of team lengths n1 (x) and n2 (y) whose rows the
// teams of twelve waves hold (plane_choice).
//
// LDS holds only the nxc occupied x columns of the plane, Q[c * NP2 + y], plus
// one all-zero column:
//   columns : backward y-FFT of every occupied column, its sticks read
//             straight from the stick buffer;
//   rows    : backward x-FFT, times V(r), forward x-FFT, in registers;
//   columns : forward y-FFT, the sticks written straight back.
//
// The backward transforms are decimation-in-frequency team FFTs, whose input
// slot s of lane t is position t + M s: the sphere's x and y extents leave
// whole slots empty for every lane (the extents of a sphere reach about a
// quarter of the grid to either side), so with KEEP naming the occupied slots
// the empty inputs are literal zeros that the compiler folds away (these files
// are built with -fno-signed-zeros for that), and the loads of them disappear.
// The forward transforms are decimation-in-time team FFTs, whose output slot s
// of lane t is again position t + M s: only the kept slots are computed and
// stored.  The row pass chains backward x-FFT (DIF), V(r) multiply and forward
// x-FFT (DIT) in registers -- the DIT consumes the DIF's output order -- at two
// team exchanges per row.
//
// LDS holds the plane and nothing else, so that more workgroups share a CU
// (FP64 at the 72^3 workload: 42 KB, three per CU): a column FFT exchanges
// through its own column (its values are in registers by then), and the row
// pass reads all its rows into registers, after which the plane's storage is
// free and each team exchanges through a line of it; the outputs wait in
// registers until every team is done, then go back to their rows.
#pragma once

#include <algorithm>

#include "qepw_internal.h"
#include "qepw_regfft.h"

namespace qepw {

// Team geometry of a line length.
template <int N> struct PlaneLine {
  static constexpr int L = team_L(N);
  static constexpr int M = N / L;
  static constexpr int per_wave = 64 / M;
  static constexpr unsigned all = (1u << L) - 1u;
  // input slots of the pruned kernels: those within a quarter of the line of
  // either end
  static constexpr int kept = ((N + 3) / 4 + M - 1) / M;
  static constexpr bool prunes = 2 * kept < L;
  static constexpr unsigned pruned =
      prunes ? (((1u << kept) - 1u) | (((1u << kept) - 1u) << (L - kept))) : all;
};

// The twiddles between the two halves of a team FFT, w_N^(t k) for lane t.
// Held in registers (TeamTwiddles), or loaded where they are used from a table
// in the order of the lanes ([k M + t] for the DIF half's k < L, N + [k L + t]
// for the DIT half's k < M) that stays in the L1 (plane_lane_table and, of the
// squares, plane_square_table).
template <typename T, int N, bool LOAD = plane_lane_table(N, sizeof(T) == 8)>
struct PlaneTwiddles {
  TeamTwiddles<T, N> reg;
  __device__ __forceinline__ void load(int t, const cplx<T>* __restrict__ tw) { reg.load(t, tw); }
  __device__ __forceinline__ void fresh() {}
  __device__ __forceinline__ cplx<T> dif(int, int k) const { return reg.w[k]; }
  __device__ __forceinline__ cplx<T> dit(int, int k) const { return reg.w[k]; }
};
template <typename T, int N> struct PlaneTwiddles<T, N, true> {
  const cplx<T>* tab;
  int zero;
  __device__ __forceinline__ void load(int, const cplx<T>* __restrict__ tw) { tab = tw; }
  // keeps the loads after this point after it (an offset, so that they stay
  // global loads)
  __device__ __forceinline__ void fresh() {
    zero = 0;
    asm volatile("" : "+s"(zero));
  }
  __device__ __forceinline__ cplx<T> dif(int t, int k) const {
    return (tab + zero)[k * PlaneLine<N>::M + t];
  }
  __device__ __forceinline__ cplx<T> dit(int t, int k) const {
    return (tab + zero)[N + k * PlaneLine<N>::L + t];
  }
};

template <typename T, int N>
using SquareTwiddles = PlaneTwiddles<T, N, plane_square_table(N, sizeof(T) == 8)>;

// Backward (DIF) and forward (DIT) team FFTs of one line through its LDS line
// S, split as in qepw_regfft.h: b, slots t + M s of lanes t < M; a, slots
// t + L k of lanes t < L.
template <typename T, int N, typename TW>
__device__ __forceinline__ void plane_backward(int t, cplx<T>* S, TW& tw,
                                               cplx<T> (&b)[PlaneLine<N>::L],
                                               cplx<T> (&a)[PlaneLine<N>::M]) {
  constexpr int L = PlaneLine<N>::L, M = PlaneLine<N>::M;
  if (t < M) {
    tw.fresh();
    RegDft<T, L, +1>::run(b);
#pragma unroll
    for (int k = 1; k < L; ++k) b[k] = cmulc(b[k], tw.dif(t, k));
#pragma unroll
    for (int k = 0; k < L; ++k) S[k * M + t] = b[k];
  }
  wave_lds_sync();
  if (t < L) {
#pragma unroll
    for (int j = 0; j < M; ++j) a[j] = S[t * M + j];
    RegDft<T, M, +1>::run(a);
  }
}

template <typename T, int N, typename TW>
__device__ __forceinline__ void plane_forward(int t, cplx<T>* S, TW& tw,
                                              cplx<T> (&a)[PlaneLine<N>::M],
                                              cplx<T> (&b)[PlaneLine<N>::L]) {
  constexpr int L = PlaneLine<N>::L, M = PlaneLine<N>::M;
  if (t < L) {
    tw.fresh();
    RegDft<T, M, -1>::run(a);
#pragma unroll
    for (int k = 1; k < M; ++k) a[k] = cmul(a[k], tw.dit(t, k));
#pragma unroll
    for (int k = 0; k < M; ++k) S[t * M + k] = a[k];
  }
  wave_lds_sync();
  if (t < M) {
#pragma unroll
    for (int j = 0; j < L; ++j) b[j] = S[j * M + t];
    RegDft<T, L, -1>::run(b);
  }
}

// One problem's plane stage.
template <typename T> struct PlaneArgs {
  cplx<T>* work;        // stick buffers (band, z, stick)
  int64_t bstride;
  int nst, n1, n2, nxc;
  const int* colpos;    // (nxc, n2): stick at (column c, y), or -1
  const int* colmap;    // n1: rank of x among the occupied columns, or -1
  const T* V;           // (n3, n2, n1)
  const cplx<T>* tw1;
  const cplx<T>* tw2;
};

template <int N> struct PlaneLane {
  int t, team;
  bool on;
  __device__ __forceinline__ explicit PlaneLane(int tid = threadIdx.x) {
    const int lane = tid & 63, wave = tid >> 6;
    const int i = lane / PlaneLine<N>::M;
    t = lane - i * PlaneLine<N>::M;
    on = i < PlaneLine<N>::per_wave;
    team = wave * PlaneLine<N>::per_wave + i;
  }
};

// Backward y-FFT of every occupied column, in place in LDS: the column is the
// team's exchange line.  Column nxc is zeroed: the row pass reads the
// unoccupied x positions from it (and writes their discarded outputs to it).
template <typename T, int N2, bool PRUNE, bool ZERO = true, typename TW>
__device__ __forceinline__ void plane_cols_backward(const PlaneArgs<T>& g, const cplx<T>* w,
                                                    cplx<T>* Q, int waves, TW& tw,
                                                    int tid = threadIdx.x) {
  using G = PlaneLine<N2>;
  constexpr int L = G::L, M = G::M, NP = N2 + 1;
  constexpr unsigned KEEP = PRUNE ? G::pruned : G::all;
  const PlaneLane<N2> ln(tid);
  const int t = ln.t;
  const cplx<T> zero = mk<T>(T(0), T(0));
  if (ZERO)
    for (int i = tid; i < NP; i += waves * 64) Q[g.nxc * NP + i] = zero;
  if (!ln.on) return;
  for (int c = ln.team; c < g.nxc; c += waves * G::per_wave) {
    cplx<T>* col = Q + c * NP;
    const int* pos = g.colpos + c * N2;
    cplx<T> bb[L], a[M];
    if (t < M) {
      // every position first, then every stick load (from element 0 where
      // the slot holds no stick, replaced by zero): two memory round trips
      // per column instead of two per slot
      int st[L];
#pragma unroll
      for (int s = 0; s < L; ++s) st[s] = ((KEEP >> s) & 1u) ? pos[t + M * s] : -1;
#pragma unroll
      for (int s = 0; s < L; ++s) {
        bb[s] = zero;
        if ((KEEP >> s) & 1u) {
          const cplx<T> v = w[st[s] >= 0 ? st[s] : 0];
          bb[s] = st[s] >= 0 ? v : zero;
        }
      }
    }
    plane_backward<T, N2>(t, col, tw, bb, a);
    wave_lds_sync();
    if (t < L) {
#pragma unroll
      for (int k = 0; k < M; ++k) col[t + L * k] = a[k];
    }
  }
}

// The LDS offsets of this lane's row slots x = t + M s (lanes t < M, kept s),
// which are both the backward inputs and the forward outputs: its column's,
// or the zero column's.  The same for every row of the plane.
template <typename T, int N1, bool PRUNE>
__device__ __forceinline__ void plane_row_slots(const PlaneArgs<T>& g, int np2,
                                                int (&cq)[PlaneLine<N1>::L],
                                                int tid = threadIdx.x) {
  using G = PlaneLine<N1>;
  constexpr unsigned KEEP = PRUNE ? G::pruned : G::all;
  const PlaneLane<N1> ln(tid);
#pragma unroll
  for (int s = 0; s < G::L; ++s) {
    const int c =
        (ln.on && ln.t < G::M && ((KEEP >> s) & 1u)) ? g.colmap[ln.t + G::M * s] : -1;
    cq[s] = (c < 0 ? g.nxc : c) * np2;
  }
}

// Rows, RB per team (RB teams >= n2): backward x-FFT (inputs only at occupied
// columns), V, forward x-FFT (outputs only at occupied columns).  np2: the
// LDS column stride.  Called by the whole workgroup (it synchronises).
template <typename T, int N1, bool PRUNE, int RB, typename TW>
__device__ __forceinline__ void plane_rows(const PlaneArgs<T>& g, int z, cplx<T>* Q, int n2,
                                           int np2, int waves, TW& tw,
                                           const int (&cq)[PlaneLine<N1>::L]) {
  using G = PlaneLine<N1>;
  constexpr int L = G::L, M = G::M, NP = N1 + 1;
  constexpr unsigned KEEP = PRUNE ? G::pruned : G::all;
  const PlaneLane<N1> ln;
  const int t = ln.t, team = ln.team, teams = waves * G::per_wave;
  const cplx<T> zero = mk<T>(T(0), T(0));
  cplx<T>* E = Q + team * NP;
  const T* vz = g.V + (int64_t)z * n2 * N1;
  cplx<T> rows[RB][L];
#pragma unroll
  for (int r = 0; r < RB; ++r) {
    const int y = team + r * teams;
    if (ln.on && y < n2 && t < M) {
#pragma unroll
      for (int s = 0; s < L; ++s) rows[r][s] = ((KEEP >> s) & 1u) ? Q[cq[s] + y] : zero;
    }
  }
  __syncthreads();
  if (ln.on) {
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      const int y = team + r * teams;
      if (y < n2) {
        // V(r) at this lane's backward outputs x = t + L k, fetched first
        T vv[M];
#pragma unroll
        for (int k = 0; k < M; ++k) vv[k] = t < L ? vz[y * N1 + t + L * k] : T(0);
        cplx<T> a[M];
        // consecutive rows reuse the line: a DIF after a DIT writes only
        // the slots the same lane read last
        plane_backward<T, N1>(t, E, tw, rows[r], a);
        if (t < L) {
#pragma unroll
          for (int k = 0; k < M; ++k) a[k] = cscale(a[k], vv[k]);
        }
        plane_forward<T, N1>(t, E, tw, a, rows[r]);
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < RB; ++r) {
    const int y = team + r * teams;
    if (ln.on && y < n2 && t < M) {
#pragma unroll
      for (int s = 0; s < L; ++s)
        if ((KEEP >> s) & 1u) Q[cq[s] + y] = rows[r][s];
    }
  }
}

// Forward y-FFT of every occupied column, in place; only the kept y slots,
// which hold every stick, are computed, and the sticks among them go straight
// to the stick buffer.
template <typename T, int N2, bool PRUNE, typename TW>
__device__ __forceinline__ void plane_cols_forward(const PlaneArgs<T>& g, cplx<T>* w, cplx<T>* Q,
                                                   int waves, TW& tw) {
  using G = PlaneLine<N2>;
  constexpr int L = G::L, M = G::M, NP = N2 + 1;
  constexpr unsigned KEEP = PRUNE ? G::pruned : G::all;
  const PlaneLane<N2> ln;
  if (!ln.on) return;
  const int t = ln.t;
  for (int c = ln.team; c < g.nxc; c += waves * G::per_wave) {
    cplx<T>* col = Q + c * NP;
    const int* pos = g.colpos + c * N2;
    cplx<T> a[M], bb[L];
    // the stick positions are fetched before the transform, so that the
    // stores below wait for nothing
    int st[L];
#pragma unroll
    for (int k = 0; k < L; ++k) st[k] = ((KEEP >> k) & 1u) ? pos[t + M * k] : -1;
    if (t < L) {
#pragma unroll
      for (int s = 0; s < M; ++s) a[s] = col[t + L * s];
    }
    wave_lds_sync();
    plane_forward<T, N2>(t, col, tw, a, bb);
    if (t < M) {
      // every position is consumed before the first store: one wait for
      // the loads above, none between the stores (stores count in vmcnt)
#pragma unroll
      for (int k = 0; k < L; ++k)
        if ((KEEP >> k) & 1u) asm volatile("" ::"v"(st[k]));
#pragma unroll
      for (int k = 0; k < L; ++k)
        if (((KEEP >> k) & 1u) && st[k] >= 0) w[st[k]] = bb[k];
    }
  }
}

// Elements of row data a lane may hold across the row pass.
template <typename T> constexpr int plane_row_budget() { return sizeof(T) == 8 ? 16 : 36; }

template <int N, bool PRUNE> constexpr int plane_kept() {
  return PRUNE && PlaneLine<N>::prunes ? 2 * PlaneLine<N>::kept : PlaneLine<N>::L;
}

// Waves of the square N x N kernel's workgroup, measured over 2 .. 12 (FFT phase
// of 128 bands, or as many as 3e8 bytes of sticks hold).  Whole quads of waves
// win (they load the four SIMDs evenly: 72^2 in FP64 takes 292 us with four
// waves, 403 with six): four while several workgroups share a CU (two are up to
// 5% faster below 64^2, and slower for a few bands), twelve where an FP64
// plane's LDS admits one or two per CU and four waves' rows would not fit
// their registers.  24 planes of 128 bands in FP64, four (what the rows need where
// that is more) and twelve, us: 60^2 88 and 114, 72^2 96 and 128, 80^2 155 and 164,
// 75^2 (whose four waves' rows do not fit: eight) 249 and 221, 81^2 (eight) 162 and
// 178, 90^2 190 and 186, 96^2 246 and 215, 128^2 569 and 452; FP32, four and eight,
// 108^2 145 and 143, 120^2 180 and 161.  The kernels of four waves before, with
// exchange lines of their own above 72^2, took: FP64 75^2 1007 us
// (now 732), 80^2 662 (475), 90^2 1029 (797), 100^2 1298 (773), 108^2 1441
// (890), 120^2 1348 (822), 128^2 in the split stage 3323 (1034); FP32 90^2 386
// (322), 108^2 502 (380), 120^2 464 (361), 128^2 2640 (684).
template <typename T, int N, bool PRUNE> constexpr int plane_waves() {
  constexpr int kept = plane_kept<N, PRUNE>();
  constexpr bool fp64 = sizeof(T) == 8;
  int w = fp64 ? (N <= 80 && N != 75 ? 4 : 12) : (N < 120 ? 4 : 8);
  while (w < 16) {
    const int teams = w * PlaneLine<N>::per_wave;
    const int rows = (N + teams - 1) / teams;
    if (rows <= 6 && rows * kept <= plane_row_budget<T>()) break;
    w += w < 4 ? 1 : 4;
  }
  return w;
}

template <typename T, int N, bool PRUNE, int W>
__device__ __forceinline__ void plane_square_body(const PlaneArgs<T>& g, int z, int64_t b) {
  extern __shared__ unsigned char smem_raw[];
  cplx<T>* Q = reinterpret_cast<cplx<T>*>(smem_raw);
  cplx<T>* w = g.work + b * g.bstride + (int64_t)z * g.nst;
  constexpr int teams = W * PlaneLine<N>::per_wave;
  // the per-lane tables of all passes, fetched while the sticks are
  SquareTwiddles<T, N> tw;
  tw.load(PlaneLane<N>().t, g.tw1);
  int cq[PlaneLine<N>::L];
  plane_row_slots<T, N, PRUNE>(g, N + 1, cq);
  plane_cols_backward<T, N, PRUNE>(g, w, Q, W, tw);
  __syncthreads();
  plane_rows<T, N, PRUNE, (N + teams - 1) / teams>(g, z, Q, N, N + 1, W, tw, cq);
  __syncthreads();
  plane_cols_forward<T, N, PRUNE>(g, w, Q, W, tw);
}

template <typename T, int N, bool PRUNE, int W>
__global__ __launch_bounds__(64 * W, W > 12 ? 4 : 3) void k_plane_square(PlaneArgs<T> g) {
  plane_square_body<T, N, PRUNE, W>(g, blockIdx.x, blockIdx.y);
}

// Any two lengths: the passes are chosen at run time (uniform branches).  Two
// kernels: the lengths whose halves need few registers, and all.  Against the
// Stockham plane kernel that served them (128 bands, FP64 / FP32): 48 x 60 x 80
// 1069 / 925 us -> 221 / 127 us, 36 x 40 x 160 1731 / 1551 -> 263 / 190, 72 x 75
// x 90 1751 / 1440 -> 458 / 277, 108 x 120 x 60 3857 / 3192 -> 926 / 386.
constexpr int kPlaneAnyWaves = 12;
// Rows per team of the run-time kernels: with six kept slots three FP64 rows
// spill (90 x 108 x 60, 128 bands: 913 us with three, 685 us with two).  Planes of
// more rows than that on twelve waves' teams (in FP64 n2 > 24 or 36 teams of a wave:
// 120 x 128, 90 x 160, 108 x 128, 100 x 150) are left to the generic and split
// stages, as they were.
template <typename T, int N1> constexpr int plane_any_rows() {
  return sizeof(T) == 8 && plane_kept<N1, true>() > 4 ? 2 : 3;
}
constexpr bool plane_any_small(int n) { return n <= 108 && n / team_L(n) <= 12; }

template <typename T, bool SMALL>
__global__ __launch_bounds__(64 * kPlaneAnyWaves, 3) void k_plane_any(PlaneArgs<T> g) {
  extern __shared__ unsigned char smem_raw[];
  cplx<T>* Q = reinterpret_cast<cplx<T>*>(smem_raw);
  cplx<T>* w = g.work + blockIdx.y * g.bstride + (int64_t)blockIdx.x * g.nst;
  const int waves = blockDim.x >> 6;
  switch (g.n2) {
#define QEPW_PLANE_CASE(NN)                                                               \
  case NN:                                                                                \
    if constexpr (!SMALL || plane_any_small(NN)) {                                        \
      PlaneTwiddles<T, NN> tw;                                                            \
      tw.load(PlaneLane<NN>().t, g.tw2);                                                  \
      plane_cols_backward<T, NN, true>(g, w, Q, waves, tw);                               \
    }                                                                                     \
    break;
    QEPW_TEAM_SIZES(QEPW_PLANE_CASE)
#undef QEPW_PLANE_CASE
    default: break;
  }
  __syncthreads();
  switch (g.n1) {
#define QEPW_PLANE_CASE(NN)                                                               \
  case NN:                                                                                \
    if constexpr (!SMALL || plane_any_small(NN)) {                                        \
      PlaneTwiddles<T, NN> tw;                                                            \
      tw.load(PlaneLane<NN>().t, g.tw1);                                                  \
      int cq[PlaneLine<NN>::L];                                                           \
      plane_row_slots<T, NN, true>(g, g.n2 + 1, cq);                                      \
      plane_rows<T, NN, true, plane_any_rows<T, NN>()>(g, blockIdx.x, Q, g.n2, g.n2 + 1,  \
                                                       waves, tw, cq);                    \
    }                                                                                     \
    break;
    QEPW_TEAM_SIZES(QEPW_PLANE_CASE)
#undef QEPW_PLANE_CASE
    default: break;
  }
  __syncthreads();
  switch (g.n2) {
#define QEPW_PLANE_CASE(NN)                                                               \
  case NN:                                                                                \
    if constexpr (!SMALL || plane_any_small(NN)) {                                        \
      PlaneTwiddles<T, NN> tw;                                                            \
      tw.load(PlaneLane<NN>().t, g.tw2);                                                  \
      plane_cols_forward<T, NN, true>(g, w, Q, waves, tw);                                \
    }                                                                                     \
    break;
    QEPW_TEAM_SIZES(QEPW_PLANE_CASE)
#undef QEPW_PLANE_CASE
    default: break;
  }
}

// ---- one launch for many problems ---------------------------------------------
// The plane stage of up to kMaxFftGroup square problems of one class
// (plane_group_class): workgroups of all problems end to end along x, each finding
// its problem in a prefix table and running the one-problem body of its length.
// A class's lengths have the same waves, pruning and about the same registers: one
// kernel for all, on the most waves that any length needs, took 1.2 - 2.4 times as
// long (FFT phase, us: 24 problems of 36^3 with 16 bands, FP64 318 -> 160, FP32 240
// -> 107; 8 of 72^3 with 32 bands 858 -> 601, 565 -> 335), and one of all lengths and both
// prunings of the same waves 10 - 20% longer in FP32, whose waves it cuts to three a
// SIMD.
template <typename T> struct PlaneGroup {
  int count;
  int start[kMaxFftGroup + 1];
  int n3[kMaxFftGroup];
  PlaneArgs<T> plane[kMaxFftGroup];
};

template <typename T> constexpr bool plane_group_waves() {
  bool ok = true;
  const auto one = [](int w) { return w == 4 || w == 8 || w == 12; };
#define QEPW_PLANE_CASE(NN) \
  ok = ok && one(plane_waves<T, NN, true>()) && one(plane_waves<T, NN, false>());
  QEPW_GROUP_SIZES(QEPW_PLANE_CASE)
#undef QEPW_PLANE_CASE
  return ok;
}

// Whether a length's kernel is of a group kernel's class.
template <typename T, int N, int W, bool PRUNE, int KIND> constexpr bool plane_group_case() {
  return plane_waves<T, N, PRUNE>() == W && plane_group_kind(N, sizeof(T) == 8) == KIND;
}
template <typename T, int W, bool PRUNE, int KIND> constexpr bool plane_group_any() {
  bool any = false;
#define QEPW_PLANE_CASE(NN) any = any || plane_group_case<T, NN, W, PRUNE, KIND>();
  QEPW_GROUP_SIZES(QEPW_PLANE_CASE)
#undef QEPW_PLANE_CASE
  return any;
}

template <typename T, int W, bool PRUNE, int KIND>
__global__ __launch_bounds__(64 * W, sizeof(T) == 4 && PRUNE ? 4 : 3) void k_plane_group(
    const PlaneGroup<T> g) {
  const int p = group_of(g.start, g.count, blockIdx.x);
  const int l = blockIdx.x - g.start[p];
  const int z = l % g.n3[p];
  const int64_t b = l / g.n3[p];
  switch (g.plane[p].n1) {
#define QEPW_PLANE_CASE(NN)                                           \
  case NN:                                                            \
    if constexpr (plane_group_case<T, NN, W, PRUNE, KIND>())          \
      plane_square_body<T, NN, PRUNE, W>(g.plane[p], z, b);           \
    break;
    QEPW_GROUP_SIZES(QEPW_PLANE_CASE)
#undef QEPW_PLANE_CASE
    default: break;
  }
}

// ---- density ----------------------------------------------------------------------
// rho(r) += w_b |psi_b(r)|^2 over the bands of a slice: the backward half of the
// plane stage, with each lane's outputs x = t + L k of its rows accumulated in
// registers over the bands (FP64) and written once to the slice's partial plane.
// Bound by the chain of each band (sticks, two FFT passes, two barriers) at the
// waves that its registers and LDS leave a CU, eight to twelve.  Whole density of
// 128 bands (or as many as 3e8 bytes of sticks hold), against a team kernel for
// squares up to 120 and the Stockham and split stages for all else, in FP64 and
// FP32, us: 36^2 44 / 34 as before, 60^2 145 / 104 -> 140 / 95, 72^2 189 / 122 ->
// 173 / 119, 75^2 498 / 275 -> 397 / 244, 80^2 352 / 162 -> 342 / 152, 90^2 as
// before, 96^2 566 / 290 -> 493 / 268, 120^2 663 / 332 -> 566 / 235, 128^2 1624 /
// 1318 -> 795 / 495, 48 x 60 x 80 816 / 615 -> 188 / 102, 36 x 40 x 160 952 / 770
// -> 272 / 153, 72 x 75 x 90 1707 / 1294 -> 943 / 370, 108 x 120 x 60 1835 / 1547
// -> 1374 / 385.
template <typename T> struct DensityArgs {
  PlaneArgs<T> plane;   // V unused
  int nb, per;          // bands, bands of a slice
  int accumulate;       // add to the partial planes of an earlier chunk of bands
  const double* weights;
  double* partial;      // (slice, n3, n2, n1)
};

// Rows, RB per team, of one band; called by the whole workgroup (it
// synchronises, and leaves the LDS free).  DIRECT: row by row through exchange
// lines of their own behind the columns (Q + own), for planes whose LDS then
// still leaves two workgroups a CU; else as in plane_rows, the rows read first
// and the plane's storage reused.
template <typename T, int N1, bool PRUNE, int RB, bool DIRECT, int A, typename TW>
__device__ __forceinline__ void density_rows(cplx<T>* Q, int own, int n2, int waves, TW& tw,
                                             const int (&cq)[PlaneLine<N1>::L], double wb,
                                             double (&acc)[A], int tid = threadIdx.x) {
  using G = PlaneLine<N1>;
  constexpr int L = G::L, M = G::M, NP = N1 + 1;
  constexpr unsigned KEEP = PRUNE ? G::pruned : G::all;
  static_assert(RB * M <= A, "accumulators");
  const PlaneLane<N1> ln(tid);
  const int t = ln.t, team = ln.team, teams = waves * G::per_wave;
  const cplx<T> zero = mk<T>(T(0), T(0));
  cplx<T>* E = Q + (DIRECT ? own : 0) + team * NP;
  cplx<T> rows[DIRECT ? 1 : RB][L];
  auto read = [&](int r, int y) __attribute__((always_inline)) {
    if (t < M) {
#pragma unroll
      for (int s = 0; s < L; ++s) rows[r][s] = ((KEEP >> s) & 1u) ? Q[cq[s] + y] : zero;
    }
  };
  if constexpr (!DIRECT) {
#pragma unroll
    for (int r = 0; r < RB; ++r)
      if (ln.on && team + r * teams < n2) read(r, team + r * teams);
    __syncthreads();
  }
  if (ln.on) {
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      const int y = team + r * teams;
      if (y < n2) {
        cplx<T> a[M];
        if (DIRECT) read(0, y);
        if (r > 0) wave_lds_sync();  // the line is read across lanes above
        plane_backward<T, N1>(t, E, tw, rows[DIRECT ? 0 : r], a);
        if (t < L) {
#pragma unroll
          for (int k = 0; k < M; ++k)
            acc[r * M + k] =
                fma(wb, fma((double)a[k].x, (double)a[k].x, (double)a[k].y * (double)a[k].y),
                    acc[r * M + k]);
        }
      }
    }
  }
  __syncthreads();
}

template <typename T, int N1, int RB, int A>
__device__ __forceinline__ void density_store(const DensityArgs<T>& d, int z, int slice, int waves,
                                              const double (&acc)[A]) {
  using G = PlaneLine<N1>;
  const PlaneLane<N1> ln;
  const int n2 = d.plane.n2;
  double* out = d.partial + ((int64_t)slice * gridDim.x + z) * n2 * N1;
  if (!ln.on || ln.t >= G::L) return;
#pragma unroll
  for (int r = 0; r < RB; ++r) {
    const int y = ln.team + r * waves * G::per_wave;
    if (y < n2) {
#pragma unroll
      for (int k = 0; k < G::M; ++k) {
        const int i = y * N1 + ln.t + G::L * k;
        out[i] = (d.accumulate ? out[i] : 0.0) + acc[r * G::M + k];
      }
    }
  }
}

// Whether the square kernel's rows have exchange lines of their own, measured
// where the LDS holds them beside the columns: 24 planes of 128 bands, with and
// without, us: FP64 60^2 71 and 87, 72^2 75 and 103, 80^2 101 and 106, 90^2 124 and
// 128, 81^2 86 and 84, 75^2 118 and 122, 100^2 121 and 144 (the last two not taken);
// FP32 40^2 35 and 38, 54^2 47 and 47, 72^2 62 and 68.
template <typename T> constexpr bool density_direct(int n, bool prune) {
  return sizeof(T) == 8 ? n <= 72 || (prune && (n == 80 || n == 81 || n == 90)) : n <= 54;
}

// Waves of the square kernel's workgroup: four up to 72 (24 planes of 128 bands,
// four and eight, us: FP64 27^2 30 and 32, 48^2 46 and 45, 60^2 71 and 63, 72^2 75
// and 68; FP32 36^2 28 and 32, 72^2 68 and 58), then eight where the lines leave one
// workgroup a CU (90^2 124, twelve 442: no room) or twelve (96^2 124, eight 123).
template <typename T, int N, bool PRUNE> constexpr int density_waves() {
  constexpr bool direct = density_direct<T>(N, PRUNE);
  int w = N <= 72 ? 4 : direct || (N <= 80 && N != 75) ? 8 : 12;
  while (w < 16) {
    const int teams = w * PlaneLine<N>::per_wave;
    const int rows = (N + teams - 1) / teams;
    const int held = direct ? 0 : rows * plane_kept<N, PRUNE>();
    if (rows * PlaneLine<N>::M <= 32 && held <= plane_row_budget<T>()) break;
    w += 4;
  }
  return w;
}

// Waves a SIMD that its registers are bounded for: 72^2 in FP64 spills in three
// waves' (128 bands: 234 us with three, 176 with two).
template <typename T, int N, bool PRUNE> constexpr int density_simd_waves() {
  constexpr int W = density_waves<T, N, PRUNE>();
  return W > 12 ? 4 : sizeof(T) == 8 && N >= 60 && density_direct<T>(N, PRUNE) ? 2 : 3;
}

template <typename T, int N, bool PRUNE, int W>
__global__ __launch_bounds__(64 * W, (density_simd_waves<T, N, PRUNE>())) void k_density_square(DensityArgs<T> d) {
  extern __shared__ unsigned char smem_raw[];
  cplx<T>* Q = reinterpret_cast<cplx<T>*>(smem_raw);
  constexpr int teams = W * PlaneLine<N>::per_wave, RB = (N + teams - 1) / teams;
  constexpr int A = RB * PlaneLine<N>::M;
  const PlaneArgs<T>& g = d.plane;
  const int z = blockIdx.x, b0 = blockIdx.y * d.per, b1 = min(d.nb, b0 + d.per);
  SquareTwiddles<T, N> tw;
  tw.load(PlaneLane<N>().t, g.tw1);
  int cq[PlaneLine<N>::L];
  plane_row_slots<T, N, PRUNE>(g, N + 1, cq);
  double acc[A];
#pragma unroll
  for (int k = 0; k < A; ++k) acc[k] = 0.0;
  constexpr bool DIRECT = density_direct<T>(N, PRUNE);
  if (DIRECT)  // nothing overwrites the zero column
    for (int i = threadIdx.x; i <= N; i += W * 64) Q[g.nxc * (N + 1) + i] = mk<T>(T(0), T(0));
  for (int b = b0; b < b1; ++b) {
    const cplx<T>* w = g.work + (int64_t)b * g.bstride + (int64_t)z * g.nst;
    const double wb = d.weights[b];
    plane_cols_backward<T, N, PRUNE, !DIRECT>(g, w, Q, W, tw);
    __syncthreads();
    density_rows<T, N, PRUNE, RB, DIRECT, A>(Q, (g.nxc + 1) * (N + 1), N, W, tw, cq, wb, acc);
  }
  density_store<T, N, RB, A>(d, z, blockIdx.y, W, acc);
}

// Any two lengths, chosen at run time as in k_plane_any; two rows per team.
// Nothing of a length's tables and lane indexes may be held over the band loop
// (the compiler would hold all lengths'): they are derived from an offset that
// it takes to be new in every round.
template <typename T, bool SMALL, bool DIRECT>
__global__ __launch_bounds__(64 * kPlaneAnyWaves, 3) void k_density_any(DensityArgs<T> d) {
  extern __shared__ unsigned char smem_raw[];
  cplx<T>* Q = reinterpret_cast<cplx<T>*>(smem_raw);
  constexpr int RB = 2, A = RB * (SMALL ? 12 : 16);
  const int waves = blockDim.x >> 6;
  const int z = blockIdx.x, b0 = blockIdx.y * d.per, b1 = min(d.nb, b0 + d.per);
  double acc[A];
#pragma unroll
  for (int k = 0; k < A; ++k) acc[k] = 0.0;
  for (int b = b0; b < b1; ++b) {
    int tid = threadIdx.x, zero = 0;
    asm volatile("" : "+v"(tid), "+s"(zero));
    PlaneArgs<T> g = d.plane;
    g.colpos += zero;
    g.colmap += zero;
    g.tw1 += zero;
    g.tw2 += zero;
    const cplx<T>* w = g.work + (int64_t)b * g.bstride + (int64_t)z * g.nst;
    const int own = (g.nxc + 1) * (g.n2 + 1);
    const double wb = d.weights[b];
    switch (g.n2) {
#define QEPW_PLANE_CASE(NN)                                                               \
  case NN:                                                                                \
    if constexpr (!SMALL || plane_any_small(NN)) {                                        \
      PlaneTwiddles<T, NN> tw;                                                            \
      tw.load(PlaneLane<NN>(tid).t, g.tw2);                                               \
      plane_cols_backward<T, NN, true>(g, w, Q, waves, tw, tid);                          \
    }                                                                                     \
    break;
      QEPW_TEAM_SIZES(QEPW_PLANE_CASE)
#undef QEPW_PLANE_CASE
      default: break;
    }
    __syncthreads();
    switch (g.n1) {
#define QEPW_PLANE_CASE(NN)                                                               \
  case NN:                                                                                \
    if constexpr (!SMALL || plane_any_small(NN)) {                                        \
      PlaneTwiddles<T, NN> tw;                                                            \
      tw.load(PlaneLane<NN>(tid).t, g.tw1);                                               \
      int cq[PlaneLine<NN>::L];                                                           \
      plane_row_slots<T, NN, true>(g, g.n2 + 1, cq, tid);                                 \
      density_rows<T, NN, true, RB, DIRECT, A>(Q, own, g.n2, waves, tw, cq, wb, acc,      \
                                               tid);                                      \
    }                                                                                     \
    break;
      QEPW_TEAM_SIZES(QEPW_PLANE_CASE)
#undef QEPW_PLANE_CASE
      default: break;
    }
  }
  const PlaneArgs<T>& g = d.plane;
  switch (g.n1) {
#define QEPW_PLANE_CASE(NN)                                                               \
  case NN:                                                                                \
    if constexpr (!SMALL || plane_any_small(NN))                                          \
      density_store<T, NN, RB, A>(d, z, blockIdx.y, waves, acc);                          \
    break;
    QEPW_TEAM_SIZES(QEPW_PLANE_CASE)
#undef QEPW_PLANE_CASE
    default: break;
  }
}

// ---- host side ------------------------------------------------------------------
template <typename T> const cplx<T>* plane_twiddles(const Plan& p, int axis, bool square);

template <typename T>
static PlaneArgs<T> plane_args(const Plan& p, const StickTables& st, cplx<T>* work,
                               int64_t bstride, const T* V, bool square) {
  PlaneArgs<T> g{};
  g.work = work;
  g.bstride = bstride;
  g.nst = st.nst;
  g.n1 = p.n1;
  g.n2 = p.n2;
  g.nxc = st.nxcols;
  g.colpos = st.d_colpos;
  g.colmap = st.d_colmap;
  g.V = V;
  g.tw1 = plane_twiddles<T>(p, 0, square);
  g.tw2 = plane_twiddles<T>(p, 1, square);
  return g;
}

template <typename T> PlaneChoice plane_choice(const Plan& p, const StickTables& st) {
  PlaneChoice c;
  const bool square = p.n1 == p.n2 && p.n1 <= 128;
  if (!st.d_colpos || !st.d_colmap || !plane_twiddles<T>(p, 0, square) ||
      !plane_twiddles<T>(p, 1, square))
    return c;
  int per1 = 0, per2 = 0, wprune = 0, wfull = 0, any_rows = 0;
  bool prune1 = false, prune2 = false;
#define QEPW_PLANE_N(NN)                                                     \
  if (p.n1 == NN) {                                                          \
    per1 = PlaneLine<NN>::per_wave;                                          \
    any_rows = plane_any_rows<T, NN>();                                      \
    prune1 = (st.xmask & ~PlaneLine<NN>::pruned) == 0u;                      \
    wprune = plane_waves<T, NN, true>();                                     \
    wfull = plane_waves<T, NN, false>();                                     \
  }                                                                          \
  if (p.n2 == NN) {                                                          \
    per2 = PlaneLine<NN>::per_wave;                                          \
    prune2 = (st.ymask & ~PlaneLine<NN>::pruned) == 0u;                      \
  }
  QEPW_TEAM_SIZES(QEPW_PLANE_N)
#undef QEPW_PLANE_N
  if (per1 == 0 || per2 == 0) return c;
  c.prune = prune1 && prune2;
  c.square = square;
  if (c.square) {
    c.waves = c.prune ? wprune : wfull;
  } else if (c.prune) {
    // whole quads of waves where more than two are needed: a workgroup's waves
    // then share the four SIMDs evenly
    for (int w : {2, 4, 8, 12}) {
      if (p.n2 > any_rows * w * per1) continue;
      c.waves = w;
      break;
    }
  }
  c.lds = std::max((size_t)(st.nxcols + 1) * (p.n2 + 1), (size_t)c.waves * per1 * (p.n1 + 1)) *
          sizeof(cplx<T>);
  if (c.lds > (size_t)kMaxLdsBytes) c.waves = 0;
  return c;
}

template <typename T>
bool launch_plane_stage(const Plan& p, const StickTables& st, cplx<T>* work, int64_t bstride,
                        const T* V, int nb, hipStream_t stream) {
  const PlaneChoice& c = sizeof(T) == 8 ? st.plane64 : st.plane32;
  if (c.waves == 0) return false;
  const PlaneArgs<T> g = plane_args<T>(p, st, work, bstride, V, c.square);
  const dim3 grid(p.n3, nb);
#define QEPW_PLANE_LAUNCH(K)                                                            \
  do {                                                                                  \
    allow_lds(reinterpret_cast<const void*>(&K), c.lds);                                \
    hipLaunchKernelGGL(K, grid, dim3(64 * c.waves), c.lds, stream, g);                  \
    return true;                                                                        \
  } while (0)
  if (c.square) {
#define QEPW_PLANE_SQUARE(NN)                                                           \
  if constexpr (NN <= 128) {                                                            \
    if (p.n1 == NN && c.prune)                                                          \
      QEPW_PLANE_LAUNCH((k_plane_square<T, NN, true, plane_waves<T, NN, true>()>));     \
    if (p.n1 == NN)                                                                     \
      QEPW_PLANE_LAUNCH((k_plane_square<T, NN, false, plane_waves<T, NN, false>()>));   \
  }
    QEPW_TEAM_SIZES(QEPW_PLANE_SQUARE)
#undef QEPW_PLANE_SQUARE
    return false;
  }
  if (plane_any_small(p.n1) && plane_any_small(p.n2)) QEPW_PLANE_LAUNCH((k_plane_any<T, true>));
  QEPW_PLANE_LAUNCH((k_plane_any<T, false>));
#undef QEPW_PLANE_LAUNCH
  return false;
}

template <typename T> PlaneChoice density_choice(const Plan& p, const StickTables& st) {
  // the plane stage's, with the waves that the density kernels take
  PlaneChoice c = sizeof(T) == 8 ? st.plane64 : st.plane32;
  if (c.waves == 0) return c;
  int per1 = 0, w = 0, simd = 3;
  bool direct = false;
#define QEPW_PLANE_N(NN)                                                                        \
  if (p.n1 == NN) {                                                                             \
    per1 = PlaneLine<NN>::per_wave;                                                             \
    w = c.prune ? density_waves<T, NN, true>() : density_waves<T, NN, false>();                 \
    direct = density_direct<T>(NN, c.prune);                                                    \
    simd = c.prune ? density_simd_waves<T, NN, true>() : density_simd_waves<T, NN, false>();    \
  }
  QEPW_TEAM_SIZES(QEPW_PLANE_N)
#undef QEPW_PLANE_N
  if (!c.square) {
    w = 0;
    simd = 3;
    direct = true;
    for (int v : {4, 8, 12}) {
      if (p.n2 > 2 * v * per1) continue;
      w = v;
      break;
    }
  }
  c.waves = w;
  const size_t columns = (size_t)(st.nxcols + 1) * (p.n2 + 1), lines = (size_t)w * per1 * (p.n1 + 1);
  c.lds = (direct ? columns + lines : std::max(columns, lines)) * sizeof(cplx<T>);
  if (!c.square && c.lds > (size_t)kMaxLdsBytes) {
    direct = false;
    c.lds = std::max(columns, lines) * sizeof(cplx<T>);
  }
  c.direct = direct;
  if (c.lds > (size_t)kMaxLdsBytes) c.waves = 0;
  if (c.waves > 0)
    c.hold = std::max(1, std::min(4 * simd / c.waves, (int)((size_t)(160 << 10) / c.lds)));
  return c;
}

// Slices of the bands: every slice is a workgroup per plane that takes
// ceil(nb / slices) bands; as many as give the fewest rounds of bands.
static int density_slices(const PlaneChoice& c, int n3, int nb, int most) {
  const int slots = 256 * c.hold;
  int best = 1;
  int64_t cost = INT64_MAX;
  for (int s = 1; s <= most && s <= nb; ++s) {
    const int64_t rounds = ((int64_t)n3 * s + slots - 1) / slots;
    const int64_t t = rounds * ((nb + s - 1) / s);
    if (t < cost) {
      cost = t;
      best = s;
    }
  }
  return best;
}

// The partial density planes of nb bands; *slices of them are written (given
// *slices > 0, that many).  False where the team stage does not serve the plan.
template <typename T>
bool launch_density_stage(const Plan& p, const StickTables& st, cplx<T>* work, int64_t bstride,
                          const double* weights, int nb, int most, int* slices, bool accumulate,
                          double* partial, hipStream_t stream) {
  const PlaneChoice& c = sizeof(T) == 8 ? st.density64 : st.density32;
  if (c.waves == 0) return false;
  if (*slices == 0) *slices = density_slices(c, p.n3, nb, most);
  DensityArgs<T> d{};
  d.plane = plane_args<T>(p, st, work, bstride, nullptr, c.square);
  d.nb = nb;
  d.per = (nb + *slices - 1) / *slices;
  d.accumulate = accumulate ? 1 : 0;
  d.weights = weights;
  d.partial = partial;
  const dim3 grid(p.n3, *slices);
#define QEPW_DENSITY_LAUNCH(K)                                                          \
  do {                                                                                  \
    allow_lds(reinterpret_cast<const void*>(&K), c.lds);                                \
    hipLaunchKernelGGL(K, grid, dim3(64 * c.waves), c.lds, stream, d);                  \
    return true;                                                                        \
  } while (0)
  if (c.square) {
#define QEPW_DENSITY_SQUARE(NN)                                                               \
  if constexpr (NN <= 128) {                                                                  \
    if (p.n1 == NN && c.prune)                                                                \
      QEPW_DENSITY_LAUNCH((k_density_square<T, NN, true, density_waves<T, NN, true>()>));     \
    if (p.n1 == NN)                                                                           \
      QEPW_DENSITY_LAUNCH((k_density_square<T, NN, false, density_waves<T, NN, false>()>));   \
  }
    QEPW_TEAM_SIZES(QEPW_DENSITY_SQUARE)
#undef QEPW_DENSITY_SQUARE
    return false;
  }
  const bool small = plane_any_small(p.n1) && plane_any_small(p.n2);
  if (small && c.direct) QEPW_DENSITY_LAUNCH((k_density_any<T, true, true>));
  if (small) QEPW_DENSITY_LAUNCH((k_density_any<T, true, false>));
  if (c.direct) QEPW_DENSITY_LAUNCH((k_density_any<T, false, true>));
  QEPW_DENSITY_LAUNCH((k_density_any<T, false, false>));
#undef QEPW_DENSITY_LAUNCH
  return false;
}

// The grouped plane stage of ``count`` square problems of one class whose lengths
// are among QEPW_GROUP_SIZES (nb bands each).
template <typename T>
int launch_plane_group(int count, const Plan* const* plans, cplx<T>* const* work,
                       const int64_t* bstride, const T* const* V, const int* nb,
                       hipStream_t stream) {
  static_assert(plane_group_waves<T>(), "waves of the group kernels");
  PlaneGroup<T> g{};
  g.count = count;
  int64_t total = 0;
  size_t lds = 0;
  const auto choice = [](const Plan& p) -> const PlaneChoice& {
    return sizeof(T) == 8 ? p.sphere.plane64 : p.sphere.plane32;
  };
  const int kind = plane_group_class(*plans[0], choice(*plans[0]), sizeof(T) == 8);
  for (int j = 0; j < count; ++j) {
    const Plan& p = *plans[j];
    const PlaneChoice& c = choice(p);
    if (plane_group_class(p, c, sizeof(T) == 8) != kind) return QEPW_ERR_UNSUPPORTED;
    g.start[j] = (int)total;
    g.n3[j] = p.n3;
    g.plane[j] = plane_args<T>(p, p.sphere, work[j], bstride[j], V[j], true);
    total += (int64_t)p.n3 * nb[j];
    lds = std::max(lds, c.lds);
  }
  const PlaneChoice& c = choice(*plans[0]);
  const int length_kind = plane_group_kind(plans[0]->n1, sizeof(T) == 8);
  if (total > plane_group_most(c.waves)) return QEPW_ERR_UNSUPPORTED;
  g.start[count] = (int)total;
#define QEPW_GROUP_KERNEL(W, PRUNE, KIND)                                                      \
  if constexpr (plane_group_any<T, W, PRUNE, KIND>())                                          \
    if (c.waves == W && c.prune == PRUNE && length_kind == KIND) {                             \
      allow_lds(reinterpret_cast<const void*>(&k_plane_group<T, W, PRUNE, KIND>), lds);        \
      hipLaunchKernelGGL((k_plane_group<T, W, PRUNE, KIND>), dim3((unsigned)total),            \
                         dim3(64 * W), lds, stream, g);                                        \
      return QEPW_OK;                                                                          \
    }
#define QEPW_GROUP_KIND(KIND)        \
  QEPW_GROUP_KERNEL(4, true, KIND)   \
  QEPW_GROUP_KERNEL(4, false, KIND)  \
  QEPW_GROUP_KERNEL(8, true, KIND)   \
  QEPW_GROUP_KERNEL(8, false, KIND)  \
  QEPW_GROUP_KERNEL(12, true, KIND)  \
  QEPW_GROUP_KERNEL(12, false, KIND)
  QEPW_GROUP_KIND(0)
  QEPW_GROUP_KIND(60)
  QEPW_GROUP_KIND(72)
  QEPW_GROUP_KIND(80)
  QEPW_GROUP_KIND(96)
#undef QEPW_GROUP_KIND
#undef QEPW_GROUP_KERNEL
  return QEPW_ERR_UNSUPPORTED;
}

}  // namespace qepw
