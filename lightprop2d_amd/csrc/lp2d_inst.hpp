// Kernel templates, their launchers and the per-size variant lists.  Included by the
// per-precision translation units (lp2d_f32_*.hip, lp2d_f64_*.hip) so the large set
// of instantiations compiles in parallel.
#pragma once
#include <atomic>

#include "lp2d_registry.hpp"

namespace lp2d {

constexpr int ilog2c(int n) { return n <= 1 ? 0 : 1 + ilog2c(n >> 1); }
constexpr int cmin(int a, int b) { return a < b ? a : b; }
constexpr int cmax(int a, int b) { return a > b ? a : b; }
constexpr int floor_pow2(int n) { return n < 2 ? 1 : 2 * floor_pow2(n >> 1); }
constexpr int kLdsBudget = 160 * 1024 - 2048;

// ----------------------------------------------------------------- kernels
// Every pass kernel asks for at least two waves per SIMD: the compiler then budgets at
// most 256 registers per lane (one more and a 256-thread workgroup drops to a single
// wave per SIMD, halving the latency hiding).
#define LP2D_OCC __attribute__((amdgpu_waves_per_eu(2)))
template <typename T, int N, int E, int LINES, bool INV, int PS, bool FEAT>
__global__ __launch_bounds__((N / E) * LINES) LP2D_OCC void k_rows(PassArgs<T> a) {
  __shared__ cx<T> lds[LINES * RowPitch<N, PS, LINES>::value];
  constexpr int TPF = (N + LINES - 1) / LINES;  // row tiles per field
  const int tile = blockIdx.x;
  const int b = tile / TPF;
  const int y0 = (tile - b * TPF) * LINES;
  rows_body<T, N, E, LINES, INV, PS, FEAT>(a, b, y0, cmin(LINES, N - y0), lds, threadIdx.x);
}

// The row pass of one tile per workgroup with its twiddles staged in LDS and each row's
// threads in one wave.
template <typename T, int N, int E, int LINES, bool INV, int PS, bool FEAT, int CL, bool PHO,
          int WPE>
__global__ __launch_bounds__((N / E) * LINES) __attribute__((amdgpu_waves_per_eu(WPE)))
void k_rows_occ(PassArgs<T> a) {
  __shared__ cx<T> lds[LINES * RowPitch<N, PS, LINES>::value];
  __shared__ cx<T> twl[TwlLen<N, E, CL>::value];
  static_assert(N % LINES == 0, "whole tiles");
  constexpr int TPF = N / LINES;
  twl_fill<T, N, E, (N / E) * LINES, 1, CL>(twl, a.tw, threadIdx.x);
  __syncthreads();
  const int tile = blockIdx.x;
  const int b = tile / TPF;
  rows_occ_body<T, N, E, LINES, INV, PS, FEAT, CL, PHO>(a, b, (tile - b * TPF) * LINES, lds, twl,
                                                        threadIdx.x);
}

// The pipelined gradient body when its screen factor is hoisted and the LDS twiddle
// tables fit beside the row tiles.
template <typename T, int N, int E, int LINES, int PS>
struct GradPipe {
  static constexpr bool value =
      LINES * PaddedLen<N, PS>::value * (int)sizeof(cx<T>) +
          TwlLen<N, E>::value * (int)sizeof(cx<T>) <= kLdsBudget;
};

template <typename T, int N, int E, int LINES, int PS, bool HOIST>
__global__ __launch_bounds__((N / E) * LINES) LP2D_OCC void k_rows_grad(PassArgs<T> a, int groups,
                                                                float* partial) {
  constexpr bool PIPE = HOIST && GradPipe<T, N, E, LINES, PS>::value;
  __shared__ cx<T> lds[LINES * PaddedLen<N, PS>::value];
  __shared__ cx<T> twl[PIPE ? TwlLen<N, E>::value : 1];
  constexpr int TPF = (N + LINES - 1) / LINES;
  const int tile = blockIdx.x % TPF, g = blockIdx.x / TPF;
  const int per = (a.batch + groups - 1) / groups;
  const int b0 = g * per, b1 = cmin(a.batch, b0 + per);
  const int y0 = tile * LINES;
  if constexpr (PIPE) {
    twl_fill<T, N, E, (N / E) * LINES>(twl, a.tw, threadIdx.x);
    __syncthreads();
    rows_grad_pipe_body<T, N, E, LINES, PS>(a, b0, b1, y0, cmin(LINES, N - y0),
                                            partial + (long long)g * N * N, lds, twl,
                                            threadIdx.x);
  } else {
    rows_grad_body<T, N, E, LINES, PS, HOIST>(a, b0, b1, y0, cmin(LINES, N - y0),
                                              partial + (long long)g * N * N, lds, threadIdx.x);
  }
}

// Chained-plane row pass: one workgroup per row tile of LINES rows of one field.
// WPE: waves per SIMD the register budget is sized for.
template <typename T, int N, int E, int LINES, int PS, int CL, int WPE>
__global__ __launch_bounds__((N / E) * LINES) __attribute__((amdgpu_waves_per_eu(WPE)))
void k_rows_chain(PassArgs<T> a) {
  __shared__ cx<T> lds[LINES * RowPitch<N, PS, LINES>::value];
  __shared__ cx<T> twl[TwlLen<N, E, CL>::value];
  constexpr int TPF = N / LINES;
  twl_fill<T, N, E, (N / E) * LINES, 1, CL>(twl, a.tw, threadIdx.x);
  __syncthreads();
  const int tile = blockIdx.x;
  const int b = tile / TPF;
  rows_chain_body<T, N, E, LINES, PS, CL>(a, b, (tile - b * TPF) * LINES, lds, twl, threadIdx.x);
}

// Grid: (N/W strips) x fields.
template <typename T, int N, int E, int W, int MODE, int PS, int MIDK>
__global__ __launch_bounds__((N / E) * W) LP2D_OCC void k_cols(PassArgs<T> a) {
  __shared__ cx<T> lds[W * PaddedLen<N, PS>::value];
  constexpr int SPF = N / W;  // column strips per field
  const int g = gridDim.x, i = blockIdx.x;
  // Workgroups go to the 8 XCDs round robin.  Give each XCD a contiguous run of
  // strips so that narrow strips sharing 128-byte lines meet in the same L2.
  const int blk = (g % 8 == 0) ? (i % 8) * (g / 8) + i / 8 : i;
  const int b = blk / SPF;
  cols_body<T, N, E, W, MODE, PS, MIDK>(a, b, (blk - b * SPF) * W, lds, threadIdx.x);
}

// Column strips by occupancy: grid (N/W strips) x (field groups of `per` fields).
template <typename T, int N, int E, int W, int PS, int CL, int MODE, bool MID, bool SPEC, int WPE>
__global__ __launch_bounds__((N / E) * W) __attribute__((amdgpu_waves_per_eu(WPE)))
void k_cols_occ(PassArgs<T> a, int per) {
  __shared__ cx<T> lds[W * PaddedLen<N, PS>::value];
  __shared__ cx<T> twl[TwlLen<N, E, CL>::value];
  constexpr int SPF = N / W;
  const int g = gridDim.x, i = blockIdx.x;
  const int blk = (g % 8 == 0) ? (i % 8) * (g / 8) + i / 8 : i;
  const int grp = blk / SPF;
  const int b0 = grp * per;
  twl_fill<T, N, E, (N / E) * W, 1, CL>(twl, a.tw, threadIdx.x);
  __syncthreads();
  cols_occ_body<T, N, E, W, PS, CL, MODE, MID, SPEC>(
      a, b0, cmin(a.batch, b0 + per), (blk - grp * SPF) * W, lds, twl, threadIdx.x);
}

// Whole field in LDS, pipelined over groups of `per` <= kPipeMaxPer fields.
template <typename T, int N, int E, int PS, bool PHO, bool GRAD>
__global__ __launch_bounds__(N * (N / E)) void k_small_pipe(PassArgs<T> a, int per) {
  __shared__ cx<T> lds[N * SmallPitch<N, PS>::value];
  __shared__ cx<T> twl[TwlLen<N, E>::value];
  __shared__ PipeField pf[kPipeMaxPer];
  constexpr int THREADS = N * (N / E);
  static_assert(THREADS >= kPipeMaxPer, "one thread per staged field");
  const int b0 = blockIdx.x * per;
  const int b1 = cmin(a.batch, b0 + per);
  twl_fill<T, N, E, THREADS>(twl, a.tw, threadIdx.x);
  pipe_stage_fields(a, b0, b1, pf, threadIdx.x);
  __syncthreads();
  small_pipe_body<T, N, E, PS, PHO, GRAD>(a, b0, b1, lds, twl, pf, threadIdx.x);
}

template <typename T, int N, int E, int PS>
__global__ __launch_bounds__(N * (N / E)) void k_small(PassArgs<T> a, int mode) {
  __shared__ cx<T> lds[N * SmallPitch<N, PS>::value];
  small_body<T, N, E, PS>(a, blockIdx.x, mode, lds, threadIdx.x);
}

// ----------------------------------------------------------------- shapes
template <typename T, int N, int E>
struct RowShape {
  static constexpr int TL = N / E;
  static constexpr int PS = cmax(1, ilog2c(E));
  static constexpr int LINES = cmax(1, cmin(N, 256 / TL));
  static constexpr int THREADS = TL * LINES;
  static constexpr int LDS = LINES * RowPitch<N, PS, LINES>::value * (int)sizeof(cx<T>);
};

template <typename T, int N, int E, int WT>
struct ColShape {
  static constexpr int TL = N / E;
  static constexpr int PS = cmax(1, ilog2c(E));
  static constexpr int L = PaddedLen<N, PS>::value;
  static constexpr int W = floor_pow2(
      cmax(1, cmin(cmin(WT, N), cmin(1024 / TL, kLdsBudget / (L * (int)sizeof(cx<T>))))));
  static constexpr int THREADS = TL * W;
  static constexpr int LDS = W * L * (int)sizeof(cx<T>);
};

template <typename T, int N, int EMAX>
struct SmallShape {
  static constexpr int E = cmin(N, EMAX);
  static constexpr int PS = cmax(1, ilog2c(E));
  static constexpr int THREADS = N * (N / E);
  static constexpr int LDS = N * SmallPitch<N, PS>::value * (int)sizeof(cx<T>);
  static constexpr bool OK = THREADS <= 1024 && LDS <= kLdsBudget;
};

// ----------------------------------------------------------------- launchers
// Workgroups of `kernel` resident at once on the current device: measured on first
// use and kept per kernel (every caller computes the same value).
inline int cached_slots(std::atomic<int>& slot, const void* kernel, int threads) {
  int v = slot.load(std::memory_order_relaxed);
  if (v == 0) {
    v = resident_groups(kernel, threads);
    slot.store(v, std::memory_order_relaxed);
  }
  return v;
}

template <typename T, int N, int E, int LINES, int PS>
hipError_t launch_rows(const PassArgs<T>& a, bool inv, hipStream_t s) {
  if ((a.flags & F_TILED) && (LINES % tile_rows(N) != 0 || (N / E) % tile_cols<T>(N) != 0))
    return hipErrorInvalidValue;
  constexpr int threads = (N / E) * LINES;
  constexpr int TPF = (N + LINES - 1) / LINES;
  const unsigned grid = (unsigned)((long long)a.batch * TPF);
  const bool feat = (a.flags & (F_SPATIAL | F_GRAD | F_INTENSITY | F_NO_STORE)) != 0;
  if (inv) {
    if (feat)
      k_rows<T, N, E, LINES, true, PS, true><<<grid, threads, 0, s>>>(a);
    else
      k_rows<T, N, E, LINES, true, PS, false><<<grid, threads, 0, s>>>(a);
  } else {
    if (feat)
      k_rows<T, N, E, LINES, false, PS, true><<<grid, threads, 0, s>>>(a);
    else
      k_rows<T, N, E, LINES, false, PS, false><<<grid, threads, 0, s>>>(a);
  }
  return hipGetLastError();
}

// One tile per workgroup, rows within waves; every feature and the per-field tables.
template <typename T, int N, int E, int LINES, int PS, int CL, int WPE>
hipError_t launch_rows_occ(const PassArgs<T>& a, bool inv, hipStream_t s) {
  if ((a.flags & F_TILED) && (LINES % tile_rows(N) != 0 || (N / E) % tile_cols<T>(N) != 0))
    return hipErrorInvalidValue;
  constexpr int threads = (N / E) * LINES;
  const unsigned grid = (unsigned)((long long)a.batch * (N / LINES));
  const int fl = a.flags & (F_SPATIAL | F_GRAD | F_INTENSITY | F_NO_STORE);
  if (inv) {
    if (fl)
      k_rows_occ<T, N, E, LINES, true, PS, true, CL, false, 2><<<grid, threads, 0, s>>>(a);
    else
      k_rows_occ<T, N, E, LINES, true, PS, false, CL, false, WPE><<<grid, threads, 0, s>>>(a);
  } else if (fl == F_PHASE && a.phase) {
    k_rows_occ<T, N, E, LINES, false, PS, false, CL, true, WPE><<<grid, threads, 0, s>>>(a);
  } else if (fl) {
    k_rows_occ<T, N, E, LINES, false, PS, true, CL, false, 2><<<grid, threads, 0, s>>>(a);
  } else {
    k_rows_occ<T, N, E, LINES, false, PS, false, CL, false, WPE><<<grid, threads, 0, s>>>(a);
  }
  return hipGetLastError();
}

template <typename T, int N, int E, int LINES, int PS, bool HOIST>
hipError_t launch_rows_grad(const PassArgs<T>& a, int groups, float* partial, hipStream_t s) {
  // reading a tiled plane in place needs whole row blocks unless nothing is stored
  const bool in_place = (const void*)a.src == (const void*)a.dst;
  if ((a.flags & F_TILED) &&
      (((LINES % tile_rows(N)) != 0 && !(a.flags & F_NO_STORE) && in_place) ||
       (N / E) % tile_cols<T>(N) != 0))
    return hipErrorInvalidValue;
  constexpr int threads = (N / E) * LINES;
  constexpr int TPF = (N + LINES - 1) / LINES;
  k_rows_grad<T, N, E, LINES, PS, HOIST><<<(unsigned)(TPF * groups), threads, 0, s>>>(a, groups,
                                                                                   partial);
  return hipGetLastError();
}

// The chained-plane passes run on block-tiled planes only.
template <typename T, int N, int E, int LINES, int PS, int CL, int WPE>
hipError_t launch_rows_chain(const PassArgs<T>& a, hipStream_t s) {
  if (!(a.flags & F_TILED) || !a.phase || a.src_tab || a.dst_tab) return hipErrorInvalidValue;
  constexpr int threads = (N / E) * LINES;
  const unsigned grid = (unsigned)((long long)a.batch * (N / LINES));
  k_rows_chain<T, N, E, LINES, PS, CL, WPE><<<grid, threads, 0, s>>>(a);
  return hipGetLastError();
}

// Adjoint chained pass: grid (N/LINES row tiles) x (field groups).
template <typename T, int N, int E, int LINES, int PS, int CL, bool LAST, int WPE>
__global__ __launch_bounds__((N / E) * LINES) __attribute__((amdgpu_waves_per_eu(WPE)))
void k_rows_adj_chain(PassArgs<T> a, int groups, float* partial) {
  __shared__ cx<T> lds[LINES * RowPitch<N, PS, LINES>::value];
  __shared__ cx<T> twl[TwlLen<N, E, CL>::value];
  constexpr int TPF = N / LINES;
  const int tile = blockIdx.x % TPF, g = blockIdx.x / TPF;
  const int per = (a.batch + groups - 1) / groups;
  const int b0 = g * per, b1 = cmin(a.batch, b0 + per);
  twl_fill<T, N, E, (N / E) * LINES, 1, CL>(twl, a.tw, threadIdx.x);
  __syncthreads();
  rows_adj_chain_body<T, N, E, LINES, PS, CL, LAST>(
      a, b0, b1, tile * LINES, partial ? partial + (long long)g * N * N : nullptr, lds, twl,
      threadIdx.x);
}

template <typename T, int N, int E, int LINES, int PS, int CL, bool LAST, int WPE>
hipError_t launch_rows_adj_chain(const PassArgs<T>& a, int groups, float* partial, hipStream_t s) {
  if (!(a.flags & F_TILED) || !a.phase || (partial && !a.u_saved) || a.src_tab || a.dst_tab ||
      groups < 1)
    return hipErrorInvalidValue;
  constexpr int threads = (N / E) * LINES;
  const long long grid = (long long)(N / LINES) * groups;
  k_rows_adj_chain<T, N, E, LINES, PS, CL, LAST, WPE><<<(unsigned)grid, threads, 0, s>>>(
      a, groups, partial);
  return hipGetLastError();
}

template <typename T, int N, int E, int W, int PS>
hipError_t launch_cols(const PassArgs<T>& a, int mode, hipStream_t s) {
  if (a.flags & F_TILED) return hipErrorInvalidValue;  // natural layout only
  constexpr int threads = (N / E) * W;
  constexpr int SPF = N / W;
  const unsigned grid = (unsigned)((long long)a.batch * SPF);
  // spectral stage class: none / transfer function + aperture + store / with masks
  const int midk = (a.flags & (F_SMASK0 | F_SMASK1)) ? 2 : (a.flags & F_MID) ? 1 : 0;
  constexpr int FI = MODE_FWD | MODE_INV;
  switch (mode * 4 + midk) {
    case MODE_FWD * 4 + 0:
      k_cols<T, N, E, W, MODE_FWD, PS, 0><<<grid, threads, 0, s>>>(a);
      break;
    case MODE_INV * 4 + 0:
      k_cols<T, N, E, W, MODE_INV, PS, 0><<<grid, threads, 0, s>>>(a);
      break;
    case MODE_INV * 4 + 1:
      k_cols<T, N, E, W, MODE_INV, PS, 1><<<grid, threads, 0, s>>>(a);
      break;
    case FI * 4 + 0:
    case FI * 4 + 1:
      k_cols<T, N, E, W, FI, PS, 1><<<grid, threads, 0, s>>>(a);
      break;
    case FI * 4 + 2:
      k_cols<T, N, E, W, FI, PS, 2><<<grid, threads, 0, s>>>(a);
      break;
    default:  // forward-only passes with a spectral stage, and inverse ones with masks
      if (mode == MODE_FWD)
        k_cols<T, N, E, W, MODE_FWD, PS, 2><<<grid, threads, 0, s>>>(a);
      else
        k_cols<T, N, E, W, MODE_INV, PS, 2><<<grid, threads, 0, s>>>(a);
      break;
  }
  return hipGetLastError();
}

// Column strips by occupancy for the calls of occ_eligible; anything else runs the plain
// class of the same shape.  Groups of up to GMAX fields share one transfer function where
// the call has one set of optics, sized so that the grid is one resident round; per-field
// tables run one field per workgroup.  (256 MB of fields, groups of one against GMAX:
// 256 points 81 / 70 us, 512 84 / 78, 1024 117 / 89.)
template <typename T, int N, int E, int W, int PS, int CL, int GMAX, int WPE>
hipError_t launch_cols_occ(const PassArgs<T>& a, int mode, hipStream_t s) {
  constexpr int TR = tile_rows(N), TC = tile_cols<T>(N);
  constexpr bool TILE_OK = (N / E) % TR == 0 && (W % TC == 0 || TC % W == 0);
  const bool ok = occ_eligible(a, mode);
  if ((a.flags & F_TILED) && (!ok || !TILE_OK)) return hipErrorInvalidValue;
  constexpr int threads = (N / E) * W;
  constexpr int SPF = N / W;
  constexpr int FI = MODE_FWD | MODE_INV;
  if (ok) {
    int per = 1;
    if constexpr (GMAX > 1) {
      if (a.fopt == nullptr) {
        static std::atomic<int> slot{0};
        const int slots = cached_slots(
            slot, (const void*)&k_cols_occ<T, N, E, W, PS, CL, FI, true, false, WPE>, threads);
        int groups = slots / SPF;
        if (groups < 1) groups = 1;
        if (groups > a.batch) groups = a.batch;
        per = (a.batch + groups - 1) / groups;
        if (per > GMAX) per = GMAX;
      }
    }
    const unsigned grid = (unsigned)((long long)((a.batch + per - 1) / per) * SPF);
    if (a.flags & F_SPEC_OUT)
      k_cols_occ<T, N, E, W, PS, CL, FI, true, true, WPE><<<grid, threads, 0, s>>>(a, per);
    else
      k_cols_occ<T, N, E, W, PS, CL, FI, true, false, WPE><<<grid, threads, 0, s>>>(a, per);
    return hipGetLastError();
  }
  // one direction: a forward pass, or an inverse one without factor or with a transfer
  // function (a pupil alone multiplies nothing, so infinities pass it unchanged: the plain
  // class), one field per workgroup
  const unsigned grid = (unsigned)((long long)a.batch * SPF);
  const int mid = a.flags & F_MID;
  if (mode == MODE_FWD && mid == 0) {
    k_cols_occ<T, N, E, W, PS, CL, MODE_FWD, false, false, WPE><<<grid, threads, 0, s>>>(a, 1);
    return hipGetLastError();
  }
  if (mode == MODE_INV && mid == 0) {
    k_cols_occ<T, N, E, W, PS, CL, MODE_INV, false, false, WPE><<<grid, threads, 0, s>>>(a, 1);
    return hipGetLastError();
  }
  if (mode == MODE_INV && a.evan == EV_PASS && (mid & (F_H | F_SMASK0 | F_SMASK1)) == F_H) {
    if (mid & F_SPEC_OUT)
      k_cols_occ<T, N, E, W, PS, CL, MODE_INV, true, true, WPE><<<grid, threads, 0, s>>>(a, 1);
    else
      k_cols_occ<T, N, E, W, PS, CL, MODE_INV, true, false, WPE><<<grid, threads, 0, s>>>(a, 1);
    return hipGetLastError();
  }
  return launch_cols<T, N, E, W, PS>(a, mode, s);
}

// 1024 points: strips of 8 columns with 32 elements per thread (two transforms in two
// passes each) once they fill the chip (512 resident workgroups), narrower strips of 4
// with 16 elements below that: in place, 1 field 11.6 against 9.2 us, 4 fields 17.4
// against 18.1, 32 fields 89 against 99.
template <typename T, int N, int E, int W, int PS, int CL, int GMAX, int WPE, int E2, int W2,
          int CL2, int WPE2>
hipError_t launch_cols_pick(const PassArgs<T>& a, int mode, hipStream_t s) {
  if ((long long)a.batch * (N / W) < 512)
    return launch_cols_occ<T, N, E2, W2, cmax(1, ilog2c(E2)), CL2, GMAX, WPE2>(a, mode, s);
  return launch_cols_occ<T, N, E, W, PS, CL, GMAX, WPE>(a, mode, s);
}

// Field groups of the pipelined whole-field kernel: one resident round.
template <typename T, int N, int E, int PS, bool PHO, bool GRAD>
hipError_t launch_small_pipe(const PassArgs<T>& a, hipStream_t s) {
  constexpr int threads = N * (N / E);
  static std::atomic<int> slot{0};
  const int slots =
      cached_slots(slot, (const void*)&k_small_pipe<T, N, E, PS, PHO, GRAD>, threads);
  int groups = slots < a.batch ? slots : a.batch;
  if (groups < 1) groups = 1;
  int per = (a.batch + groups - 1) / groups;
  if (per > kPipeMaxPer) per = kPipeMaxPer;
  groups = (a.batch + per - 1) / per;
  k_small_pipe<T, N, E, PS, PHO, GRAD><<<(unsigned)groups, threads, 0, s>>>(a, per);
  return hipGetLastError();
}

// The fused propagation (transfer function / pupil / scale / spectrum output, with or
// without a phase screen) and its adjoint run the pipelined whole-field kernel; every
// other combination the general one.
template <typename T, int N, int E, int PS>
hipError_t launch_small(const PassArgs<T>& a, int mode, hipStream_t s) {
  constexpr int BASE = F_H | F_APERTURE | F_SCALE | F_SPEC_OUT;
  constexpr int lds = N * SmallPitch<N, PS>::value * (int)sizeof(cx<T>) +
                      TwlLen<N, E>::value * (int)sizeof(cx<T>) +
                      kPipeMaxPer * (int)sizeof(PipeField);
  // (complex128 of 32 points, two waves per field: 4096 fields 39.7 us here, 34.6 in the
  // general kernel; 64 points 74.4 -> 64.4 us for 2048 fields)
  constexpr int NMIN = sizeof(T) == 4 ? 32 : 64;
  if constexpr (N >= NMIN && E == (sizeof(T) == 4 ? 16 : 8) && lds <= kLdsBudget) {
    if (mode == (MODE_FWD | MODE_INV) && a.evan == EV_PASS) {
      const int x = a.flags & ~BASE;
      if (x == 0) return launch_small_pipe<T, N, E, PS, false, false>(a, s);
      if (x == F_PHASE) return launch_small_pipe<T, N, E, PS, true, false>(a, s);
      if ((x == F_GRAD || x == (F_GRAD | F_NO_STORE)) && a.lens_rev == 0.0)
        return launch_small_pipe<T, N, E, PS, false, true>(a, s);
    }
  }
  k_small<T, N, E, PS><<<(unsigned)a.batch, N * (N / E), 0, s>>>(a, mode);
  return hipGetLastError();
}

// ----------------------------------------------------------------- registration
template <typename T, int N, int E>
void add_row(Registry<T>& r) {
  using S = RowShape<T, N, E>;
  constexpr int lg = ilog2c(N);
  int& k = r.nrows[lg];
  if (k >= kMaxVariants) return;
  // (taller gradient tiles measured slower: 8 rows, for reading a block-tiled plane in
  // place, because a 1024-thread workgroup per CU stalls the CU at every exchange
  // barrier; 4 rows at 1024 (512 threads), reading the adjoint's workspace in 256-byte
  // pieces, by 5% on the gradient pass)
  // (at 4096 points, 2-row gradient tiles over the 2 x 4 block-tiled workspace, 1024
  // threads, measured 1156 us against 749 us for one row per workgroup)
  r.rows[lg][k++] = RowVar<T>{&launch_rows<T, N, E, S::LINES, S::PS>,
                              &launch_rows_grad<T, N, E, S::LINES, S::PS, (E <= 8)>, E,
                              S::LINES, S::THREADS, S::LDS, S::LINES, 0};
}

// One tile per workgroup, rows within waves (kind bit 3): LINES rows of N points.
template <typename T, int N, int E, int LINES, int CL, int WPE>
void add_row_occ(Registry<T>& r) {
  constexpr int PS = cmax(1, ilog2c(E));
  constexpr int lg = ilog2c(N);
  int& k = r.nrows[lg];
  if (k >= kMaxVariants) return;
  constexpr int lds = (LINES * RowPitch<N, PS, LINES>::value + TwlLen<N, E, CL>::value) *
                      (int)sizeof(cx<T>);
  static_assert(lds <= kLdsBudget, "LDS");
  r.rows[lg][k++] = RowVar<T>{&launch_rows_occ<T, N, E, LINES, PS, CL, WPE>, nullptr, E, LINES,
                              (N / E) * LINES, lds, LINES, 8};
}

template <typename T, int N, int E, int WT>
void add_col(Registry<T>& r) {
  using S = ColShape<T, N, E, WT>;
  constexpr int lg = ilog2c(N);
  int& k = r.ncols[lg];
  if (k >= kMaxVariants) return;
  r.cols[lg][k++] = ColVar<T>{&launch_cols<T, N, E, S::W, S::PS>, E, S::W, S::THREADS,
                              S::LDS, 0};
}

template <typename T, int N, int E, int W, int CL, int GMAX, int WPE>
void add_col_occ(Registry<T>& r) {
  constexpr int PS = cmax(1, ilog2c(E));
  constexpr int lg = ilog2c(N);
  int& k = r.ncols[lg];
  if (k >= kMaxVariants) return;
  constexpr int lds = (W * PaddedLen<N, PS>::value + TwlLen<N, E, CL>::value) *
                      (int)sizeof(cx<T>);
  static_assert(lds <= kLdsBudget, "LDS");
  r.cols[lg][k++] = ColVar<T>{&launch_cols_occ<T, N, E, W, PS, CL, GMAX, WPE>, E, W,
                              (N / E) * W, lds, 9};
}

template <typename T, int N, int E, int LINES, int CL, int WPE>
void add_chain(Registry<T>& r) {
  constexpr int PS = cmax(1, ilog2c(E));
  constexpr int lg = ilog2c(N);
  const int k = r.nchain[lg]++;
  r.chain[lg][k] = &launch_rows_chain<T, N, E, LINES, PS, CL, WPE>;
  r.chain_E[lg][k] = E;
  r.chain_lines[lg][k] = LINES;
}

template <typename T, int N, int E, int LINES, int CL, int WPE>
void set_adj_chain(Registry<T>& r) {
  constexpr int PS = cmax(1, ilog2c(E));
  constexpr int lg = ilog2c(N);
  r.adj_chain[lg][0] = &launch_rows_adj_chain<T, N, E, LINES, PS, CL, false, WPE>;
  r.adj_chain[lg][1] = &launch_rows_adj_chain<T, N, E, LINES, PS, CL, true, WPE>;
  r.adj_threads[lg] = (N / E) * LINES;
  r.adj_lines[lg] = LINES;
}

template <typename T, int N>
void register_n(Registry<T>& r) {
  constexpr int lg = ilog2c(N);
  constexpr bool F32 = sizeof(T) == 4;
  constexpr int EMAX = F32 ? 16 : 8;
  constexpr int E0 = cmin(N, EMAX);
  constexpr int E1 = cmin(N, EMAX / 2);
  constexpr int WT = F32 ? 16 : 8;  // 128-byte row segments
  r.nrows[lg] = 0;
  r.ncols[lg] = 0;
  // the default schedules (measured: see the bodies), then the plain ones
  if constexpr (F32 && N == 256) {
    add_row_occ<T, N, 8, 8, 0, 4>(r);
    add_col_occ<T, N, 8, 8, 0, 4, 6>(r);
    add_col_occ<T, N, 16, 8, 0, 4, 4>(r);
  } else if constexpr (F32 && N == 512) {
    add_row_occ<T, N, 8, 4, 0, 4>(r);
    add_row_occ<T, N, 16, 8, 0, 3>(r);
    add_col_occ<T, N, 8, 8, 0, 4, 6>(r);
  } else if constexpr (F32 && N == 1024) {
    // (the quarter table leaves room for four workgroups per CU instead of three with the
    // full one: 4 fields, one round of 1024 workgroups, 50.4 -> 44.6 us; 32 fields 262 ->
    // 260)
    add_row_occ<T, N, 16, 4, 4, 4>(r);
    add_row_occ<T, N, 32, 8, 0, 2>(r);
    add_col_occ<T, N, 32, 8, 0, 8, 2>(r);
    r.cols[lg][0].fn = &launch_cols_pick<T, N, 32, 8, 5, 0, 8, 2, 16, 4, 4, 3>;
    add_col_occ<T, N, 16, 4, 4, 8, 3>(r);
  } else if constexpr (F32 && N == 2048) {
    add_row_occ<T, N, 16, 2, 3, 4>(r);
    add_col_occ<T, N, 32, 4, 4, 4, 2>(r);
  } else if constexpr (F32 && N == 4096) {
    // (the columns with the split tables: 10 spilled registers, 205 us for 2 fields
    // against 152)
    add_row_occ<T, N, 32, 2, 2, 2>(r);
    add_col_occ<T, N, 32, 4, 1, 4, 2>(r);
  }
  // complex128, a propagation with the plain passes and these: 512 fields of 128 points
  // 141 -> 128 us, 64 of 256 84 -> 74, 16 of 512 91 -> 76, 5 of 1024 119 -> 100, 2 of
  // 2048 210 -> 161.  At 4096
  // points a row of 2-row tiles takes a CU's whole LDS (133-158 us against 109 of the
  // plain pass with 16 elements per thread), so the plane stays row-major and only the
  // columns change: 479 -> 430.
  if constexpr (!F32 && N == 256) {
    add_row_occ<T, N, 8, 4, 0, 3>(r);
    add_col_occ<T, N, 8, 4, 0, 4, 3>(r);
  } else if constexpr (!F32 && N == 512) {
    add_row_occ<T, N, 8, 2, 0, 3>(r);
    add_col_occ<T, N, 8, 4, 4, 4, 4>(r);
  } else if constexpr (!F32 && N == 1024) {
    add_row_occ<T, N, 8, 2, 3, 4>(r);
    add_col_occ<T, N, 16, 4, 4, 4, 2>(r);
  } else if constexpr (!F32 && N == 2048) {
    add_row_occ<T, N, 16, 2, 3, 2>(r);
    add_col_occ<T, N, 16, 2, 3, 4, 2>(r);
  } else if constexpr (!F32 && N == 4096) {
    add_row<T, N, 16>(r);
    add_col_occ<T, N, 32, 2, 3, 4, 1>(r);
  } else if constexpr (!F32 && N == 128) {
    add_row_occ<T, N, 8, 4, 0, 3>(r);
    add_col_occ<T, N, 8, 4, 0, 4, 3>(r);
  }
  add_row<T, N, E0>(r);
  add_col<T, N, E0, WT>(r);
  if constexpr (E1 != E0 && N >= 16) {
    add_row<T, N, E1>(r);
    add_col<T, N, E1, WT>(r);
  }
  if constexpr (N >= 256) {
    add_col<T, N, E0, WT / 2>(r);
    if constexpr (!F32) {
      if constexpr (N != 4096) add_row<T, N, 16>(r);
      add_col<T, N, 16, 8>(r);
    }
  }
  // chained-plane row passes of the stack (the first is the default; the other, forward
  // with 5 screens: 128 x 256^2 310 / 309 us and 8 x 256^2 68 / 72, 64 x 512^2 545 / 565,
  // 32 x 1024^2 1055 / 1116, 8 x 2048^2 1432 / 1530, 8 x 4096^2 6329 / 6339, 4096^2 862 /
  // 890) and its adjoint, where 16 elements per thread leave room for the group's
  // gradient sums
  r.nchain[lg] = 0;
  r.adj_chain[lg][0] = r.adj_chain[lg][1] = nullptr;
  r.adj_threads[lg] = r.adj_lines[lg] = 0;
  if constexpr (F32 && N == 256) {
    add_chain<T, N, 8, 8, 0, 4>(r);
    add_chain<T, N, 16, 16, 0, 4>(r);
    set_adj_chain<T, N, 16, 16, 0, 4>(r);
  } else if constexpr (F32 && N == 512) {
    add_chain<T, N, 8, 4, 0, 4>(r);
    add_chain<T, N, 16, 8, 4, 4>(r);
    set_adj_chain<T, N, 16, 8, 4, 3>(r);
  } else if constexpr (F32 && N == 1024) {
    add_chain<T, N, 16, 4, 4, 4>(r);
    add_chain<T, N, 32, 8, 0, 2>(r);
    set_adj_chain<T, N, 16, 4, 4, 3>(r);
  } else if constexpr (F32 && N == 2048) {
    add_chain<T, N, 16, 2, 3, 4>(r);
    add_chain<T, N, 32, 4, 4, 2>(r);
    set_adj_chain<T, N, 16, 2, 3, 3>(r);
  } else if constexpr (F32 && N == 4096) {
    add_chain<T, N, 16, 2, 3, 4>(r);
    add_chain<T, N, 32, 2, 2, 2>(r);
    set_adj_chain<T, N, 16, 2, 3, 4>(r);
  }
  using SS = SmallShape<T, N, EMAX>;
  if constexpr (SS::OK) {
    r.small[lg] = SmallVar<T>{&launch_small<T, N, SS::E, SS::PS>, SS::E, SS::THREADS, SS::LDS};
    r.has_small[lg] = true;
  } else {
    r.has_small[lg] = false;
  }
}

}  // namespace lp2d
