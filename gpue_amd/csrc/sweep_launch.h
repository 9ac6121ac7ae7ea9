// sweep_launch.h -- grid shapes and launchers for the sweep kernels.
#pragma once
#include "sweep_kernels.h"

namespace gpue {

template <int N, int V>
inline int row_blocks(int lines) { return (lines + RowCfg<N, V>::LPW - 1) / RowCfg<N, V>::LPW; }
template <typename T, int N, int CV>
inline int col_blocks(int xDim, int others) {
  return ((xDim + ColCfg<T, N, CV>::TC - 1) / ColCfg<T, N, CV>::TC) * others;
}

// Real-time steps run the kernels whose mode carries bit 16 (sweep_kernels.h),
// closing row sweeps without a gauge operator those with bit 64.
inline int row_kernel(int mode, unsigned flags, int gstate) {
  if (mode == RM_KSUM) return mode;
  if (gstate != 0) mode |= 16;
  const int m = mode & 15;
  if ((m == RM_INV || m == RM_INV_FWD) && !(flags & F_GAUGE_POST)) mode |= 64;
  return mode;
}
inline int col_kernel(int mode, int gstate) { return gstate != 0 && col_phase_mode(mode) ? mode | 16 : mode; }

// One problem; `m` as row_kernel / col_kernel give it.
template <typename T, int N, int V>
hipError_t launch_row_t(int m, const SweepArgs& a, hipStream_t s) {
  dim3 grid(row_blocks<N, V>(a.lines)), block(RowCfg<N, V>::WG);
#define GPUE_ROW(M_) \
  case (M_): hipLaunchKernelGGL((row_sweep<T, N, V, (M_)>), grid, block, 0, s, a); break;
  switch (m) {
    GPUE_ROW(RM_FWD) GPUE_ROW(RM_FWD | 16) GPUE_ROW(RM_INV) GPUE_ROW(RM_INV | 16) GPUE_ROW(RM_INV | 64)
    GPUE_ROW(RM_INV | 16 | 64) GPUE_ROW(RM_GAUGE) GPUE_ROW(RM_GAUGE | 16) GPUE_ROW(RM_FULL) GPUE_ROW(RM_FULL | 16)
    GPUE_ROW(RM_K) GPUE_ROW(RM_K | 16) GPUE_ROW(RM_KSUM) GPUE_ROW(RM_INV_FWD | 16 | 64) GPUE_ROW(RM_GAUGE_FWD | 16)
    default: return hipErrorInvalidValue;
  }
#undef GPUE_ROW
  return hipGetLastError();
}

// 1D: nsteps whole steps of one line in one workgroup.  Twiddles in registers up to 256
// lanes (one wave per SIMD); beyond, two waves share a SIMD's registers.
template <typename T, int N, int V>
hipError_t launch_line_t(const SweepArgs& a, int nsteps, hipStream_t s) {
  constexpr int RV = V + (Plan<N, V>::TPL <= 256 ? 2 : 0);
  dim3 grid(1), block(RowCfg<N, RV>::WG);
  if (a.ph.gstate) hipLaunchKernelGGL((line_steps<T, N, RV, true>), grid, block, 0, s, a, nsteps);
  else hipLaunchKernelGGL((line_steps<T, N, RV, false>), grid, block, 0, s, a, nsteps);
  return hipGetLastError();
}

template <typename T, int N, int V>
hipError_t launch_col_t(int m, const SweepArgs& a, hipStream_t s) {
  const int others = a.axis == 1 ? a.ph.zDim : a.ph.yDim;
  dim3 grid(col_blocks<T, N, V>(a.ph.xDim, others)), block(ColCfg<T, N, V>::WG);
#define GPUE_COL(M_) \
  case (M_): hipLaunchKernelGGL((col_sweep<T, N, V, (M_)>), grid, block, 0, s, a); break;
  switch (m) {
    GPUE_COL(CM_FWD) GPUE_COL(CM_INV) GPUE_COL(CM_KSUM) GPUE_COL(CM_K) GPUE_COL(CM_K | 16) GPUE_COL(CM_GAUGE)
    GPUE_COL(CM_GAUGE | 16) GPUE_COL(CM_FWD_V) GPUE_COL(CM_FWD_V | 16) GPUE_COL(CM_INV_VG) GPUE_COL(CM_INV_VG | 16)
    GPUE_COL(CM_GAUGE_FWD | 16)
    default: return hipErrorInvalidValue;
  }
#undef GPUE_COL
  return hipGetLastError();
}

// Batched: `ninst` problems of one shape, arguments in device memory.
template <typename T, int N, int V>
hipError_t launch_row_b_t(int m, const SweepArgs* d, int ninst, int lines, hipStream_t s) {
  const int bpi = row_blocks<N, V>(lines);
  dim3 grid(bpi * ninst), block(RowCfg<N, V>::WG);
#define GPUE_ROW(M_) \
  case (M_): hipLaunchKernelGGL((row_sweep_b<T, N, V, (M_)>), grid, block, 0, s, d, bpi); break;
  switch (m) {
    GPUE_ROW(RM_FWD) GPUE_ROW(RM_FWD | 16) GPUE_ROW(RM_INV) GPUE_ROW(RM_INV | 16) GPUE_ROW(RM_INV | 64)
    GPUE_ROW(RM_INV | 16 | 64) GPUE_ROW(RM_GAUGE) GPUE_ROW(RM_GAUGE | 16) GPUE_ROW(RM_FULL) GPUE_ROW(RM_FULL | 16)
    GPUE_ROW(RM_K) GPUE_ROW(RM_K | 16)
    default: return hipErrorInvalidValue;
  }
#undef GPUE_ROW
  return hipGetLastError();
}

template <typename T, int N, int V>
hipError_t launch_col_b_t(int m, const SweepArgs* d, int ninst, int xDim, int others, hipStream_t s) {
  const int bpi = col_blocks<T, N, V>(xDim, others);
  dim3 grid(bpi * ninst), block(ColCfg<T, N, V>::WG);
#define GPUE_COL(M_) \
  case (M_): hipLaunchKernelGGL((col_sweep_b<T, N, V, (M_)>), grid, block, 0, s, d, bpi); break;
  switch (m) {
    GPUE_COL(CM_FWD) GPUE_COL(CM_INV) GPUE_COL(CM_K) GPUE_COL(CM_K | 16) GPUE_COL(CM_GAUGE) GPUE_COL(CM_GAUGE | 16)
    GPUE_COL(CM_FWD_V) GPUE_COL(CM_FWD_V | 16) GPUE_COL(CM_INV_VG) GPUE_COL(CM_INV_VG | 16)
    default: return hipErrorInvalidValue;
  }
#undef GPUE_COL
  return hipGetLastError();
}

}  // namespace gpue

// One translation unit per (precision, N, plan) keeps the build parallel; it
// holds the strided sweeps of every tile width (narrow = 0, 1, 2) and the row
// sweeps with per-pass or up-front twiddle loads (narrow = 0 or > 0).
#define GPUE_SWEEP_TU(T_, N_, V_, NAME_)                                                          \
  namespace gpue {                                                                                \
  hipError_t NAME_(bool row, int narrow, int mode, const SweepArgs& a, hipStream_t s) {           \
    if (row) return narrow ? launch_row_t<T_, N_, V_ + 2>(mode, a, s) : launch_row_t<T_, N_, V_>(mode, a, s); \
    if (narrow == 1) return launch_col_t<T_, N_, V_ + 2>(mode, a, s);                             \
    if (narrow == 2) return launch_col_t<T_, N_, V_ + 4>(mode, a, s);                             \
    return launch_col_t<T_, N_, V_>(mode, a, s);                                                  \
  }                                                                                               \
  hipError_t NAME_##_line(const SweepArgs& a, int nsteps, hipStream_t s) {                        \
    return launch_line_t<T_, N_, V_>(a, nsteps, s);                                               \
  }                                                                                               \
  hipError_t NAME_##_b(bool row, int narrow, int mode, const SweepArgs* d, int ninst, int lx,     \
                       int others, hipStream_t s) {                                               \
    if (row)                                                                                      \
      return narrow ? launch_row_b_t<T_, N_, V_ + 2>(mode, d, ninst, lx, s)                       \
                    : launch_row_b_t<T_, N_, V_>(mode, d, ninst, lx, s);                          \
    if (narrow == 1) return launch_col_b_t<T_, N_, V_ + 2>(mode, d, ninst, lx, others, s);        \
    if (narrow == 2) return launch_col_b_t<T_, N_, V_ + 4>(mode, d, ninst, lx, others, s);        \
    return launch_col_b_t<T_, N_, V_>(mode, d, ninst, lx, others, s);                             \
  }                                                                                               \
  }
