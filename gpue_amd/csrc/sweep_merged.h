// sweep_merged.h -- one launch over problems of different sizes (batches).
//
// A batch of uneven 2D problems spends its time in the chain of small launches of each
// size, not in their work: per step 4 sweeps of 5-11 us a size, where the work of
// sixteen FP32 problems of 128^2-512^2 would keep the VALUs busy for 23 us in all.  Here
// a workgroup of 256 lanes takes 256 / WG blocks of ONE problem's sweep, with the plan,
// tile width and blocks that a launch of that problem alone has for small grids (wide
// enough for 512 points; the same arithmetic, bit for bit), and looks up which in a map
// the host lays out once: every problem's blocks fill the chip together, and a step of
// the whole batch is four launches.
// Measured on those sixteen problems (imaginary time, us a step): launches per size on
// four streams 110 in FP32 and 138 in FP64, merged 65 and 82; three of 512^2 alone 53
// and 69, now 37 and 54.  Equal shapes gain too, by shape / merged: sixteen 128^2 FP64 with
// rotation 27.7 / 27.3, sixteen 256^2 FP32 57 / 38, thirty-two 512^2 FP64 372 / 260, thirty-two
// 64^3 FP32 164 / 127; not FP64 boxes (merge_pays).  A merged sweep takes 13-20 us, in which its waves wait half
// of their life for memory and exchanges.
#pragma once
#include "sweep_launch.h"

namespace gpue {

// One workgroup's share: instance, first block, axis length, blocks of the instance.
struct MergeMap {
  int inst, block, n, nblk;
};

constexpr int MERGE_WG = 256;
// lengths with merged kernels; variants: narrow lines, twiddles up front, quarter tiles
#define GPUE_MERGE_LENGTHS(X) X(64) X(96) X(128) X(192) X(256) X(384) X(512)
constexpr int MERGE_ROW = 3, MERGE_COL = 5;
constexpr int MERGE_TILES = 4;   // quarter tiles of a default one (ColCfg::G)
// Twiddles are read pass by pass, unlike in the lone kernels: all of them up front cost
// registers that these kernels, with every length in one, need for waves (FP64: 121
// instead of 89 us a step on the sixteen problems).
constexpr bool MERGE_TW = false;

template <typename T, int N, int MODE>
__device__ __forceinline__ void row_part(const SweepArgs& a, const MergeMap& e, char* smem, double* sh) {
  using C = RowCfg<N, MERGE_ROW>;
  static_assert(C::WG <= MERGE_WG && C::WG % 64 == 0, "a part is whole waves");
  const int sub = threadIdx.x / C::WG, tx = threadIdx.x % C::WG;
  row_body<T, N, MERGE_ROW, MODE, C::WG == 64, MERGE_TW>(a, e.block + sub, e.nblk, tx, (cx<T>*)smem + sub * C::LDS, sh + sub * 16);
}
template <typename T, int N, int MODE>
__device__ __forceinline__ void col_part(const SweepArgs& a, const MergeMap& e, char* smem, double* sh) {
  using C = ColCfg<T, N, MERGE_COL>;
  static_assert(C::WG <= MERGE_WG && C::WG % 64 == 0 && C::G == MERGE_TILES, "a part is whole waves");
  const int sub = threadIdx.x / C::WG, tx = threadIdx.x % C::WG;
  col_body<T, N, MERGE_COL, MODE, C::WG == 64, MERGE_TW>(a, e.block + sub, e.nblk, tx, (cx<T>*)smem + sub * C::LDS, sh + sub * 16);
}

// Every lane of a workgroup has the same map entry, so the branches here are uniform
// and the parts reach the same barriers.
template <typename T, int MODE>
__global__ void __launch_bounds__(MERGE_WG) row_merged(const SweepArgs* __restrict__ args, const MergeMap* __restrict__ map) {
  extern __shared__ __align__(16) char smem[];
  __shared__ double sh[64];
  const MergeMap e = map[blockIdx.x];
  if (e.inst < 0) return;
  const SweepArgs& a = args[e.inst];
  if (!a.active) return;
  switch (e.n) {
#define GPUE_X(N_) \
  case N_: row_part<T, N_, MODE>(a, e, smem, sh); break;
    GPUE_MERGE_LENGTHS(GPUE_X)
#undef GPUE_X
  }
}
template <typename T, int MODE>
__global__ void __launch_bounds__(MERGE_WG) col_merged(const SweepArgs* __restrict__ args, const MergeMap* __restrict__ map) {
  extern __shared__ __align__(16) char smem[];
  __shared__ double sh[64];
  const MergeMap e = map[blockIdx.x];
  if (e.inst < 0) return;
  const SweepArgs& a = args[e.inst];
  if (!a.active) return;
  switch (e.n) {
#define GPUE_X(N_) \
  case N_: col_part<T, N_, MODE>(a, e, smem, sh); break;
    GPUE_MERGE_LENGTHS(GPUE_X)
#undef GPUE_X
  }
}

// Lanes of one block and LDS bytes of a workgroup for a length; 0 lanes: no kernel.
template <typename T>
inline int merged_row_shape(int n, int* lds) {
  switch (n) {
#define GPUE_X(N_)                                                                             \
  case N_:                                                                                     \
    *lds = MERGE_WG / RowCfg<N_, MERGE_ROW>::WG * RowCfg<N_, MERGE_ROW>::LDS * (int)sizeof(cx<T>); \
    return RowCfg<N_, MERGE_ROW>::WG;
    GPUE_MERGE_LENGTHS(GPUE_X)
#undef GPUE_X
    default: return 0;
  }
}
template <typename T>
inline int merged_col_shape(int n, int* lds) {
  switch (n) {
#define GPUE_X(N_)                                                                                   \
  case N_:                                                                                           \
    *lds = MERGE_WG / ColCfg<T, N_, MERGE_COL>::WG * ColCfg<T, N_, MERGE_COL>::LDS * (int)sizeof(cx<T>); \
    return ColCfg<T, N_, MERGE_COL>::WG;
    GPUE_MERGE_LENGTHS(GPUE_X)
#undef GPUE_X
    default: return 0;
  }
}

// `m` as row_kernel / col_kernel give it.
template <typename T>
hipError_t launch_row_merged(int m, const SweepArgs* d, const MergeMap* map, int grid, int lds, hipStream_t s) {
#define GPUE_ROW(M_) \
  case (M_): hipLaunchKernelGGL((row_merged<T, (M_)>), dim3(grid), dim3(MERGE_WG), lds, s, d, map); break;
  switch (m) {
    GPUE_ROW(RM_FWD) GPUE_ROW(RM_FWD | 16) GPUE_ROW(RM_INV) GPUE_ROW(RM_INV | 16) GPUE_ROW(RM_INV | 64)
    GPUE_ROW(RM_INV | 16 | 64) GPUE_ROW(RM_GAUGE) GPUE_ROW(RM_GAUGE | 16) GPUE_ROW(RM_K) GPUE_ROW(RM_K | 16)
    default: return hipErrorInvalidValue;
  }
#undef GPUE_ROW
  return hipGetLastError();
}
template <typename T>
hipError_t launch_col_merged(int m, const SweepArgs* d, const MergeMap* map, int grid, int lds, hipStream_t s) {
#define GPUE_COL(M_) \
  case (M_): hipLaunchKernelGGL((col_merged<T, (M_)>), dim3(grid), dim3(MERGE_WG), lds, s, d, map); break;
  switch (m) {
    GPUE_COL(CM_FWD) GPUE_COL(CM_INV) GPUE_COL(CM_K) GPUE_COL(CM_K | 16) GPUE_COL(CM_GAUGE) GPUE_COL(CM_GAUGE | 16)
    GPUE_COL(CM_FWD_V) GPUE_COL(CM_FWD_V | 16) GPUE_COL(CM_INV_VG) GPUE_COL(CM_INV_VG | 16)
    default: return hipErrorInvalidValue;
  }
#undef GPUE_COL
  return hipGetLastError();
}

}  // namespace gpue
