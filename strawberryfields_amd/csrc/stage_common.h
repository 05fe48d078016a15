// Device helpers shared by the fused-stage kernels: tile walks over a ket,
// digit extraction and wave reductions.
#pragma once

#include "common.h"

namespace {

// One DPP lane move of a double (two 32-bit moves); lanes of rows outside
// RowMask receive 0.
template <int Ctrl, int RowMask>
__device__ __forceinline__ double dpp_move(double v) {
  const unsigned long long u = (unsigned long long)__double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)u, Ctrl, RowMask, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(u >> 32), Ctrl, RowMask, 0xf, false);
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

// Sum over the 64 lanes of a wave by DPP moves, which stay in the VALU instead
// of a round trip through the LDS crossbar per step as shuffles do: swaps
// within pairs and quads, then the half-row and row mirrors leave every lane of
// a 16-lane row with the row's sum; row broadcast 15 adds row 0 into row 1 and
// row 2 into row 3, row broadcast 31 adds rows 0-1 into row 3.  The total is
// valid in lane 63 (the summation order is fixed, so results are
// deterministic).
__device__ __forceinline__ double wave_sum(double v) {
  v += dpp_move<0xB1, 0xF>(v);   // quad_perm [1, 0, 3, 2]
  v += dpp_move<0x4E, 0xF>(v);   // quad_perm [2, 3, 0, 1]
  v += dpp_move<0x141, 0xF>(v);  // row_half_mirror
  v += dpp_move<0x140, 0xF>(v);  // row_mirror
  v += dpp_move<0x142, 0xA>(v);  // row_bcast:15 into rows 1, 3
  v += dpp_move<0x143, 0xC>(v);  // row_bcast:31 into rows 2, 3
  return v;
}
constexpr int kWaveSumLane = 63;

// the same reduction in single precision (complex64 stages: 64 lanes' partial
// products, well inside single precision; the per-wave sums are added in
// double), one DPP add per step
template <int Ctrl, int RowMask>
__device__ __forceinline__ float dpp_move_f(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), Ctrl, RowMask, 0xf, false));
}
__device__ __forceinline__ float wave_sum(float v) {
  v += dpp_move_f<0xB1, 0xF>(v);
  v += dpp_move_f<0x4E, 0xF>(v);
  v += dpp_move_f<0x141, 0xF>(v);
  v += dpp_move_f<0x140, 0xF>(v);
  v += dpp_move_f<0x142, 0xA>(v);
  v += dpp_move_f<0x143, 0xC>(v);
  return v;
}

// x + y after their upper and lower halves (or odd and even rows of 16 lanes) were
// swapped: x's pair sums in the lower half (even rows), y's in the upper (odd rows)
template <bool ROWS>
__device__ __forceinline__ double swap_add(double x, double y) {
  const unsigned long long ux = (unsigned long long)__double_as_longlong(x);
  const unsigned long long uy = (unsigned long long)__double_as_longlong(y);
  const auto lo = ROWS ? __builtin_amdgcn_permlane16_swap((unsigned)ux, (unsigned)uy, false, false)
                       : __builtin_amdgcn_permlane32_swap((unsigned)ux, (unsigned)uy, false, false);
  const auto hi = ROWS ? __builtin_amdgcn_permlane16_swap((unsigned)(ux >> 32), (unsigned)(uy >> 32), false, false)
                       : __builtin_amdgcn_permlane32_swap((unsigned)(ux >> 32), (unsigned)(uy >> 32), false, false);
  return __longlong_as_double((long long)(((unsigned long long)hi[0] << 32) | lo[0])) +
         __longlong_as_double((long long)(((unsigned long long)hi[1] << 32) | lo[1]));
}

// Sums of a and b over the 64 lanes of a wave in one reduction: a's in lane 31, b's in
// lane 63.
__device__ __forceinline__ double wave_sum_pair(double a, double b) {
  double v = swap_add<false>(a, b);
  v += dpp_move<0xB1, 0xF>(v);   // quad_perm [1, 0, 3, 2]
  v += dpp_move<0x4E, 0xF>(v);   // quad_perm [2, 3, 0, 1]
  v += dpp_move<0x141, 0xF>(v);  // row_half_mirror
  v += dpp_move<0x140, 0xF>(v);  // row_mirror
  v += dpp_move<0x142, 0xA>(v);  // row_bcast:15 into rows 1, 3
  return v;
}

// Sums of a, b, c and d over the 64 lanes of a wave in one reduction of six steps, as
// many as one sum takes: every lane of row 0 (lanes 0 to 15) receives a's, of row 1 b's, of
// row 2 c's and of row 3 d's.  The summation order is fixed.
__device__ __forceinline__ double wave_sum_four(double a, double b, double c, double d) {
  double v = swap_add<true>(swap_add<false>(a, c), swap_add<false>(b, d));
  v += dpp_move<0xB1, 0xF>(v);   // quad_perm [1, 0, 3, 2]
  v += dpp_move<0x4E, 0xF>(v);   // quad_perm [2, 3, 0, 1]
  v += dpp_move<0x141, 0xF>(v);  // row_half_mirror
  v += dpp_move<0x140, 0xF>(v);  // row_mirror
  return v;
}

// Workgroups are dealt to the 8 XCDs round-robin (block b runs on XCD b % 8),
// and each XCD has its own L2.  Neighbouring tiles share cache lines whenever
// the innermost non-local mode has a small stride, so the tiles are cut into 8
// contiguous ranges and XCD x's blocks (b = x + 8 k) walk range x; every line
// is then fetched into one L2 instead of eight.
struct TileRange {
  int first, end, step;
};

__device__ __forceinline__ TileRange xcd_tiles(int ntiles, int G) {
  const int b = blockIdx.x;
  if (G % 8) return TileRange{b, ntiles, G};
  const int per = (ntiles + 7) / 8;
  const int x = b % 8;
  const int end = (x + 1) * per < ntiles ? (x + 1) * per : ntiles;
  return TileRange{x * per + b / 8, end, G / 8};
}

// Im(conj(a) b)
template <typename T>
__device__ __forceinline__ T im_conj_mul(cpx<T> a, cpx<T> b) {
  return a.re * b.im - a.im * b.re;
}

}  // namespace
