// Fused gate stages on the matrix cores: descriptors shared by the planner
// (program.hip), the table build (gates.hip) and the kernels (mstage_impl.h).
#pragma once

#include "common.h"

namespace sfamd {

constexpr int kMstMaxK = 6;        // local modes per tile
constexpr int kMstMaxD = 20;       // cutoffs with compiled kernels: 2..20
constexpr int kMstMaxGates = 40;   // gates per stage (kernel-argument space, 4 KB)
constexpr int kMstMaxModes = 24;   // modes outside the tile
// tile of K >= 4 local modes: at most this many amplitudes (K = 3 takes every cutoff)
constexpr int kMstMaxTile = 4096;

constexpr int64_t kMstLds = 160 * 1024;      // LDS per compute unit (gfx950)
constexpr int64_t kMstLdsMax = kMstLds - 1024;
constexpr int kMstMaxLgt = 2;                // at most 2^kMstMaxLgt tiles per workgroup

// LDS strides of a tile's axes, in amplitudes: every stride is odd, so the 16
// columns of a matrix-core operand, one stride apart on any axis, fall into
// different LDS banks.
__host__ __device__ constexpr int mst_stride(int D, int K, int axis) {
  int s = 1;
  for (int t = K - 1; t > axis; --t) s = (s * D) | 1;
  return s;
}
// LDS amplitudes of one tile (a whole number of 16-byte units in complex64)
__host__ __device__ constexpr int mst_tile_lds(int D, int K) { return (mst_stride(D, K, 0) * D + 1) & ~1; }
__host__ __device__ constexpr int mst_tile(int D, int K) {
  int s = 1;
  for (int t = 0; t < K; ++t) s *= D;
  return s;
}

// Matrix-core image of one operator of size D (mstage_impl.h): amplitudes per
// lane group, 16-row blocks and complex entries.
__host__ __device__ constexpr int mst_p(int D) { return (D + 3) / 4; }
__host__ __device__ constexpr int mst_mb(int D) { return (mst_p(D) + 1) / 2; }
__host__ __device__ constexpr int mst_img(int D) { return mst_p(D) * mst_mb(D) * 32; }
// two-mode gates of a stage: the photon-number sum or (S2) difference is conserved
__host__ __device__ constexpr bool mst_two_mode(int kind) {
  return kind == SFAMD_OP_BEAMSPLITTER || kind == SFAMD_OP_MZGATE || kind == SFAMD_OP_CROSS_KERR ||
         kind == SFAMD_OP_TWO_MODE_SQUEEZE;
}
// operators of a gate: one for a single-mode gate, one per modular
// anti-diagonal (S2: diagonal) of the two modes for a two-mode gate
__host__ __device__ constexpr int mst_nop(int kind, int D) { return mst_two_mode(kind) ? D : 1; }
// Derivative by the second parameter (the first of a gate with one is read as
// zero weights): dG/dp1 = (i / 2) (wa n + wb N) G with the first mode's digit n
// before and N after the gate; both weights in bits 4 to 9 of MGate::two.
constexpr int mst_weights(int kind) {
  const int wa = kind == SFAMD_OP_BEAMSPLITTER || kind == SFAMD_OP_MZGATE ? 2
                 : kind == SFAMD_OP_DISPLACEMENT || kind == SFAMD_OP_TWO_MODE_SQUEEZE ? -2
                 : kind == SFAMD_OP_SQUEEZE ? -1
                                            : 0;
  const int wb = kind == SFAMD_OP_MZGATE ? 0 : -wa;
  return (wa + 2) << 4 | (wb + 2) << 7;
}
// image entries of a gate: forward (G) and adjoint (G^H, then dG/dp0^H); rotation and Kerr gates use their
// table entry
__host__ __device__ constexpr int64_t mst_img_elems(int kind, int D, bool adj) {
  return kind == SFAMD_OP_ROTATION || kind == SFAMD_OP_KERR ? 0 : (int64_t)mst_nop(kind, D) * mst_img(D) * (adj ? 2 : 1);
}

// Work items of a gate in a group of 2^lgt tiles: 16 columns of one operator.
__host__ __device__ constexpr int mst_items(int D, int K, int lgt, bool two) {
  return two ? D * (((mst_tile(D, K) / (D * D) << lgt) + 15) / 16) : ((mst_tile(D, K) / D << lgt) + 15) / 16;
}
// waves per workgroup: one item per wave and gate, up to 8 (16 waves leave the
// registers for one workgroup per compute unit at cutoff 16, so that nothing
// overlaps its loads and stores: 6 modes, cutoff 16, complex64, one gate on
// the last modes: 75 -> 58 us, a device copy of the state 38 us), and at least
// one thread per tile and element of the K - 1 inner axes (the tile walk)
__host__ __device__ constexpr int mst_waves(int D, int K, int lgt) {
  const int i1 = mst_items(D, K, lgt, false), i2 = mst_items(D, K, lgt, true), it = i1 > i2 ? i1 : i2;
  int w = 4;
  while (w < it && w < 8) w *= 2;
  while (64 * w < (mst_tile(D, K) / D << lgt) && w < 16) w *= 2;
  return w;
}
// Do the registers of the adjoint kernel let two workgroups share a compute
// unit (8 waves each: 128 vector registers per lane)?  At cutoffs 9 to 12 in
// complex64 the compiler is held to that (131 without: 6 modes, cutoff 9,
// forward and adjoint 991 -> 842 us); complex128 needs 205 there, complex64 172
// and more from cutoff 13 on.
__host__ __device__ constexpr bool mst_two_groups(int D, int dtype) {
  return D <= 8 || (D <= 12 && dtype == SFAMD_C64);
}
// kernels exist for groups of 2^lgt tiles up to 1024 inner elements
__host__ __device__ constexpr bool mst_group_ok(int D, int K, int lgt) {
  return lgt <= kMstMaxLgt && (mst_tile(D, K) / D << lgt) <= 1024 && (lgt == 0 || mst_tile(D, K) << lgt <= 16384);
}
// groups that fill the 16 columns of a two-mode gate's operand; larger ones (for longer
// runs of the store, program.hip: order_stages) are forward only
__host__ __device__ constexpr bool mst_group_fills(int D, int K, int lgt) {
  return mst_group_ok(D, K, lgt) && (lgt == 0 || (mst_tile(D, K) / (D * D) << (lgt - 1)) <= 8);
}

// One gate, 64 bytes.  Every field is 32 bits wide: with narrower ones the
// compiler walked the list through a base pointer one byte past a dword, and
// scalar loads drop the two low bits of their base.
struct MGate {
  int32_t kind;
  int32_t a0;         // rotation / Kerr: local axis of the mode (0 = slowest); two modes: -1 if their photon-number
                      // difference is conserved, 0 if the sum is
  int32_t ds, wrap;   // LDS step from amplitude k to k + 1, and what is added where the second digit wraps
  int32_t l1;         // LDS stride of the second axis (0: one mode)
  int32_t cs[kMstMaxK - 1];  // LDS strides of the other local axes, slowest first
  int32_t op;         // program operation index (gradient slot)
  int32_t fwd, adj;   // table offsets of the images (rotation / Kerr: fwd = index of its phases in LDS)
  int32_t nfwd, padj; // the next gate's forward and the previous gate's adjoint image (gates with operators)
  int32_t two;        // bit 0: this gate has two modes, bit 1: the next one, bit 2: the previous one; and mst_weights
};

// The fields every workgroup reads first come first.
struct MArgs {
  int32_t ngates;
  int32_t nheavy;  // gates with operators
  int32_t ndiag;   // rotation and Kerr gates
  int32_t ntiles;  // D^nnl
  int32_t grid;    // workgroups of the launch (set by the launcher)
  int32_t nnl;     // modes outside the tile
  int32_t h0_fwd, h0_two;  // the first gate with operators: its image, whether it has two modes
  int32_t hl_adj, hl_two;  // the last one
  int32_t lgt;     // log2 of the tiles a workgroup holds at once
  int32_t phases;  // table offset of the rotation / Kerr phases, in gate order
  int32_t permuted;  // the output's mode order is not the input's
  int32_t side;      // 1: conjugate gates (column axes of a density matrix), gradients to the second pass
  int64_t loc_stride[kMstMaxK];     // input strides of the local modes, in tile axis order (slowest first)
  int64_t nl_stride[kMstMaxModes];  // input strides of the other modes, fastest first (zeros past nnl)
  // The output's mode order may differ from the input's (forward-only plans):
  // its strides, the local modes slowest first with the LDS strides of their tile axes
  int64_t out_stride[kMstMaxK];
  int32_t out_lds[kMstMaxK];
  int64_t out_nl_stride[kMstMaxModes];
  MGate g[kMstMaxGates];
};

bool mst_supported(int D, int K);
// dynamic LDS bytes of the kernels
int64_t mst_lds_fwd(int D, int K, int lgt, int ndiag, int dtype);
int64_t mst_lds_adj(int D, int K, int lgt, int ndiag, int nheavy, int dtype);
int mst_fwd(int D, int K, const void* in, void* out, const void* table, const MArgs& a, int grid, int dtype,
            hipStream_t s);
int mst_adj(int D, int K, const void* psi, const void* lam_out, void* lam_in, const void* table, const MArgs& a,
            int grid, double* partial, int nwg, int dtype, hipStream_t s);

// per-cutoff launchers (mstage_dNN_MM.hip)
#define SFAMD_MST_FOR_EACH_D(X) \
  X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) X(13) X(14) X(15) X(16) X(17) X(18) X(19) X(20)
#define SFAMD_MST_DECLARE_D(d)                                                                                  \
  int mst_fwd_d##d(int K, const void* in, void* out, const void* table, const MArgs& a, int grid, int dtype,     \
                   hipStream_t s);                                                                              \
  int mst_adj_d##d(int K, const void* psi, const void* lo, void* li, const void* table, const MArgs& a, int grid, \
                   double* partial, int nwg, int dtype, hipStream_t s);
SFAMD_MST_FOR_EACH_D(SFAMD_MST_DECLARE_D)
#undef SFAMD_MST_DECLARE_D

}  // namespace sfamd
