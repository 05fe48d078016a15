// Matrix-core gate stages: host-side sizes and the dispatch to the per-cutoff
// launchers (the kernels are in mstage_impl.h, instantiated by the
// mstage_dNN_MM.hip translation units).
#include "mstage.h"

namespace sfamd {

bool mst_supported(int D, int K) {
  if (D < 2 || D > kMstMaxD || K < 3 || K > kMstMaxK) return false;
  return K == 3 || ipow(D, K) <= kMstMaxTile;
}

int64_t mst_lds_fwd(int D, int K, int lgt, int ndiag, int dtype) {
  const int64_t esz = dtype == SFAMD_C64 ? 8 : 16;
  return (((int64_t)mst_tile_lds(D, K) << lgt) + (int64_t)((ndiag * D + 1) & ~1)) * esz;
}

int64_t mst_lds_adj(int D, int K, int lgt, int ndiag, int nheavy, int dtype) {
  const int64_t esz = dtype == SFAMD_C64 ? 8 : 16;
  return (((int64_t)(nheavy + 2) * mst_tile_lds(D, K) << lgt) + (int64_t)((ndiag * D + 1) & ~1)) * esz +
         (int64_t)(ndiag + nheavy) * 2 * mst_waves(D, K, lgt) * 8;
}

int mst_fwd(int D, int K, const void* in, void* out, const void* table, const MArgs& a, int grid, int dtype,
            hipStream_t s) {
  switch (D) {
#define CASE_D(d) \
  case d:         \
    return mst_fwd_d##d(K, in, out, table, a, grid, dtype, s);
    SFAMD_MST_FOR_EACH_D(CASE_D)
#undef CASE_D
    default:
      return SFAMD_E_CUTOFF;
  }
}

int mst_adj(int D, int K, const void* psi, const void* lam_out, void* lam_in, const void* table, const MArgs& a,
            int grid, double* partial, int nwg, int dtype, hipStream_t s) {
  switch (D) {
#define CASE_D(d) \
  case d:         \
    return mst_adj_d##d(K, psi, lam_out, lam_in, table, a, grid, partial, nwg, dtype, s);
    SFAMD_MST_FOR_EACH_D(CASE_D)
#undef CASE_D
    default:
      return SFAMD_E_CUTOFF;
  }
}

}  // namespace sfamd
