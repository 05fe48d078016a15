// Recorded-circuit executor and the C ABI entry points of libsfamd.
//
// A program is the list of Fock-backend operations the Engine issued
// (strawberryfields/engine.py:427-430 calls op.apply per command); the host
// loop below issues the kernels of each operation on one stream, keeps the
// state in caller-provided buffers, writes the inputs of requested operations
// as checkpoints and runs the reverse sweep.  The whole sequence can be
// captured into a HIP graph by the caller (sfamd_graph_*).
#include <algorithm>
#include <cstring>
#include <exception>
#include <functional>
#include <memory>
#include <vector>

#include "common.h"
#include "fiber.h"
#include "fused.h"
#include "mfma.h"
#include "mstage.h"
#include "slab.h"

using namespace sfamd;

namespace {

struct OpPlan {
  int kind;
  int m0, m1;
  int mixed_in;   // state at the op input is a DM
  int mix_first;  // loss on a pure state: convert to a DM first
  int64_t off;    // table offset (complex elements)
};

// strides of mode m in a ket of n modes and in a DM of n modes
inline int64_t ket_stride(int n, int D, int m) { return ipow(D, n - 1 - m); }
inline int64_t bra_stride_dm(int n, int D, int m) { return ipow(D, 2 * (n - 1 - m) + 1); }
inline int64_t ket_stride_dm(int n, int D, int m) { return ipow(D, 2 * (n - 1 - m)); }

inline int64_t elem_size(int dtype) { return dtype == SFAMD_C64 ? 8 : 16; }

inline const char* cptr(const void* p, int64_t elems, int dtype) {
  return (const char*)p + elems * elem_size(dtype);
}

bool two_mode_kind(int kind) {
  return kind == SFAMD_OP_BEAMSPLITTER || kind == SFAMD_OP_TWO_MODE_SQUEEZE || kind == SFAMD_OP_MZGATE ||
         kind == SFAMD_OP_CROSS_KERR;
}

int validate_op(int kind, int m0, int m1, int n, int D) {
  if (kind < 0 || kind > SFAMD_OP_CUBIC_PHASE) return SFAMD_E_KIND;
  if (D < 1 || D > SFAMD_MAX_CUTOFF) return SFAMD_E_CUTOFF;
  if (two_mode_kind(kind)) {
    if (D > SFAMD_MAX_CUTOFF_BS) return SFAMD_E_CUTOFF;
    if (m0 < 0 || m0 >= n || m1 < 0 || m1 >= n || m0 == m1) return SFAMD_E_ARG;
  } else if (kind != SFAMD_OP_MIX) {
    if (kind == SFAMD_OP_CUBIC_PHASE && D > SFAMD_MAX_CUTOFF_V) return SFAMD_E_CUTOFF;
    if (m0 < 0 || m0 >= n) return SFAMD_E_ARG;
  }
  return 0;
}

// second-parameter derivative weight of a photon-number-conserving two-mode
// gate: d/dp1 G[N][n] = i (wa n + wb N) G[N][n]
void bs_weights(int kind, int* wa, int* wb) {
  *wa = kind == SFAMD_OP_CROSS_KERR ? 0 : 1;
  *wb = kind == SFAMD_OP_BEAMSPLITTER ? -1 : 0;
}

// Routing between element-wise and per-fiber kernels: per-fiber when a kernel
// is compiled for D and the innermost non-gate run is long enough to coalesce.
bool use_fib(int D, int64_t run) { return fiber_supported(D) && run >= kFiberMinRun; }

// complex64 dense gates run on the matrix cores for every axis stride
int dense_pass(const void* in, void* out, int64_t N, int D, int64_t B, const void* U, int conj, int parity, int dtype,
               hipStream_t s) {
  if (mfma_supported(D, dtype)) return axis_dense_mfma(in, out, N, D, B, U, conj, s);
  if (use_fib(D, B)) return axis_dense_fib(in, out, N, D, B, U, conj, parity, dtype, s);
  return axis_dense(in, out, N, D, B, U, conj, dtype, s);
}

int dense_adj_pass(const void* psi, const void* lo, void* li, int64_t N, int D, int64_t B, const void* U,
                   const void* dU0, const void* dU1, int conj, int parity, double* pb, int nwg, int zp1, int dtype,
                   hipStream_t s) {
  if (mfma_supported(D, dtype)) return axis_dense_adj_mfma(psi, lo, li, N, D, B, U, dU0, dU1, conj, pb, nwg, zp1, s);
  if (use_fib(D, B)) return axis_dense_adj_fib(psi, lo, li, N, D, B, U, dU0, dU1, conj, parity, pb, nwg, zp1, dtype, s);
  return axis_dense_adj(psi, lo, li, N, D, B, U, dU0, dU1, conj, pb, nwg, zp1, dtype, s);
}

// Two-axis gates: per-fiber kernels when the inner gate axis has a long
// coalesced run; LDS slab tiles when it is (nearly) innermost and a tile fits;
// element-wise kernels otherwise.  Slab tiles need a large enough state to pay
// for their staging, so tiny states stay element-wise.
constexpr int64_t kSlabMinState = 1 << 16;

bool use_slab(int64_t N, int D, int64_t sa, int64_t sb, int dtype, int adjoint) {
  const int64_t so = sa > sb ? sa : sb, si = sa > sb ? sb : sa;
  return N >= kSlabMinState && slab_supported(N, D, so, si, dtype, adjoint);
}

int bs_pass(const void* in, void* out, int64_t N, int D, int64_t sp, int64_t sq, const void* g, int conj, int dtype,
            hipStream_t s) {
  if (use_fib(D, sp < sq ? sp : sq)) {
    if (mfma_supported(D, dtype)) return pair_bs_mfma(in, out, N, D, sp, sq, g, conj, s);
    return pair_bs_fib(in, out, N, D, sp, sq, g, conj, dtype, s);
  }
  if (use_slab(N, D, sp, sq, dtype, 0)) return pair_bs_slab(in, out, N, D, sp, sq, g, conj, dtype, s);
  return pair_bs(in, out, N, D, sp, sq, g, conj, dtype, s);
}

int bs_adj_pass(const void* psi, const void* lo, void* li, int64_t N, int D, int64_t sp, int64_t sq, const void* g,
                const void* dB, int conj, int wa, int wb, double* pb, int nwg, int zp1, int dtype, hipStream_t s) {
  if (use_fib(D, sp < sq ? sp : sq)) {
    if (mfma_supported(D, dtype))
      return pair_bs_adj_mfma(psi, lo, li, N, D, sp, sq, g, dB, conj, wa, wb, pb, nwg, zp1, s);
    return pair_bs_adj_fib(psi, lo, li, N, D, sp, sq, g, dB, conj, wa, wb, pb, nwg, zp1, dtype, s);
  }
  if (use_slab(N, D, sp, sq, dtype, 1))
    return pair_bs_adj_slab(psi, lo, li, N, D, sp, sq, g, dB, conj, wa, wb, pb, nwg, zp1, dtype, s);
  return pair_bs_adj(psi, lo, li, N, D, sp, sq, g, dB, conj, wa, wb, pb, nwg, zp1, dtype, s);
}

// two-mode pass of any two-mode kind (S2 on its own kernels, the others on the
// beamsplitter family)
int pair_pass(int kind, const void* in, void* out, int64_t N, int D, int64_t sp, int64_t sq, const void* g, int conj,
              int dtype, hipStream_t s) {
  if (kind == SFAMD_OP_TWO_MODE_SQUEEZE) {
    // the beamsplitter's per-fiber (matrix-core for complex64) and slab kernels on
    // difference blocks; the element-wise S2 kernel otherwise
    const bool fib = use_fib(D, sp < sq ? sp : sq);
    if (mfma_supported(D, dtype)) {
      if (fib) return pair_bs_mfma(in, out, N, D, sp, sq, g, conj, s, 1);
      if (use_slab(N, D, sp, sq, dtype, 0)) return pair_bs_slab(in, out, N, D, sp, sq, g, conj, dtype, s, 1);
    } else if (fib) {
      return pair_bs_fib(in, out, N, D, sp, sq, g, conj, dtype, s, 1);
    }
    return pair_s2(in, out, N, D, sp, sq, g, conj, dtype, s);
  }
  return bs_pass(in, out, N, D, sp, sq, g, conj, dtype, s);
}

int pair_adj_pass(int kind, const void* psi, const void* lo, void* li, int64_t N, int D, int64_t sp, int64_t sq,
                  const void* g, const void* dG, int conj, double* pb, int nwg, int zp1, int dtype, hipStream_t s) {
  if (kind == SFAMD_OP_TWO_MODE_SQUEEZE) {
    // d/dphi G[N][n] = i (N - n) G[N][n]: weights wa = -1, wb = 1
    const bool fib = use_fib(D, sp < sq ? sp : sq);
    if (mfma_supported(D, dtype)) {
      if (fib) return pair_bs_adj_mfma(psi, lo, li, N, D, sp, sq, g, dG, conj, -1, 1, pb, nwg, zp1, s, 1);
      if (use_slab(N, D, sp, sq, dtype, 1))
        return pair_bs_adj_slab(psi, lo, li, N, D, sp, sq, g, dG, conj, -1, 1, pb, nwg, zp1, dtype, s, 1);
    } else if (fib) {
      return pair_bs_adj_fib(psi, lo, li, N, D, sp, sq, g, dG, conj, -1, 1, pb, nwg, zp1, dtype, s, 1);
    }
    return pair_s2_adj(psi, lo, li, N, D, sp, sq, g, dG, conj, pb, nwg, zp1, dtype, s);
  }
  int wa, wb;
  bs_weights(kind, &wa, &wb);
  return bs_adj_pass(psi, lo, li, N, D, sp, sq, g, dG, conj, wa, wb, pb, nwg, zp1, dtype, s);
}

int loss_pass(const void* in, void* out, int64_t N, int D, int64_t sb, int64_t sk, const void* c, int dtype,
              hipStream_t s) {
  if (use_fib(D, sk)) return loss_fib(in, out, N, D, sk, c, dtype, s);
  if (use_slab(N, D, sb, sk, dtype, 0)) return loss_slab(in, out, N, D, sb, sk, c, dtype, s);
  return loss_fwd(in, out, N, D, sb, sk, c, dtype, s);
}

int loss_adj_pass(const void* psi, const void* lo, void* li, int64_t N, int D, int64_t sb, int64_t sk, const void* c,
                  const void* dc, double* pb, int nwg, int zp1, int dtype, hipStream_t s) {
  if (use_fib(D, sk)) return loss_adj_fib(psi, lo, li, N, D, sk, c, dc, pb, nwg, zp1, dtype, s);
  if (use_slab(N, D, sb, sk, dtype, 1)) return loss_adj_slab(psi, lo, li, N, D, sb, sk, c, dc, pb, nwg, zp1, dtype, s);
  return loss_adj(psi, lo, li, N, D, sb, sk, c, dc, pb, nwg, zp1, dtype, s);
}

// forward of one operation: in -> out (tmp: scratch state for two-pass ops)
int apply_op(const OpPlan& op, int n, int D, const void* table, const void* in, void* out, void* tmp, int dtype,
             hipStream_t s) {
  const int64_t NK = ipow(D, n), NM = ipow(D, 2 * n);
  const void* g = cptr(table, op.off, dtype);
  switch (op.kind) {
    case SFAMD_OP_ROTATION:
    case SFAMD_OP_KERR:
      if (op.mixed_in)
        return pair_diag(in, out, NM, D, bra_stride_dm(n, D, op.m0), ket_stride_dm(n, D, op.m0), g, dtype, s);
      return axis_diag(in, out, NK, D, ket_stride(n, D, op.m0), g, 0, dtype, s);
    case SFAMD_OP_DISPLACEMENT:
    case SFAMD_OP_SQUEEZE:
    case SFAMD_OP_CUBIC_PHASE: {
      const int par = op.kind == SFAMD_OP_SQUEEZE;
      if (op.mixed_in) {
        const int64_t sk = ket_stride_dm(n, D, op.m0);
        if (dm_dense_mfma_supported(D, dtype, sk)) return dm_dense_mfma(in, out, NM, D, sk, g, s);
        if (!tmp) return SFAMD_E_WORKSPACE;
        RET_IF(dense_pass(in, tmp, NM, D, bra_stride_dm(n, D, op.m0), g, 0, par, dtype, s));
        return dense_pass(tmp, out, NM, D, ket_stride_dm(n, D, op.m0), g, 1, par, dtype, s);
      }
      return dense_pass(in, out, NK, D, ket_stride(n, D, op.m0), g, 0, par, dtype, s);
    }
    case SFAMD_OP_BEAMSPLITTER:
    case SFAMD_OP_TWO_MODE_SQUEEZE:
    case SFAMD_OP_MZGATE:
    case SFAMD_OP_CROSS_KERR:
      if (op.mixed_in) {
        // one pass (rho' = G rho G^H) when a run of inner modes follows the pair
        if (dm_pair_mfma_supported(n, D, op.m0, op.m1, dtype))
          return dm_pair_mfma(in, out, n, D, op.m0, op.m1, g, op.kind == SFAMD_OP_TWO_MODE_SQUEEZE, s);
        if (!tmp) return SFAMD_E_WORKSPACE;
        RET_IF(pair_pass(op.kind, in, tmp, NM, D, bra_stride_dm(n, D, op.m0), bra_stride_dm(n, D, op.m1), g, 0,
                         dtype, s));
        return pair_pass(op.kind, tmp, out, NM, D, ket_stride_dm(n, D, op.m0), ket_stride_dm(n, D, op.m1), g, 1,
                         dtype, s);
      }
      return pair_pass(op.kind, in, out, NK, D, ket_stride(n, D, op.m0), ket_stride(n, D, op.m1), g, 0, dtype, s);
    case SFAMD_OP_LOSS: {
      const void* src = in;
      if (op.mix_first) {
        if (!tmp) return SFAMD_E_WORKSPACE;
        RET_IF(mix_fwd(in, tmp, n, D, dtype, s));
        src = tmp;
      }
      return loss_pass(src, out, NM, D, bra_stride_dm(n, D, op.m0), ket_stride_dm(n, D, op.m0), g, dtype, s);
    }
    case SFAMD_OP_MIX:
      return mix_fwd(in, out, n, D, dtype, s);
    default:
      return SFAMD_E_KIND;
  }
}

// adjoint of one operation.  pb = partial base of this op: pass p writes
// slot 0 at pb + (2p)*nwg and slot 1 at pb + (2p+1)*nwg.
int adjoint_op(const OpPlan& op, int n, int D, const void* table, const void* psi, const void* lo, void* li,
               void* t1, void* t2, double* pb, int nwg, int dtype, hipStream_t s) {
  const int64_t NK = ipow(D, n), NM = ipow(D, 2 * n);
  const void* g = cptr(table, op.off, dtype);
  double* pass0 = pb;
  double* pass1 = pb + 2 * (int64_t)nwg;
  const int kerr = op.kind == SFAMD_OP_KERR;
  switch (op.kind) {
    case SFAMD_OP_ROTATION:
    case SFAMD_OP_KERR:
      if (op.mixed_in)
        return pair_diag_adj(psi, lo, li, NM, D, bra_stride_dm(n, D, op.m0), ket_stride_dm(n, D, op.m0), g, kerr,
                             pass0, nwg, 1, dtype, s);
      return axis_diag_adj(psi, lo, li, NK, D, ket_stride(n, D, op.m0), g, kerr, 0, pass0, nwg, 1, dtype, s);
    case SFAMD_OP_DISPLACEMENT:
    case SFAMD_OP_SQUEEZE:
    case SFAMD_OP_CUBIC_PHASE: {
      const int64_t DD = (int64_t)D * D;
      const void* dU0 = cptr(g, DD, dtype);
      const void* dU1 = cptr(g, 2 * DD, dtype);
      const int par = op.kind == SFAMD_OP_SQUEEZE;
      if (op.mixed_in) {
        const int64_t sb = bra_stride_dm(n, D, op.m0), sk = ket_stride_dm(n, D, op.m0);
        // rho1 = U rho (bra side) recomputed; then the ket-side pass, then the bra-side pass
        RET_IF(dense_pass(psi, t1, NM, D, sb, g, 0, par, dtype, s));
        RET_IF(dense_adj_pass(t1, lo, t2, NM, D, sk, g, dU0, dU1, 1, par, pass1, nwg, 0, dtype, s));
        return dense_adj_pass(psi, t2, li, NM, D, sb, g, dU0, dU1, 0, par, pass0, nwg, 0, dtype, s);
      }
      return dense_adj_pass(psi, lo, li, NK, D, ket_stride(n, D, op.m0), g, dU0, dU1, 0, par, pass0, nwg, 1, dtype, s);
    }
    case SFAMD_OP_BEAMSPLITTER:
    case SFAMD_OP_TWO_MODE_SQUEEZE:
    case SFAMD_OP_MZGATE:
    case SFAMD_OP_CROSS_KERR: {
      const void* dB = cptr(g, bs_nb(D), dtype);
      const int k = op.kind;
      if (op.mixed_in) {
        const int64_t bp = bra_stride_dm(n, D, op.m0), bq = bra_stride_dm(n, D, op.m1);
        const int64_t kp = ket_stride_dm(n, D, op.m0), kq = ket_stride_dm(n, D, op.m1);
        RET_IF(pair_pass(k, psi, t1, NM, D, bp, bq, g, 0, dtype, s));
        RET_IF(pair_adj_pass(k, t1, lo, t2, NM, D, kp, kq, g, dB, 1, pass1, nwg, 0, dtype, s));
        return pair_adj_pass(k, psi, t2, li, NM, D, bp, bq, g, dB, 0, pass0, nwg, 0, dtype, s);
      }
      return pair_adj_pass(k, psi, lo, li, NK, D, ket_stride(n, D, op.m0), ket_stride(n, D, op.m1), g, dB, 0, pass0,
                           nwg, 1, dtype, s);
    }
    case SFAMD_OP_LOSS: {
      const int64_t D3 = (int64_t)D * D * D;
      const char* c = (const char*)g;
      const char* dc = c + D3 * (elem_size(dtype) / 2);
      const int64_t sb = bra_stride_dm(n, D, op.m0), sk = ket_stride_dm(n, D, op.m0);
      if (op.mix_first) {
        RET_IF(mix_fwd(psi, t1, n, D, dtype, s));
        RET_IF(loss_adj_pass(t1, lo, t2, NM, D, sb, sk, c, dc, pass0, nwg, 1, dtype, s));
        return mix_adj(psi, t2, li, n, D, dtype, s);
      }
      return loss_adj_pass(psi, lo, li, NM, D, sb, sk, c, dc, pass0, nwg, 1, dtype, s);
    }
    case SFAMD_OP_MIX:
      RET_IF(fill_zero(pb, 4 * (int64_t)nwg * sizeof(double), s));
      return mix_adj(psi, lo, li, n, D, dtype, s);
    default:
      return SFAMD_E_KIND;
  }
}

}  // namespace

// One step of execution: a single operation (or a run of diagonal gates), or a
// fused stage of gates on K local modes: on the vector ALUs (two modes of a ket, at some
// cutoffs three; fused.hip) or on the matrix cores (K >= 3, mstage.hip).  On a density
// matrix a matrix-core stage is two launches: the gates on the row axes of its
// modes, then their conjugates on the column axes.
enum StepKind { kStepSingle = 0, kStepDiagRun, kStepStage, kStepMatrixStage };
struct Step {
  int kind;
  int op;  // single operation index (kStepSingle)
  int K;
  std::vector<int> ops;  // operation indices in execution order
  StageArgs args;
  std::vector<MArgs> margs;  // of a matrix-core stage; [1]: the column axes of a density matrix
  bool mixed;      // the stage acts on a density matrix
  DiagRun run;
};

struct sfamd_prog {
  int n, D, dtype, mixed_in, nops, nwg, fuse_K, fuse_mixed, fuse_paying;
  std::vector<OpPlan> ops;
  std::vector<int32_t> img0, img1;          // per op: its vector-ALU stage images, or copies of its phases; -1: none
  std::vector<int32_t> mimg_fwd, mimg_adj;  // per op: its matrix-core images, or -1
  std::vector<Step> steps;
  // the whole program without checkpoints or adjoint (sfamd_prog_run): matrix-core
  // stages hold one tile in LDS, so they take more gates; empty: the same as steps
  std::vector<Step> fsteps;
  std::vector<int64_t> state_elems;  // elements at the input of step i (i = nsteps: output)
  int64_t table_elems, max_state;
  int final_mixed;
};

namespace {

// The stages of one representation: its axes (n of a ket, 2 n of a density
// matrix: row and column of each mode in turn, slowest first), the kind of its
// stages and their local axes (0: no stages).
struct Stages {
  bool mixed;
  int axes, kind, Kc;
  int modes(int n) const { return Kc < n ? Kc : n; }  // that a stage takes gates of
};

// the vector-ALU stages hold the gates of the layered circuit, the matrix-core stages every unitary gate
bool fusable(const OpPlan& op, const Stages& sg) {
  return op.kind == SFAMD_OP_ROTATION || op.kind == SFAMD_OP_KERR || op.kind == SFAMD_OP_DISPLACEMENT ||
         op.kind == SFAMD_OP_SQUEEZE || op.kind == SFAMD_OP_BEAMSPLITTER ||
         (sg.kind == kStepMatrixStage && (mst_two_mode(op.kind) || op.kind == SFAMD_OP_CUBIC_PHASE));
}


int op_nmodes(const OpPlan& op) { return two_mode_kind(op.kind) ? 2 : 1; }

unsigned op_mask(const OpPlan& op) {
  unsigned m = 1u << op.m0;
  if (two_mode_kind(op.kind)) m |= 1u << op.m1;
  return m;
}

// LDS a stage needs, by the kernels that run it: fixed bytes and bytes per gate
struct StageCost {
  int64_t base, budget, budget_full;
  int max_gates;
  std::function<int64_t(const OpPlan&)> gate;
};

// An operation as the stage search sees it.
struct StageOp {
  unsigned modes;
  int64_t cost;
};

// ops of `rem` (program order) absorbable into a stage on `mask`: an op joins
// if its modes lie in the mask, no earlier op left outside the stage touches
// one of them (gates on disjoint modes commute) and the stage's LDS fits.
// Returns their number; `skip` marks operations that an earlier stage takes,
// `got` receives the indices; `ops` and `skip` begin at operation `base`.
int absorb(const std::vector<StageOp>& ops, int base, const std::vector<int>& rem, unsigned mask, const StageCost& sc,
           int64_t budget, const char* skip, std::vector<int>* got) {
  if (got) got->clear();
  unsigned blocked = 0;
  int64_t used = sc.base;
  int count = 0;
  for (int i : rem) {
    const StageOp& op = ops[i - base];
    if (!(op.modes & mask) || (skip && skip[i - base])) continue;
    if (count < sc.max_gates && !(op.modes & ~mask) && !(op.modes & blocked) && used + op.cost <= budget) {
      if (got) got->push_back(i);
      ++count;
      used += op.cost;
    } else {
      blocked |= op.modes;
      if ((blocked & mask) == mask) break;  // nothing further can join
    }
  }
  return count;
}

bool is_diag_kind(int kind) { return kind == SFAMD_OP_ROTATION || kind == SFAMD_OP_KERR; }

Step new_step(int kind, int op) {
  Step st;
  st.kind = kind;
  st.op = op;
  st.K = 0;
  st.mixed = false;
  memset(&st.args, 0, sizeof(st.args));
  memset(&st.run, 0, sizeof(st.run));
  return st;
}

// An operation on its own: consecutive rotation / Kerr gates on the same
// representation share one pass
void add_single(const sfamd_prog* p, int i, std::vector<Step>* steps) {
  if (is_diag_kind(p->ops[i].kind) && !steps->empty()) {
    Step& last = steps->back();
    if (last.kind <= kStepDiagRun && is_diag_kind(p->ops[last.ops.back()].kind) &&
        p->ops[last.ops.back()].mixed_in == p->ops[i].mixed_in && (int)last.ops.size() < kDiagRunMax) {
      last.ops.push_back(i);
      last.kind = kStepDiagRun;
      return;
    }
  }
  Step st = new_step(kStepSingle, i);
  st.ops.push_back(i);
  steps->push_back(st);
}

constexpr int kMstGatesForTwo = 4;            // gates each of two workgroups per CU must still hold

// log2 of the tiles a workgroup of a matrix-core stage holds: as many as fill
// the 16 columns of a beamsplitter's matrix-core operand, if every CU still
// has a group
int group_log2(const sfamd_prog* p, int axes, int Kc) {
  const int D = p->D;
  const int64_t ntiles = ipow(D, axes - Kc);
  int l = 0;
  while (mst_group_fills(D, Kc, l + 1) && (ntiles >> (l + 1)) >= kComputeUnits) ++l;
  return l;
}

// What a stage of Kc local modes may hold.  kStepStage: one tile per gate plus
// three and every gate's matrices (the adjoint kernel's LDS).
// kStepMatrixStage: the adjoint keeps one tile per gate with operators plus two,
// the forward-only plan one tile group.
StageCost stage_cost(const sfamd_prog* p, const Stages& sg, bool forward_only) {
  const int D = p->D, kind = sg.kind, Kc = sg.Kc;
  const int64_t esz = elem_size(p->dtype);
  // a launch has one workgroup per tile (up to the grid cap): when that is
  // more than one per compute unit, two should fit in a CU's LDS at once
  const bool many = ipow(D, sg.axes - Kc) > kComputeUnits;
  StageCost sc;
  sc.budget_full = kStageLdsBudget;
  sc.budget = many ? kStageLdsPerCu / 2 - 512 : kStageLdsBudget;
  if (kind == kStepStage) {
    const int64_t tile = stage_tile(D, Kc) * esz, slots = 2 * (stage_threads(D, Kc) / 64) * 8;
    sc.max_gates = kStageMaxGates;
    sc.base = 3 * tile;  // the stage input and two cotangent tiles
    sc.gate = [=](const OpPlan& op) {
      return tile + (((stage_gate_elems(op.kind, D, true) + 1) & ~(int64_t)1) * esz) + slots;
    };
    return sc;
  }
  const int lgt = group_log2(p, sg.axes, Kc);
  const int64_t tile = ((int64_t)mst_tile_lds(D, Kc) << lgt) * esz, phases = (int64_t)(D + 1) * esz;
  sc.max_gates = kMstMaxGates;
  sc.budget_full = kMstLdsMax;
  if ((ipow(D, sg.axes - Kc) >> lgt) <= kComputeUnits) sc.budget = sc.budget_full;
  if (forward_only) {
    sc.base = tile;
    sc.budget = sc.budget_full;
    sc.gate = [=](const OpPlan& op) { return is_diag_kind(op.kind) ? phases : 0; };
    return sc;
  }
  const int64_t slots = 2 * mst_waves(D, Kc, lgt) * 8;
  // two workgroups per CU only if the kernel's registers allow it and each still holds kMstGatesForTwo gates
  if (!mst_two_groups(D, p->dtype) || sc.budget < 2 * tile + kMstGatesForTwo * (tile + slots))
    sc.budget = sc.budget_full;
  sc.base = 2 * tile;
  sc.gate = [=](const OpPlan& op) { return (is_diag_kind(op.kind) ? phases : tile) + slots; };
  return sc;
}

// Can a stage of this kind hold one gate of any kind?
bool stage_fits(const sfamd_prog* p, const Stages& sg, bool forward_only) {
  if (sg.Kc < 2 || sg.Kc > sg.axes) return false;
  if (sg.kind == kStepStage ? (sg.mixed || sg.axes > kStageMaxModes || !stage_supported(p->D, sg.Kc, p->dtype))
                            : (sg.axes > kMstMaxModes || !mst_supported(p->D, sg.Kc)))
    return false;
  int64_t tiles = 1;
  for (int i = sg.Kc; i < sg.axes; ++i)
    if ((tiles *= p->D) >= ((int64_t)1 << 31)) return false;
  const StageCost sc = stage_cost(p, sg, forward_only);
  OpPlan bs{SFAMD_OP_BEAMSPLITTER, 0, 1, 0, 0, 0};
  return sc.base + sc.gate(bs) <= sc.budget_full;
}

void fill_stage(const sfamd_prog* p, Step& st, unsigned mask) {
  const int n = p->n, D = p->D, Kc = st.K;
  StageArgs& a = st.args;
  a.ngates = (int)st.ops.size();
  int lmodes[4], nl = 0, nlc = 0;
  for (int md = 0; md < n; ++md) {
    if (mask >> md & 1u)
      lmodes[nl++] = md;
    else
      a.nl_stride[nlc++] = ipow(D, n - 1 - md);
  }
  a.nnl = nlc;
  a.ntiles = (int32_t)ipow(D, nlc);
  for (int t = 0; t < Kc; ++t) a.loc_stride[t] = ipow(D, n - 1 - lmodes[t]);
  int64_t mf = 0, ma = 0;
  for (int gi = 0; gi < a.ngates; ++gi) {
    const OpPlan& op = p->ops[st.ops[gi]];
    StageGate& g = a.g[gi];
    g.kind = (int8_t)op.kind;
    g.a0 = g.a1 = 0;
    for (int t = 0; t < Kc; ++t) {
      if (lmodes[t] == op.m0) g.a0 = (int8_t)t;
      if (op.kind == SFAMD_OP_BEAMSPLITTER && lmodes[t] == op.m1) g.a1 = (int8_t)t;
    }
    g.op = st.ops[gi];
    g.s0 = (int32_t)ipow(D, Kc - 1 - g.a0);
    g.s1 = (int32_t)ipow(D, Kc - 1 - g.a1);
    // one region per gate, 16-byte aligned in LDS: the matrix in the
    // forward kernel, matrix + derivative in the adjoint
    g.moff = (int32_t)mf;
    g.amoff = (int32_t)ma;
    mf += (stage_gate_elems(op.kind, D, false) + 1) & ~(int64_t)1;
    ma += (stage_gate_elems(op.kind, D, true) + 1) & ~(int64_t)1;
  }
  a.mat_fwd = (int32_t)mf;
  a.mat_adj = (int32_t)ma;
}

// order of the modes in a state, slowest first, and their strides
struct ModeOrder {
  int n = 0, at[32];
  int64_t stride[32];  // by mode
  void set_strides(int D) {
    int64_t s = 1;
    for (int i = n - 1; i >= 0; --i) {
      stride[at[i]] = s;
      s *= D;
    }
  }
};

ModeOrder canonical_order(int n, int D) {
  ModeOrder o;
  o.n = n;
  for (int m = 0; m < n; ++m) o.at[m] = m;
  o.set_strides(D);
  return o;
}

// a matrix-core stage on the axes of `mask`, from states in axis order `in` to
// states in axis order `out`; side 1: on the column axes of a density matrix
void fill_matrix_stage(const sfamd_prog* p, Step& st, unsigned mask, const ModeOrder& in, const ModeOrder& out,
                       int side) {
  const int n = in.n, D = p->D, Kc = st.K;
  if ((int)st.margs.size() <= side) st.margs.resize(side + 1);
  MArgs& a = st.margs[side];
  memset(&a, 0, sizeof(a));
  a.side = side;
  a.ngates = (int)st.ops.size();
  int lmodes[kMstMaxK], nl = 0;
  for (int i = n - 1; i >= 0; --i)  // fastest first
    if (!(mask >> in.at[i] & 1u)) {
      a.nl_stride[a.nnl] = in.stride[in.at[i]];
      a.out_nl_stride[a.nnl++] = out.stride[in.at[i]];
    }
  for (int i = 0; i < n; ++i)  // slowest first
    if (mask >> in.at[i] & 1u) lmodes[nl++] = in.at[i];
  a.ntiles = (int32_t)ipow(D, a.nnl);
  a.lgt = group_log2(p, n, Kc);
  for (int t = 0; t < Kc; ++t) a.loc_stride[t] = in.stride[lmodes[t]];
  int u = 0;
  for (int i = 0; i < n; ++i)
    for (int t = 0; t < Kc; ++t)
      if (lmodes[t] == out.at[i]) {
        a.out_stride[u] = out.stride[out.at[i]];
        a.out_lds[u++] = mst_stride(D, Kc, t);
      }
  for (int gi = 0; gi < a.ngates; ++gi) {
    const OpPlan& op = p->ops[st.ops[gi]];
    MGate& g = a.g[gi];
    const bool two = mst_two_mode(op.kind), diff = op.kind == SFAMD_OP_TWO_MODE_SQUEEZE;
    int ax0 = 0, ax1 = -1;
    const int m0 = st.mixed ? 2 * op.m0 + side : op.m0, m1 = st.mixed ? 2 * op.m1 + side : op.m1;
    for (int t = 0; t < Kc; ++t) {
      if (lmodes[t] == m0) ax0 = t;
      if (two && lmodes[t] == m1) ax1 = t;
    }
    int u = 0;
    for (int t = 0; t < Kc; ++t)
      if (t != ax0 && t != ax1) g.cs[u++] = mst_stride(D, Kc, t);
    g.kind = op.kind;
    g.a0 = !two ? ax0 : diff ? -1 : 0;
    g.l1 = two ? mst_stride(D, Kc, ax1) : 0;
    g.ds = mst_stride(D, Kc, ax0) + (diff ? g.l1 : -g.l1);
    g.wrap = (diff ? -D : D) * g.l1;
    g.op = st.ops[gi];
    g.two = (two ? 1 : 0) | mst_weights(op.kind);
    if (is_diag_kind(op.kind))
      ++a.ndiag;
    else
      ++a.nheavy;
  }
}

// a matrix-core stage on the modes of `mask`, both states in the canonical axis
// order: on a density matrix both its sides, the tile completed by the fastest
// other axes where the modes are fewer than the local axes
void fill_matrix_step(const sfamd_prog* p, Step& st, unsigned mask) {
  const int axes = st.mixed ? 2 * p->n : p->n;
  const ModeOrder order = canonical_order(axes, p->D);
  for (int side = 0; side <= (st.mixed ? 1 : 0); ++side) {
    unsigned m = mask;
    if (st.mixed) {
      m = 0;
      for (int md = 0; md < p->n; ++md)
        if (mask >> md & 1u) m |= 1u << (2 * md + side);
      for (int a = axes - 1; __builtin_popcount(m) < st.K; --a) m |= 1u << a;
    }
    fill_matrix_stage(p, st, m, order, order, side);
  }
}

// table offsets of a matrix-core stage's images, once they are placed; every
// gate, also a rotation or Kerr gate, names the forward image of the next gate
// with operators and the adjoint image of the previous one (at the ends, and in
// a stage without such gates, an image that is loaded and not used)
void link_matrix_stage(const sfamd_prog* p, MArgs& a, int spare) {
  int nd = 0;
  a.h0_fwd = a.hl_adj = spare;
  int off = spare, two = 0;
  for (int gi = 0; gi < a.ngates; ++gi) {
    MGate& g = a.g[gi];
    g.padj = off;
    g.two |= two << 2;
    if (is_diag_kind(g.kind)) {
      g.fwd = nd++ * p->D;
      continue;
    }
    g.fwd = p->mimg_fwd[g.op];
    g.adj = p->mimg_adj[g.op] < 0 ? spare : p->mimg_adj[g.op];
    off = a.hl_adj = g.adj;
    two = a.hl_two = g.two & 1;
  }
  off = spare;
  two = 0;
  for (int gi = a.ngates - 1; gi >= 0; --gi) {
    MGate& g = a.g[gi];
    g.nfwd = off;
    g.two |= two << 1;
    if (is_diag_kind(g.kind)) continue;
    off = a.h0_fwd = g.fwd;
    two = a.h0_two = g.two & 1;
  }
}

// Mode orders between the stages of a forward-only run (masks: their local
// modes, first: the first of them).  A stage whose local modes are not the
// fastest ones reads and writes single amplitudes, one cache line each (6
// modes, cutoff 16, complex64, 134 MB: two beamsplitters on modes 0 to 2 292 us,
// one on the last modes 58 us, a device copy 38 us).  The states between the
// stages are the library's own, so each stage writes its output with the next
// stage's local modes fastest: reads are whole tiles, and writes are runs of the
// mode that the two stages share, placed fastest of all.  Unused local modes are
// chosen to share one with the stage before.
void order_stages(const sfamd_prog* p, std::vector<Step>* steps, size_t first, std::vector<unsigned> masks) {
  const int n = p->n, D = p->D;
  const size_t count = masks.size();
  if (n <= (*steps)[first].K) return;
  for (size_t i = 0; i < count; ++i) {
    unsigned used = 0;
    for (int op : (*steps)[first + i].ops) used |= op_mask(p->ops[op]);
    const unsigned before = i ? masks[i - 1] : 1u << (n - 1);
    const unsigned after = i + 1 < count ? masks[i + 1] : 1u << (n - 1);
    unsigned m = used;
    auto fill = [&](unsigned from) {
      for (int md = n - 1; md >= 0; --md)
        if (__builtin_popcount(m) < (*steps)[first + i].K && (from >> md & 1u)) m |= 1u << md;
    };
    if (!(used & before)) fill(before & ~(before - 1u));  // one mode of the stage before
    if (!(used & after)) fill(after & ~(after - 1u));
    fill(before);
    fill(~0u >> (32 - n));
    masks[i] = m;
  }
  ModeOrder in = canonical_order(n, D);
  for (size_t i = 0; i < count; ++i) {
    ModeOrder out = canonical_order(n, D);
    if (i + 1 < count) {
      int k = 0;
      const unsigned next = masks[i + 1], mine = masks[i];
      for (int pass = 0; pass < 3; ++pass)  // others, the next stage's own, the shared ones (fastest)
        for (int j = 0; j < n; ++j) {
          const unsigned b = 1u << in.at[j];
          const int cls = !(next & b) ? 0 : !(mine & b) ? 1 : 2;
          if (cls == pass) out.at[k++] = in.at[j];
        }
      out.set_strides(D);
    }
    MArgs& a = (*steps)[first + i].margs[0];
    fill_matrix_stage(p, (*steps)[first + i], masks[i], in, out, 0);
    a.permuted = 1;
    // no shared mode: the workgroup takes neighbouring tiles, for runs of that many amplitudes
    if (a.out_stride[(*steps)[first + i].K - 1] != 1)
      while (mst_group_ok(D, (*steps)[first + i].K, a.lgt + 1) && (a.ntiles >> (a.lgt + 1)) >= 4 * kComputeUnits &&
             mst_lds_fwd(D, (*steps)[first + i].K, a.lgt + 1, a.ndiag, p->dtype) <= kMstLds / 2)
        ++a.lgt;
    in = out;
  }
}

int64_t state_mb(const sfamd_prog* p, bool mixed) {
  return ipow(p->D, mixed ? 2 * p->n : p->n) * elem_size(p->dtype) / 1000000;
}

// How many gates make a matrix-core stage pay?  A stage costs its launches (on a
// density matrix two, its adjoint five), tiles that stride over the state and
// the gates' operator images in the table build; a gate alone is one coalesced
// pass, or two on a density matrix.  gate_weight: what a gate alone costs, in
// halves of a single-mode gate's pass.  stage_need: what the gates of one stage
// have to weigh together.  Measured with 1 to 9 single-mode gates (d) and 1 to 4
// beamsplitters (b) in one stage, gates alone / stage, us:
//   density matrices, forward, complex64: 4 modes 8 (134 MB) 1d 42 / 129, 2d 97 /
//   145, 3d 165 / 163, 1b 202 / 132; 3 modes 9 3d 23 / 31, 6d 48 / 43, 1b 28 / 25; 12
//   3d 48 / 66, 6d 94 / 92, 1b 55 / 52; 16 6d 409 / 464, 9d 608 / 564, 2b 282 / 370, 4b
//   570 / 409; 7 modes 3 3d 104 / 142, 6d 208 / 206; 2 modes 8 1d 7 / 10, 2d 10 / 12,
//   3d 13 / 11; complex128: 3 modes 9 1d 20 / 35, 2d 43 / 50, 3d 67 / 50, 1b 26 / 38, 2b 62 /
//   48; 16 1d 320 / 390, 2d 628 / 467; 20 2d 3103 / 3172, 3d 5659 / 3627; 7 modes 3 3d
//   158 / 168, 6d 310 / 255;
//   their adjoints: complex64 4 modes 8 2d 531 / 594, 3d 802 / 704, 1b 479 / 519; 3 modes
//   12 2d 172 / 208, 3d 258 / 250, 1b 147 / 186, 2b 302 / 243; complex128 3 modes 9 1d 86 /
//   124, 2d 168 / 158; 6 modes 3 3d 109 / 135, 6d 210 / 204;
//   kets, forward: complex64 9 modes 5 1d 9 / 18, 2d 19 / 21, 3d 28 / 28; 13 modes 3 3d
//   28 / 38, 6d 56 / 48; 20 modes 2 9d 68 / 68; 8 modes 8 1d 42 / 57, 2d 86 / 69; complex128
//   13 modes 3 6d 55 / 57; adjoints: complex64 8 modes 8 1d 146 / 192, 2d 294 / 276;
//   complex128 12 modes 3 6d 82 / 90.
// Where the gate alone has no kernel that reads whole fibers with coalesced runs (a
// pair with the last mode, a complex128 gate on it), or one thread per fiber leaves
// the device idle (complex128 on few fibers), it costs a multiple: CK on 6 modes 16
// complex64 98 / 63, BS on the last modes of 6 modes 8 complex128 19 / 7, D on 4 modes
// 15 complex128 18 / 7.
int gate_weight(const sfamd_prog* p, const Stages& sg, const OpPlan& op) {
  const int n = p->n, D = p->D;
  const bool two = two_mode_kind(op.kind);
  const int64_t N = ipow(D, sg.axes);
  int64_t inner = ket_stride(n, D, op.m0);  // the innermost run of the gate's passes
  if (two) inner = std::min(inner, ket_stride(n, D, op.m1));
  if (sg.mixed) inner *= inner;
  const bool fib = use_fib(D, inner), tiny = N < kSlabMinState;
  if (p->dtype == SFAMD_C64) {
    if (!two) return 2;
    if (!sg.mixed) return tiny ? 3 : !fib ? (D <= 5 ? 6 : 5) : N <= (1 << 21) ? 4 : 3;
    if (n == 2) return D <= 12 ? 2 : 4;
    if (tiny) return 4;
    return D > 10 || (D > 8 && dm_pair_mfma_supported(n, D, op.m0, op.m1, p->dtype)) ? 6 : 8;
  }
  const bool few = D >= 8 && N / D < (sg.mixed ? 16384 : 65536);
  if (sg.mixed) {
    if (two && (D <= 3 || n == 2)) return D <= 12 && n == 2 ? 2 : 4;
    if (fib || N < 1500000) return few ? 4 : 2;
    return op.kind == SFAMD_OP_TWO_MODE_SQUEEZE || (!two && D > 12) ? 6 : 4;
  }
  if (!fib) return tiny ? 2 : two && D < 6 ? 4 : 6;
  return few || (!two && D >= 8) ? 4 : two ? 3 : 2;
}

int stage_need(const sfamd_prog* p, const Stages& sg, bool forward_only) {
  const int n = p->n, D = p->D;
  const bool c64 = p->dtype == SFAMD_C64, large = state_mb(p, sg.mixed) >= 16;
  if (sg.mixed && c64) {
    if (n == 2) return D <= 12 ? 4 : 6;
    if ((D <= 3 || D == 5) && large) return 12;  // tiles of few amplitudes, operands mostly padding
    if (forward_only) return D <= 12 ? 8 : 16;
    return D <= 3 || D == 11 || D == 12 ? 8 : 6;
  }
  if (sg.mixed) return D <= 3 ? 8 : D <= 12 || n == 2 ? 4 : 6;
  if (D <= 3 && ipow(D, n) >= kSlabMinState) return large ? 10 : c64 || forward_only ? 6 : 8;
  return D == 5 && forward_only ? 6 : 4;
}

// what the operations `ops` of a stage weigh; rotation and Kerr gates share one pass
int stage_weight(const sfamd_prog* p, const Stages& sg, const std::vector<int>& ops) {
  int w = 0, diag = 0;
  for (int i : ops) {
    if (is_diag_kind(p->ops[i].kind))
      diag = 2;
    else
      w += gate_weight(p, sg, p->ops[i]);
  }
  return w + diag;
}

// greedy partition of a run of fusable ops into stages of Kc local modes
void plan_run(const sfamd_prog* p, const std::vector<int>& run, const Stages& sg, bool forward_only,
              std::vector<Step>* steps) {
  const int n = p->n, kind = sg.kind, Kc = sg.modes(n);
  const StageCost sc = stage_cost(p, sg, forward_only);
  // stages that do not pay run gate by gate, if the caller asks for that: each by
  // itself, but kets forward only all or none (their stages share a mode order)
  const bool paying = p->fuse_paying && kind == kStepMatrixStage, ordered = forward_only && !sg.mixed;
  const int need = paying ? stage_need(p, sg, forward_only) : 0;
  std::vector<unsigned> masks;     // of this run's stages
  bool all_stages = true;
  const size_t first = steps->size();
  std::vector<int> rem = run;
  std::vector<unsigned> cands;
  // all Kc-subsets when few, else subsets grown from the next ops
  std::vector<int> idx(Kc);
  int64_t ncomb = 1;
  for (int t = 0; t < Kc; ++t) ncomb = ncomb * (n - t) / (t + 1);
  if (ncomb <= 512) {
    for (int t = 0; t < Kc; ++t) idx[t] = t;
    while (true) {
      unsigned m = 0;
      for (int t = 0; t < Kc; ++t) m |= 1u << idx[t];
      cands.push_back(m);
      int t = Kc - 1;
      while (t >= 0 && idx[t] == n - Kc + t) --t;
      if (t < 0) break;
      ++idx[t];
      for (int u = t + 1; u < Kc; ++u) idx[u] = idx[u - 1] + 1;
    }
  }
  std::vector<int> got, best;
  const int base = run.front();  // (a run's operations follow one another)
  std::vector<StageOp> sops;
  for (int i : run) sops.push_back(StageOp{op_mask(p->ops[i]), sc.gate(p->ops[i])});
  std::vector<char> taken(run.size(), 0);
  while (!rem.empty()) {
    std::vector<unsigned> local = cands;
    if (local.empty()) {
      unsigned m = 0;
      for (int i : rem) {
        const unsigned om = op_mask(p->ops[i]);
        if (__builtin_popcount(m | om) <= Kc) m |= om;
        if (__builtin_popcount(m) == Kc) break;
      }
      for (int md = n - 1; __builtin_popcount(m) < Kc && md >= 0; --md) m |= 1u << md;
      local.push_back(m);
    }
    unsigned bm = 0;
    best.clear();
    // the occupancy budget is a preference: a gate too large for it (compact
    // beamsplitter tables at high cutoff) gets a stage of the full budget
    for (int64_t bud : {sc.budget, sc.budget_full}) {
      long bkey = -1;
      for (unsigned m : local) {
        absorb(sops, base, rem, m, sc, bud, nullptr, &got);
        // one step of lookahead: the gates this stage takes plus the most the
        // next stage could take after it (on c3: 49 stages instead of 52);
        // ties go to more gates now, then to tiles that include the last
        // modes (contiguous runs)
        // (the search grows with the square of the mode sets; on a density matrix
        // of 9 to 11 modes, whose pass is short at that cutoff, it took longer than
        // tens of runs: 10 modes, cutoff 2, 2 layers 111 ms and 52 stages and losses, without
        // it 1.7 ms and 55)
        long nxt = 0;
        const bool look = local.size() > 1 && !(sg.mixed && local.size() > 100);
        if (look && !got.empty() && got.size() < rem.size()) {
          for (int i : got) taken[i - base] = 1;
          for (unsigned m2 : local) {
            const long k = absorb(sops, base, rem, m2, sc, bud, taken.data(), nullptr);
            if (k > nxt) nxt = k;
          }
          for (int i : got) taken[i - base] = 0;
        }
        const long key = (((long)got.size() + nxt) << 40) + ((long)got.size() << 26) + (long)m;
        if (key > bkey) {
          bkey = key;
          bm = m;
          best = got;
        }
      }
      if (!best.empty()) break;
    }
    if (best.empty()) {
      // no stage holds the next operation: it runs on its own, unfused
      add_single(p, rem.front(), steps);
      all_stages = false;
      rem.erase(rem.begin());
      continue;
    }
    if (paying && !ordered && stage_weight(p, sg, best) < need) {
      for (int i : best) add_single(p, i, steps);
      all_stages = false;
    } else {
      Step st = new_step(kind, best.front());
      st.K = sg.Kc;
      st.mixed = sg.mixed;
      st.ops = best;
      if (kind == kStepStage)
        fill_stage(p, st, bm);
      else
        fill_matrix_step(p, st, bm);
      steps->push_back(st);
      masks.push_back(bm);
    }
    std::vector<int> nrem;
    size_t bi = 0;
    for (int i : rem) {
      if (bi < best.size() && best[bi] == i)
        ++bi;
      else
        nrem.push_back(i);
    }
    rem.swap(nrem);
  }
  if (!ordered || kind != kStepMatrixStage) return;
  int w = 0;
  for (size_t i = first; i < steps->size(); ++i) w += stage_weight(p, sg, (*steps)[i].ops);
  if (paying && w < need * (int)(steps->size() - first)) {
    steps->resize(first, new_step(kStepSingle, 0));
    for (int i : run) add_single(p, i, steps);
  } else if (all_stages) {
    order_stages(p, steps, first, masks);
  }
}

// sg: the stages on kets and on density matrices
void plan_steps(const sfamd_prog* p, const Stages (&sg)[2], bool forward_only, std::vector<Step>* steps) {
  const int n = p->n, D = p->D;
  std::vector<int> run;
  auto flush = [&]() {
    if (run.empty()) return;
    const Stages& g = sg[p->ops[run.front()].mixed_in];
    // on a density matrix rotation and Kerr gates alone take one pass, a stage two
    bool heavy = !g.mixed;
    for (int i : run) heavy = heavy || !is_diag_kind(p->ops[i].kind);
    if (heavy)
      plan_run(p, run, g, forward_only, steps);
    else
      for (int i : run) add_single(p, i, steps);
    run.clear();
  };
  for (int i = 0; i < p->nops; ++i) {
    const Stages& g = sg[p->ops[i].mixed_in];
    if (g.Kc >= 2 && fusable(p->ops[i], g)) {
      if (!run.empty() && p->ops[run.front()].mixed_in != p->ops[i].mixed_in) flush();
      run.push_back(i);
      continue;
    }
    flush();
    add_single(p, i, steps);
  }
  flush();
  for (Step& st : *steps) {
    if (st.kind != kStepDiagRun) continue;
    DiagRun& r = st.run;
    const OpPlan& first = p->ops[st.ops.front()];
    r.n = n;
    r.D = D;
    r.mixed = first.mixed_in;
    r.ngates = (int)st.ops.size();
    r.N = ipow(D, r.mixed ? 2 * n : n);
    const int64_t R = r.mixed ? (int64_t)D * D : D;
    for (int g = 0; g < r.ngates; ++g) {
      const OpPlan& op = p->ops[st.ops[g]];
      r.mode[g] = op.m0;
      r.kind[g] = op.kind;
      r.op[g] = st.ops[g];
      int64_t dv = 1;
      for (int t = 0; t < n - 2 - op.m0; ++t) dv *= R;
      r.rowdiv[g] = dv;
    }
  }
}

// Do stages of K local modes pay on this state?  Past the caches a stage whose
// local modes are not the last ones moves single amplitudes (the forward-only
// plan orders the modes of its intermediate states against that), so kernels
// with one pass per gate catch up.  One layer of the layered circuit, forward
// and adjoint, unfused / fused, us (complex64: 6 modes cutoff 12, 24 MB: 2670 /
// 2420; 6 modes 14, 60 MB: 4570 / 6200; 7 modes 10, 80 MB: 8060 / 11100; 8 modes 8,
// 134 MB: 13950 / 10250; 9 modes 5, 16 MB: 4760 / 4280; complex128: 9 modes 5,
// 31 MB: 4310 / 6670; 6 modes 12, 48 MB: 5750 / 3630; 6 modes 14, 120 MB: 14150 /
// 13500); forward only (complex64: 6 modes 16, 134 MB: 2750 / 1930; 8 modes 8:
// 4640 / 2410; complex128: 6 modes 14: 3930 / 2390; 7 modes 10, 160 MB: 4850 / 5460).
bool stages_pay(const sfamd_prog* p, int kind, bool forward_only) {
  const int D = p->D;
  const int64_t mb = ipow(D, p->n) * elem_size(p->dtype) / 1000000, wide = p->dtype == SFAMD_C64 ? 1 : 2;
  // vector-ALU stages: 5 modes cutoff 13 (3 MB) 1154 / 728, cutoff 16 (8 MB) 1402 / 1813; complex128 cutoff 13
  // (6 MB) 1848 / 1337, cutoff 16 (17 MB) 3770 / 4640
  if (kind == kStepStage) return mb < (wide == 1 ? 6 : 10);
  if (forward_only) return !(D == 9 || D == 10) || mb < 64;
  if (D <= 5) return mb < 20;
  return D <= 8 || mb < 32 * wide;
}

// Stages on a density matrix against one or two passes per gate.  The adjoint
// of a stage is five launches (rows, then columns, forward again and backward)
// and holds few gates where a tile of cutoff 13 and more fills the LDS; the
// column of every mode strides over the rows of the others, so large states
// lose.  One layer of the noisy layered circuit, forward and adjoint, unfused /
// staged, us: complex64, 2 modes cutoff 8 177 / 91, 12 225 / 159, 16 313 / 259, 18
// 421 / 676; 3 modes 6 475 / 190, 8 679 / 176, 10 1167 / 668, 12 1763 / 1560, 13 2593 /
// 3319, 16 5886 / 10204; complex128, 2 modes 12 374 / 220; 3 modes 8 849 / 247, 12
// 4109 / 2633, 13 6514 / 7735.  Forward only they pay longer: 3 modes cutoff 16,
// complex64 1780 / 1356, complex128 5537 / 2387; 2 modes 20 159 / 134 and 442 / 242;
// but 3 modes 18 and 20, complex64 3858 / 4875 and 6362 / 7925.  States past the caches
// lose in complex128 where a stage's operands are mostly padding, with cutoffs 2, 3 and 5:
// adjoint, 10 modes 2 (17 MB) 7297 / 11013, 7 modes 3 11555 / 16077, 5 modes 5 14058 / 16726
// (6 modes 3, 9 MB, 2150 / 1747; 6 modes 4 30208 / 24439); forward only with cutoff 2: 10
// modes 2141 / 2228, 12 modes 33601 / 51918 (7 modes 3 3655 / 2948, 5 modes 5 4374 / 3821).
// So do cutoffs 9 and 10 (operands half padding) on 4 modes, in both types: 9, complex64 10507 /
// 12708 forward, 43263 / 52380 one gradient, complex128 16588 / 25757 forward; 10, complex64
// 19682 / 23069 (3 modes 10, 16 MB, complex128 491 / 275; 4 modes 8, 268 MB, 5991 / 3002).
bool dm_stages_pay(const sfamd_prog* p, bool forward_only) {
  const int D = p->D;
  const int64_t mb = state_mb(p, true);
  if (p->dtype == SFAMD_C128 && mb >= 12 && (D == 2 || (!forward_only && (D == 3 || D == 5)))) return false;
  if ((D == 9 || D == 10) && mb >= 64) return false;
  if (forward_only) return p->dtype == SFAMD_C128 || D <= 16 || p->n == 2;
  return D <= 12 || (D <= 16 && p->n == 2);
}

constexpr int kFewTilesModes = 4;  // modes up to which there are at most D tiles of three

// The stages of a plan for a requested number of local modes: matrix-core
// stages for three and more, vector-ALU stages for two (a beamsplitter on two
// local modes has one column, so a matrix-core operand would be 15/16 empty) and
// where the matrix-core adjoint's tiles exceed the LDS.  On a density matrix a
// stage of fewer modes has the other side's axes for columns.
//
// Circuits of R, K, D, S and BS also have vector-ALU stages, which the adjoint
// takes where operands padded to 16 rows and 4 columns waste the matrix cores (the
// share of an operand that an operator of size D fills is 0.39 at 5, 0.56 at 6, 0.42 at
// 9, 0.52 at 10, 0.63 and more at 11 to 16 and 1 at 8): at cutoff 9 (and 10 in
// complex64 on 4 and 5 modes; 6 modes have too many tiles for its LDS, 64 short stages
// take 4346 us, against 951 for one layer on the matrix cores) with three modes;
// and with two where there are at most D tiles of three modes, so that most
// compute units idle and two modes' stages have D times the workgroups.  It also
// takes them, with three modes, on complex128 states past the caches at cutoffs 5 and 6 (one
// layer, matrix cores or unfused / vector ALUs: 8 modes 6, 27 MB, 3217 / 2922; 9
// modes 5, 31 MB, 4453 / 4282; within the caches 8 modes 5, 6 MB, 1100 / 1202).  Three layers, one gradient from a graph,
// us, matrix-core / vector-ALU stages: complex64, 3 modes 8 165 / 231, 9 299 / 235, 10
// 308 / 230, 12 363 / 306, 14 527 / 299; 4 modes 8 306 / 453, 9 551 / 388, 12 603 / 591,
// 14 945 / 686; 5 modes 9 849 / 606, 10 833 / 740, 12 958 / 1259; 6 modes 9 2656 / 2030;
// complex128, 3 modes 8 197 / 234, 9 357 / 293, 12 498 / 341; 4 modes 9 623 / 497, 12
// 883 / 756, 14 1827 / 850; 5 modes 9 984 / 870, 10 989 / 1083.  4 modes 10 complex64 with
// stages of two / three modes 497 / 478, six layers 1019 / 891 (3 modes 270 / 286).
// Forward only they pay at cutoff 9 in complex64, on one tile's worth of workgroups per
// compute unit and less or on many: 4 modes, 6 layers, from a graph, matrix cores / vector
// ALUs 338 / 288, 5 modes 499 / 439, 7 modes, one layer 1789 / 1597 (6 modes 246 / 275).
Stages pick_stages(const sfamd_prog* p, bool forward_only, bool mixed) {
  const int K = p->fuse_K < p->n ? p->fuse_K : p->n;
  Stages sg{mixed, mixed ? 2 * p->n : p->n, kStepMatrixStage, K};
  if (mixed) {
    sg.Kc = p->fuse_K < 3 ? 3 : p->fuse_K < sg.axes ? p->fuse_K : sg.axes;
    if (!p->fuse_mixed || p->fuse_K < 2 || p->n < 2 || !stage_fits(p, sg, forward_only) || !dm_stages_pay(p, forward_only)) sg.Kc = 0;
    return sg;
  }
  const bool large =
      !forward_only && K >= 3 && p->dtype == SFAMD_C128 && (p->D == 5 || p->D == 6) && ipow(p->D, p->n) >= 1250000;
  bool layered = large || (K == 3 && stages_pay(p, kStepMatrixStage, forward_only) &&
                           (forward_only ? p->D == 9 && p->dtype == SFAMD_C64 && p->n != 6 : p->D > 8));
  for (const OpPlan& op : p->ops)
    layered = layered && (op.mixed_in || op.kind == SFAMD_OP_LOSS || op.kind == SFAMD_OP_MIX ||
                          fusable(op, Stages{false, p->n, kStepStage, 2}));
  if (layered) {
    const bool three = stage_three_modes(p->D, p->dtype) &&
                       (large || p->D == 9 || p->n == kFewTilesModes || p->n == kFewTilesModes + 1);
    const Stages valu{false, p->n, kStepStage, three ? 3 : 2};
    if ((three || p->n <= kFewTilesModes) && stage_fits(p, valu, false)) return valu;
  }
  if (K >= 3 && stage_fits(p, sg, forward_only)) {
    if (!stages_pay(p, kStepMatrixStage, forward_only)) sg.Kc = 0;
    return sg;
  }
  sg.kind = kStepStage;
  sg.Kc = 2;
  if (K < 2 || !stage_fits(p, sg, false) || !(p->fuse_K == 2 || stages_pay(p, kStepStage, false))) sg.Kc = 0;
  return sg;
}

void plan_program(sfamd_prog* p) {
  const Stages both[2] = {pick_stages(p, false, false), pick_stages(p, false, true)};
  plan_steps(p, both, false, &p->steps);
  const Stages fwd[2] = {pick_stages(p, true, false), pick_stages(p, true, true)};
  bool other = false;  // matrix-core stages differ (see stage_cost), vector-ALU stages only where the adjoint has none
  for (const OpPlan& op : p->ops) {
    const Stages &f = fwd[op.mixed_in], &b = both[op.mixed_in];
    // (an operation has one slot for the images of vector-ALU stages)
    other = other || (f.Kc >= 2 && fusable(op, f) && (f.kind == kStepMatrixStage || b.Kc < 2));
  }
  if (other) plan_steps(p, fwd, true, &p->fsteps);
  // state sizes at step inputs
  p->state_elems.clear();
  for (const Step& st : p->steps) {
    const OpPlan& op = p->ops[st.ops.front()];
    p->state_elems.push_back(ipow(p->D, op.mixed_in ? 2 * p->n : p->n));
  }
}

// Lay the gate table out: every operation's entry, followed by its matrix-core
// operator images (G; for a gate in a step with an adjoint G^H and dG/dp0^H
// too), then each matrix-core stage's phases as one region (the entries
// themselves in the forward-only plan, copies in the other) and the vector-ALU
// stages' images, one region per kernel.
void place_table(sfamd_prog* p) {
  p->img0.assign(p->nops, -1);
  p->img1.assign(p->nops, -1);
  p->mimg_fwd.assign(p->nops, -1);
  p->mimg_adj.assign(p->nops, -1);
  std::vector<char> in_phases(p->nops, 0);
  bool matrix = false;
  for (const std::vector<Step>* steps : {&p->steps, &p->fsteps})
    for (const Step& st : *steps) {
      if (st.kind != kStepMatrixStage) continue;
      matrix = true;
      for (int op : st.ops) {
        if (is_diag_kind(p->ops[op].kind)) {
          if (steps == &p->fsteps) in_phases[op] = 1;
          continue;
        }
        p->mimg_fwd[op] = 0;
        if (steps == &p->steps) p->mimg_adj[op] = 0;
      }
    }
  int64_t off = 0;
  for (int i = 0; i < p->nops; ++i) {
    OpPlan& op = p->ops[i];
    if (in_phases[i]) continue;
    op.off = off;
    off += table_size(op.kind, p->D);
    if (p->mimg_fwd[i] >= 0) {
      p->mimg_fwd[i] = (int32_t)off;
      off += mst_img_elems(op.kind, p->D, false);
    }
    if (p->mimg_adj[i] >= 0) {
      p->mimg_adj[i] = (int32_t)off;
      off += mst_img_elems(op.kind, p->D, true);
    }
  }
  const int32_t spare = (int32_t)off;  // readable where a kernel loads an operator that it does not use
  if (matrix) off += 2 * mst_img(p->D);
  for (Step& st : p->fsteps) {
    if (st.kind != kStepMatrixStage) continue;
    for (MArgs& a : st.margs) a.phases = (int32_t)off;
    for (int op : st.ops)
      if (in_phases[op]) {
        p->ops[op].off = off;
        off += p->D;
      }
  }
  auto place_images = [&](StageArgs& a, bool adjoint) {
    a.img_fwd = off;
    off += a.mat_fwd;
    a.img_adj = off;
    if (adjoint) off += a.mat_adj;
    for (int gi = 0; gi < a.ngates; ++gi) {
      p->img0[a.g[gi].op] = (int32_t)(a.img_fwd + a.g[gi].moff);
      if (adjoint) p->img1[a.g[gi].op] = (int32_t)(a.img_adj + a.g[gi].amoff);
    }
  };
  for (Step& st : p->steps) {
    if (st.kind == kStepStage) {
      place_images(st.args, true);
    } else if (st.kind == kStepMatrixStage) {
      for (MArgs& a : st.margs) a.phases = (int32_t)off;
      for (int op : st.ops)
        if (is_diag_kind(p->ops[op].kind)) {
          p->img0[op] = (int32_t)off;
          off += p->D;
        }
    }
  }
  // vector-ALU stages of both plans are the same
  for (Step& f : p->fsteps) {
    if (f.kind != kStepStage) continue;
    const Step* same = nullptr;
    for (const Step& st : p->steps)
      if (st.kind == kStepStage && st.op == f.op) same = &st;
    if (same)
      f.args = same->args;
    else
      place_images(f.args, false);
  }
  p->table_elems = off;
  for (std::vector<Step>* steps : {&p->steps, &p->fsteps})
    for (Step& st : *steps) {
      for (MArgs& a : st.margs) link_matrix_stage(p, a, spare);
      if (st.kind == kStepDiagRun)
        for (int g = 0; g < st.run.ngates; ++g) st.run.toff[g] = p->ops[st.run.op[g]].off;
    }
}

// one step forward, in -> dst (tmp: scratch state)
int step_forward(const sfamd_prog* p, const Step& st, const void* table, const void* in, void* dst, void* tmp,
                 hipStream_t s) {
  switch (st.kind) {
    case kStepStage: {
      const int grid = (int)(st.args.ntiles < p->nwg ? st.args.ntiles : p->nwg);
      return stage_fwd(p->D, st.K, in, dst, table, st.args, grid, p->dtype, s);
    }
    case kStepMatrixStage: {
      const MArgs& a = st.margs[0];
      const int groups = (a.ntiles + (1 << a.lgt) - 1) >> a.lgt, grid = groups < kMaxGrid ? groups : kMaxGrid;
      if (!st.mixed) return mst_fwd(p->D, st.K, in, dst, table, a, grid, p->dtype, s);
      RET_IF(mst_fwd(p->D, st.K, in, tmp, table, a, grid, p->dtype, s));
      return mst_fwd(p->D, st.K, tmp, dst, table, st.margs[1], grid, p->dtype, s);
    }
    case kStepDiagRun:
      return diag_run_fwd(in, dst, table, st.run, p->dtype, s);
    default:
      return apply_op(p->ops[st.op], p->n, p->D, table, in, dst, tmp, p->dtype, s);
  }
}

// partial columns that a step's adjoint writes, and whether only for one pass:
// stages one per workgroup
int step_columns(const sfamd_prog* p, const Step& st, bool* one_pass) {
  const bool stage = st.kind == kStepStage || st.kind == kStepMatrixStage;
  *one_pass = stage && !st.mixed;
  if (!stage) return p->nwg;
  const int nt = st.kind == kStepStage ? st.args.ntiles
                                       : (st.margs[0].ntiles + (1 << st.margs[0].lgt) - 1) >> st.margs[0].lgt;
  return nt < p->nwg ? nt : p->nwg;
}

}  // namespace

// ====================================================================== C ABI
extern "C" int sfamd_version(void) { return SFAMD_VERSION; }

extern "C" const char* sfamd_status_string(int code) {
  switch (code) {
    case 0:
      return "success";
    case SFAMD_E_ARG:
      return "invalid argument";
    case SFAMD_E_CUTOFF:
      return "cutoff dimension outside the supported range";
    case SFAMD_E_KIND:
      return "unknown operation kind";
    case SFAMD_E_STATE:
      return "operation not valid for this state representation";
    case SFAMD_E_WORKSPACE:
      return "workspace missing or too small";
    default:
      break;
  }
  if (code > 0) return hipGetErrorString((hipError_t)code);
  return "unknown status";
}

extern "C" int64_t sfamd_gate_table_size(int kind, int D) {
  if (D < 1 || D > SFAMD_MAX_CUTOFF) return -1;
  if (kind < 0 || kind > SFAMD_OP_CUBIC_PHASE) return -1;
  if (two_mode_kind(kind) && D > SFAMD_MAX_CUTOFF_BS) return -1;
  if (kind == SFAMD_OP_CUBIC_PHASE && D > SFAMD_MAX_CUTOFF_V) return -1;
  return table_size(kind, D);
}

extern "C" int sfamd_build_gate(int kind, double p0, double p1, int D, int dtype, void* out, void* stream) {
  CHECK_ARG(out && (dtype == SFAMD_C64 || dtype == SFAMD_C128));
  RET_IF(validate_op(kind, 0, 1, 2, D));
  if (kind == SFAMD_OP_MIX) return SFAMD_E_KIND;
  BuildBatch b;
  b.first = -1;
  b.p0 = p0;
  b.p1 = p1;
  b.d[0].kind = kind;
  b.d[0].off = 0;
  b.d[0].img0 = b.d[0].img1 = -1;
  return launch_build(b, 1, D, nullptr, out, dtype, (hipStream_t)stream);
}

extern "C" int sfamd_apply_1mode(int kind, const void* in, void* out, void* tmp, int n, int D, int mode, int mixed,
                                 const void* table, int dtype, void* stream) {
  CHECK_ARG(in && out && table && in != out && n >= 1);
  CHECK_ARG(dtype == SFAMD_C64 || dtype == SFAMD_C128);
  if (kind != SFAMD_OP_ROTATION && kind != SFAMD_OP_KERR && kind != SFAMD_OP_DISPLACEMENT &&
      kind != SFAMD_OP_SQUEEZE && kind != SFAMD_OP_CUBIC_PHASE)
    return SFAMD_E_KIND;
  RET_IF(validate_op(kind, mode, -1, n, D));
  OpPlan op{kind, mode, -1, mixed ? 1 : 0, 0, 0};
  return apply_op(op, n, D, table, in, out, tmp, dtype, (hipStream_t)stream);
}

extern "C" int sfamd_apply_matrix(const void* in, void* out, void* tmp, int n, int D, int mode, int mixed,
                                  const void* U, int dtype, void* stream) {
  CHECK_ARG(in && out && U && in != out && n >= 1);
  CHECK_ARG(dtype == SFAMD_C64 || dtype == SFAMD_C128);
  RET_IF(validate_op(SFAMD_OP_DISPLACEMENT, mode, -1, n, D));
  // the dense single-mode path reads only the leading D x D matrix of a table
  OpPlan op{SFAMD_OP_DISPLACEMENT, mode, -1, mixed ? 1 : 0, 0, 0};
  return apply_op(op, n, D, U, in, out, tmp, dtype, (hipStream_t)stream);
}

extern "C" int sfamd_apply_bs(const void* in, void* out, void* tmp, int n, int D, int mode1, int mode2, int mixed,
                              const void* table, int dtype, void* stream) {
  CHECK_ARG(in && out && table && in != out && n >= 2);
  CHECK_ARG(dtype == SFAMD_C64 || dtype == SFAMD_C128);
  RET_IF(validate_op(SFAMD_OP_BEAMSPLITTER, mode1, mode2, n, D));
  OpPlan op{SFAMD_OP_BEAMSPLITTER, mode1, mode2, mixed ? 1 : 0, 0, 0};
  return apply_op(op, n, D, table, in, out, tmp, dtype, (hipStream_t)stream);
}

extern "C" int sfamd_apply_2mode(int kind, const void* in, void* out, void* tmp, int n, int D, int mode1, int mode2,
                                 int mixed, const void* table, int dtype, void* stream) {
  CHECK_ARG(in && out && table && in != out && n >= 2);
  CHECK_ARG(dtype == SFAMD_C64 || dtype == SFAMD_C128);
  if (!two_mode_kind(kind)) return SFAMD_E_KIND;
  RET_IF(validate_op(kind, mode1, mode2, n, D));
  OpPlan op{kind, mode1, mode2, mixed ? 1 : 0, 0, 0};
  return apply_op(op, n, D, table, in, out, tmp, dtype, (hipStream_t)stream);
}

extern "C" int sfamd_apply_loss(const void* in, void* out, int n, int D, int mode, const void* table, int dtype,
                                void* stream) {
  CHECK_ARG(in && out && table && in != out && n >= 1);
  CHECK_ARG(dtype == SFAMD_C64 || dtype == SFAMD_C128);
  RET_IF(validate_op(SFAMD_OP_LOSS, mode, -1, n, D));
  OpPlan op{SFAMD_OP_LOSS, mode, -1, 1, 0, 0};
  return apply_op(op, n, D, table, in, out, nullptr, dtype, (hipStream_t)stream);
}

extern "C" int sfamd_mix(const void* ket, void* dm, int n, int D, int dtype, void* stream) {
  CHECK_ARG(ket && dm && n >= 1 && D >= 1);
  CHECK_ARG(dtype == SFAMD_C64 || dtype == SFAMD_C128);
  return mix_fwd(ket, dm, n, D, dtype, (hipStream_t)stream);
}

extern "C" int sfamd_replace_mode(const void* in, void* out, int n, int D, int mode, const void* sigma, int dtype,
                                  void* stream) {
  CHECK_ARG(in && out && sigma && in != out && n >= 1 && D >= 1 && mode >= 0 && mode < n);
  CHECK_ARG(dtype == SFAMD_C64 || dtype == SFAMD_C128);
  return replace_mode(in, out, ipow(D, 2 * n), D, bra_stride_dm(n, D, mode), ket_stride_dm(n, D, mode), sigma, dtype,
                      (hipStream_t)stream);
}

// ---------------------------------------------------------------- programs
static int create_program(const sfamd_op_t* ops, int nops, int n, int D, int mixed_in, int dtype, int fuse_K,
                          std::unique_ptr<sfamd_prog>* out) {
  std::unique_ptr<sfamd_prog> p(new sfamd_prog());
  p->n = n;
  p->D = D;
  p->dtype = dtype;
  p->mixed_in = mixed_in ? 1 : 0;
  p->nops = nops;
  // negative: none, as zero
  p->fuse_K = fuse_K < 0 ? 0 : fuse_K & ~(SFAMD_FUSE_MIXED | SFAMD_FUSE_PAYING);
  p->fuse_mixed = fuse_K >= 0 && (fuse_K & SFAMD_FUSE_MIXED) != 0;
  p->fuse_paying = fuse_K >= 0 && (fuse_K & SFAMD_FUSE_PAYING) != 0;
  int mixed = p->mixed_in;
  int64_t max_state = ipow(D, mixed ? 2 * n : n);
  for (int i = 0; i < nops; ++i) {
    const int st = validate_op(ops[i].kind, ops[i].mode0, ops[i].mode1, n, D);
    if (st != 0) return st;
    OpPlan op{ops[i].kind, ops[i].mode0, ops[i].mode1, mixed, 0, 0};
    if (op.kind == SFAMD_OP_MIX && mixed) return SFAMD_E_STATE;
    if (op.kind == SFAMD_OP_LOSS && !mixed) op.mix_first = 1;
    if (op.kind == SFAMD_OP_LOSS || op.kind == SFAMD_OP_MIX) mixed = 1;
    p->ops.push_back(op);
    const int64_t se = ipow(D, mixed ? 2 * n : n);
    if (se > max_state) max_state = se;
    // a two-pass op on a DM and a pure->mixed loss need DM-sized scratch
    if (op.mix_first) max_state = ipow(D, 2 * n) > max_state ? ipow(D, 2 * n) : max_state;
  }
  p->max_state = max_state;
  p->final_mixed = mixed;
  plan_program(p.get());
  place_table(p.get());
  p->state_elems.push_back(ipow(D, mixed ? 2 * n : n));
  int64_t nwg = (max_state + kBlock - 1) / kBlock;
  // and a workgroup for every tile of a stage (6 modes, cutoff 4, one stage of 8 gates: 256 amplitudes
  // for each of 16 workgroups against one tile for each of 64, adjoint launch and reduction 38 -> 14 us)
  for (const Step& st : p->steps) {
    bool one_pass;
    p->nwg = 4096;
    const int64_t groups = st.kind == kStepStage || st.kind == kStepMatrixStage ? step_columns(p.get(), st, &one_pass) : 0;
    if (groups > nwg) nwg = groups;
  }
  if (nwg > 4096) nwg = 4096;
  if (nwg < 1) nwg = 1;
  p->nwg = (int)nwg;
  *out = std::move(p);
  return 0;
}

extern "C" int sfamd_prog_create(const sfamd_op_t* ops, int nops, int n, int D, int mixed_in, int dtype, int fuse_K,
                                 sfamd_prog_t** out) {
  CHECK_ARG(out && nops >= 0 && n >= 1 && n <= 32 && (ops || nops == 0));
  CHECK_ARG(dtype == SFAMD_C64 || dtype == SFAMD_C128);
  if (D < 1 || D > SFAMD_MAX_CUTOFF) return SFAMD_E_CUTOFF;
  try {
    std::unique_ptr<sfamd_prog> p;
    RET_IF(create_program(ops, nops, n, D, mixed_in, dtype, fuse_K, &p));
    *out = p.release();
    return 0;
  } catch (const std::exception&) {  // out of host memory
    return SFAMD_E_ARG;
  }
}

extern "C" int sfamd_prog_info(const sfamd_prog_t* p, sfamd_prog_info_t* info) {
  CHECK_ARG(p && info);
  info->table_elems = p->table_elems;
  info->partial_doubles = (int64_t)p->nops * 4 * p->nwg;
  info->ws_elems = 4 * p->max_state;
  info->final_elems = p->state_elems.back();
  info->final_mixed = p->final_mixed;
  info->nops = p->nops;
  info->nsteps = (int32_t)p->steps.size();
  return 0;
}

extern "C" int64_t sfamd_prog_state_elems(const sfamd_prog_t* p, int i) {
  if (!p || i < 0 || i > (int)p->steps.size()) return -1;
  return p->state_elems[i];
}

extern "C" int sfamd_prog_step_ops(const sfamd_prog_t* p, int step, int32_t* ops_out, int cap) {
  if (!p || step < 0 || step >= (int)p->steps.size()) return SFAMD_E_ARG;
  const Step& st = p->steps[step];
  for (int i = 0; i < (int)st.ops.size() && i < cap; ++i) ops_out[i] = st.ops[i];
  return (int)st.ops.size();
}

extern "C" int sfamd_prog_step_kind(const sfamd_prog_t* p, int forward_only, int step) {
  if (!p) return SFAMD_E_ARG;
  const std::vector<Step>& steps = forward_only && !p->fsteps.empty() ? p->fsteps : p->steps;
  return step < 0 || step >= (int)steps.size() ? SFAMD_E_ARG : steps[step].kind;
}

extern "C" int sfamd_prog_destroy(sfamd_prog_t* p) {
  delete p;
  return 0;
}

extern "C" int sfamd_prog_build_table(const sfamd_prog_t* p, const double* params, void* table, void* stream) {
  CHECK_ARG(p && (p->nops == 0 || (params && table)));
  CHECK_ARG(p->table_elems < ((int64_t)1 << 31));
  BuildBatch b;
  b.p0 = b.p1 = 0.0;
  for (int first = 0; first < p->nops; first += kMaxBuildPerLaunch) {
    const int cnt = p->nops - first < kMaxBuildPerLaunch ? p->nops - first : kMaxBuildPerLaunch;
    b.first = first;
    for (int i = 0; i < cnt; ++i) {
      const int op = first + i;
      b.d[i].kind = p->ops[op].kind |  // MIX entries build nothing
                    (p->mimg_fwd[op] >= 0 ? kBuildMatrixFwd : 0) | (p->mimg_adj[op] >= 0 ? kBuildMatrixAdj : 0);
      b.d[i].off = (int32_t)p->ops[first + i].off;
      b.d[i].img0 = p->img0[op];
      b.d[i].img1 = p->img1[op];
    }
    RET_IF(launch_build(b, cnt, p->D, params, table, p->dtype, (hipStream_t)stream));
  }
  return 0;
}

extern "C" int sfamd_prog_forward(const sfamd_prog_t* p, int begin, int end, const void* table, const void* in,
                                  void* out, void* const* saved, void* ws, void* stream) {
  const int nsteps = p ? (int)p->steps.size() : 0;
  CHECK_ARG(p && in && out && in != out && 0 <= begin && begin <= end && end <= nsteps);
  CHECK_ARG(ws || begin == end);
  hipStream_t s = (hipStream_t)stream;
  const int64_t esz = elem_size(p->dtype);
  char* A = (char*)ws;
  char* B = A + p->max_state * esz;
  char* Ct = B + p->max_state * esz;
  if (begin == end) {
    HIP_RET(hipMemcpyAsync(out, in, p->state_elems[begin] * esz, hipMemcpyDeviceToDevice, s));
    return 0;
  }
  const void* cur = in;
  if (saved && saved[0] && saved[0] != in)
    HIP_RET(hipMemcpyAsync(saved[0], in, p->state_elems[begin] * esz, hipMemcpyDeviceToDevice, s));
  for (int i = begin; i < end; ++i) {
    void* dst;
    if (i == end - 1)
      dst = out;
    else if (saved && saved[i + 1 - begin])
      dst = saved[i + 1 - begin];
    else
      dst = (cur == A) ? B : A;
    if (dst == cur) return SFAMD_E_ARG;
    RET_IF(step_forward(p, p->steps[i], table, cur, dst, Ct, s));
    cur = dst;
  }
  return 0;
}

extern "C" int sfamd_prog_run(const sfamd_prog_t* p, const void* table, const void* in, void* out, void* ws,
                              void* stream) {
  CHECK_ARG(p);
  if (p->fsteps.empty())
    return sfamd_prog_forward(p, 0, (int)p->steps.size(), table, in, out, nullptr, ws, stream);
  CHECK_ARG(in && out && in != out && ws);
  char* A = (char*)ws;
  char* B = A + p->max_state * elem_size(p->dtype);
  char* Ct = B + p->max_state * elem_size(p->dtype);
  const void* cur = in;
  for (size_t i = 0; i < p->fsteps.size(); ++i) {
    void* dst = i + 1 == p->fsteps.size() ? out : (cur == A ? (void*)B : (void*)A);
    RET_IF(step_forward(p, p->fsteps[i], table, cur, dst, Ct, (hipStream_t)stream));
    cur = dst;
  }
  return 0;
}

extern "C" int sfamd_prog_adjoint(const sfamd_prog_t* p, int begin, int end, const void* table, void* const* saved,
                                  const void* g_out, void* g_in, double* grads, double* partial, void* ws,
                                  void* stream) {
  const int nsteps = p ? (int)p->steps.size() : 0;
  CHECK_ARG(p && saved && g_out && g_in && grads && partial && ws && g_in != g_out);
  CHECK_ARG(0 <= begin && begin < end && end <= nsteps);
  hipStream_t s = (hipStream_t)stream;
  const int64_t esz = elem_size(p->dtype);
  char* LA = (char*)ws;
  char* LB = LA + p->max_state * esz;
  char* T1 = LB + p->max_state * esz;
  char* T2 = T1 + p->max_state * esz;
  const int nwg = p->nwg;
  // every adjoint launch writes its operation's whole [pass][slot][nwg]
  // partial block, so nothing needs clearing between calls
  const void* lam = g_out;
  for (int i = end - 1; i >= begin; --i) {
    if (!saved[i - begin]) return SFAMD_E_ARG;
    void* dst = (i == begin) ? g_in : ((lam == LA) ? LB : LA);
    const Step& st = p->steps[i];
    bool one_pass;
    const int ncol = step_columns(p, st, &one_pass);
    if (st.kind == kStepStage) {
      RET_IF(stage_adj(p->D, st.K, saved[i - begin], lam, dst, table, st.args, ncol, partial, nwg, p->dtype, s));
    } else if (st.kind == kStepMatrixStage) {
      const void *psi = saved[i - begin], *lo = lam;
      if (st.mixed) {  // the rows again, the columns backward, the rows backward
        RET_IF(mst_fwd(p->D, st.K, psi, T1, table, st.margs[0], ncol, p->dtype, s));
        RET_IF(mst_adj(p->D, st.K, T1, lam, T2, table, st.margs[1], ncol, partial, nwg, p->dtype, s));
        lo = T2;
      }
      RET_IF(mst_adj(p->D, st.K, psi, lo, dst, table, st.margs[0], ncol, partial, nwg, p->dtype, s));
    } else if (st.kind == kStepDiagRun) {
      RET_IF(diag_run_adj(saved[i - begin], lam, dst, table, st.run, partial, nwg, p->dtype, s));
    } else {
      RET_IF(adjoint_op(p->ops[st.op], p->n, p->D, table, saved[i - begin], lam, dst, T1, T2,
                        partial + (int64_t)st.op * 4 * nwg, nwg, p->dtype, s));
    }
    lam = dst;
  }
  // gradients of the operations of these steps, one launch per OpList chunk
  OpList ol;
  ol.n = 0;
  for (int i = begin; i < end; ++i) {
    const Step& st = p->steps[i];
    bool one_pass;
    const int ncol = step_columns(p, st, &one_pass);
    for (int op : st.ops) {
      ol.cols[ol.n] = (uint16_t)(one_pass ? ((unsigned)ncol | kOpColsOnePass) : (unsigned)ncol);
      ol.ops[ol.n++] = op;
      if (ol.n == kOpListMax) {
        RET_IF(reduce_grads(partial, grads, ol, nwg, s));
        ol.n = 0;
      }
    }
  }
  return reduce_grads(partial, grads, ol, nwg, s);
}

// ---------------------------------------------------------------- graphs
extern "C" int sfamd_graph_begin(void* stream) {
  CHECK_ARG(stream);
  HIP_RET(hipStreamBeginCapture((hipStream_t)stream, hipStreamCaptureModeThreadLocal));
  return 0;
}

extern "C" int sfamd_graph_end(void* stream, void** graph_exec) {
  CHECK_ARG(stream && graph_exec);
  hipGraph_t g = nullptr;
  HIP_RET(hipStreamEndCapture((hipStream_t)stream, &g));
  hipGraphExec_t ex = nullptr;
  const hipError_t e = hipGraphInstantiate(&ex, g, nullptr, nullptr, 0);
  (void)hipGraphDestroy(g);
  HIP_RET(e);
  *graph_exec = (void*)ex;
  return 0;
}

extern "C" int sfamd_graph_launch(void* graph_exec, void* stream) {
  CHECK_ARG(graph_exec);
  HIP_RET(hipGraphLaunch((hipGraphExec_t)graph_exec, (hipStream_t)stream));
  return 0;
}

extern "C" int sfamd_graph_destroy(void* graph_exec) {
  if (!graph_exec) return 0;
  HIP_RET(hipGraphExecDestroy((hipGraphExec_t)graph_exec));
  return 0;
}
