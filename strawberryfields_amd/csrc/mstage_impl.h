// Fused gate stages with the gates on matrix cores: many gates per pass over a
// ket, or over a density matrix on one side.
//
// A stage is a set of K "local" modes and an ordered list of gates that act
// only on those modes (R, K, D, S, V on one local mode; BS, MZ, S2, CK on two).  The ket is
// cut into tiles of the D^K amplitudes of the local modes for one assignment
// of the other modes' digits.  A workgroup loads a tile into LDS, applies every
// gate of the stage there and writes the tile back, so a stage costs one read
// and one write of the state however many gates it holds.
//
// What bounds it: one output amplitude per thread on the vector ALUs (the
// kernels this replaces for K >= 3) reads D amplitudes and D matrix entries
// from LDS per gate, 16 D bytes per amplitude, so LDS bandwidth bounds the
// gates and the staged matrices eat the LDS that further gates need.  Here a
// gate is a small GEMM on v_mfma_*_16x16x4 in real form (mfma_ops.h has the
// register plan): a wave applies one D x D operator to 16 fibers ("columns")
// and each amplitude is read from and written to LDS once per gate.  A
// dense gate is one operator on the D^(K-1) fibers of its axis; a beamsplitter
// is D operators, one per modular anti-diagonal {(k, (p - k) mod D)} of its
// two axes (the photon-number blocks s = p and s = p + D side by side), on the
// D^(K-2) positions of the other local axes; S2 has the diagonals
// {(k, (k + p) mod D)} instead, with its difference blocks -p and D - p.  MZ and CK
// are applied like beamsplitters.  A fiber belongs to one wave, so gates work in
// place with one barrier per gate.
//
// The operators are not staged in LDS: the table build writes them in lane
// order (complex entries, each shared by the two lanes holding its real and
// imaginary rows), and a wave loads its next operator from the gate table
// (cache resident) while it applies the current one.  LDS holds amplitudes
// only, in axis strides padded to odd numbers against bank conflicts.
//
// The adjoint of a stage loads the stage's input tile and the incoming
// cotangent tile, recomputes the stage forward keeping the input tile of every
// gate with operators, and runs the gates backward: lam_in = G^H lam_out,
// mu = dG/dp0^H lam_out, g0 = Re conj(mu) psi_in, and the phase parameter from
// dG/dp1 = i (wa n + wb N) G with the (first) mode's digit n before and N after
// the gate (D: -1, 1; S: -1/2, 1/2; BS: 1, -1; MZ: 1, 0; S2: -1, 1):
//   g1 = -sum_k k [wa Im conj(lam_in[k]) psi_in[k] + wb Im conj(lam_out[k]) psi_out[k]].
// Rotation and Kerr gates multiply in place and take no tile: the backward
// sweep multiplies the state by the conjugate phases again.  Products are
// formed in the state's precision (a rotation's or Kerr gate's in double), the
// difference in g1 per amplitude, and everything past a lane's few amplitudes
// of one fiber is summed in double: per lane, per wave by lane moves and per
// workgroup in a fixed order (deterministic), one partial per workgroup.
//
// A density matrix is a ket of 2 n axes: a launch on row axes applies the gates,
// one on column axes (`side`) their conjugates, as G on the conjugated tile,
// so both read the same operators.
#pragma once

#include "mstage.h"
#include "stage_common.h"

namespace {

template <typename T>
using C = cpx<T>;

// the matrix-core instruction of a precision: v_mfma_{f32_16x16x4f32,
// f64_16x16x4f64}.  Lane l = 16 g + c supplies A[c][g] and B[g][c] and receives
// rows r(g, j), j = 0..3, of column c: 4 g + j in single, 4 j + g in double
// precision.  Row r belongs to the lane group and slot whose accumulator holds
// it: slot pair index rp(r) = 2 group + slot (slot: j / 2) and part j % 2
// (0: real, 1: imaginary).
template <typename T>
struct Mx;
template <>
struct Mx<float> {
  typedef float acc4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ acc4 mma(float a, float b, acc4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int rp(int c) { return c >> 1; }
  static __device__ __forceinline__ int part(int c) { return c & 1; }
};
template <>
struct Mx<double> {
  typedef double acc4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ acc4 mma(double a, double b, acc4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int rp(int c) { return ((c & 3) << 1) | (c >> 3); }
  static __device__ __forceinline__ int part(int c) { return (c >> 2) & 1; }
};

// wave of the workgroup, known to be uniform
__device__ __forceinline__ int wave_index() { return __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6); }

// a tile group of 2^LG tiles worked on by NW waves
template <int D_, int K_, int LG_, int NW_>
struct Geo {
  static constexpr int D = D_, K = K_, LG = LG_, NW = NW_, NT = 64 * NW_, TT = 1 << LG_;
  static constexpr int DK = sfamd::mst_tile(D, K);
  static constexpr int TS = sfamd::mst_tile_lds(D, K);  // LDS amplitudes of a tile
  static constexpr int GS = TS * TT;                    // and of the group
  static constexpr int P = sfamd::mst_p(D), MB = sfamd::mst_mb(D), NE = P * MB, IMG = sfamd::mst_img(D);
  static constexpr int items(bool two) { return sfamd::mst_items(D, K, LG, two); }
  static constexpr int per_wave(bool two) { return (items(two) + NW - 1) / NW; }
  static constexpr int cols(bool two) { return (two ? DK / (D * D) : DK / D) * TT; }
};

// x / D for x < 2^13 (D <= 20: the rounding error of the reciprocal stays
// below 1 / D), two full-rate instructions
template <int D>
__device__ __forceinline__ unsigned div_d(unsigned x) {
  constexpr unsigned M = ((1u << 20) + D - 1) / D;
  return __umul24(x, M) >> 20;
}

// The thread's elements of a tile group: a fixed position on the K - 1 inner
// axes and in the group (thread i: tile i mod TT), and every W-th digit of
// axis 0, so that index arithmetic runs once per kernel and an element costs
// an addition.  The accesses to the group's tiles of one element are
// contiguous when the last mode is not local.
template <typename T, typename Gm>
struct Walk {
  static constexpr int D = Gm::D, K = Gm::K;
  static constexpr int I = Gm::DK / D;                 // inner positions
  static constexpr int W = (Gm::NT >> Gm::LG) / I;     // digits of axis 0 at once
  static constexpr int PER = (D + W - 1) / W;          // elements per thread
  static constexpr int S0 = sfamd::mst_stride(D, K, 0);
  static constexpr bool kAll = W * I == (Gm::NT >> Gm::LG);  // every thread has elements
  int tt, d0, lds;     // tile of the group, first digit of axis 0, LDS offset at digit 0
  bool mine;           // the thread has elements (the others read element 0 and store nothing)
  unsigned digits;     // inner digits, axis t at bit 5 t
  int64_t goff, base, s0;
  T im;                // sign of the imaginary parts: conj(G) x = conj(G conj(x))
  bool valid;          // the group's tile exists and the thread has elements

  __device__ __forceinline__ explicit Walk(const sfamd::MArgs& a)
      : base(0), s0(a.loc_stride[0]), im(a.side ? (T)-1 : (T)1), valid(true) {
    tt = (int)threadIdx.x & (Gm::TT - 1);
    const unsigned i = threadIdx.x >> Gm::LG;
    d0 = (int)(i / I);
    unsigned r = i - d0 * I;
    mine = kAll || d0 < W;
    if (!mine) d0 = 0;
    lds = tt * Gm::TS;
    goff = 0;
    digits = 0;
#pragma unroll
    for (int t = K - 1; t >= 1; --t) {
      const unsigned q = div_d<D>(r), d = r - q * D;
      lds += (int)d * sfamd::mst_stride(D, K, t);
      goff += (int64_t)d * a.loc_stride[t];
      digits |= d << (5 * t);
      r = q;
    }
  }
  // move to a tile group
  __device__ __forceinline__ void at(int group, const sfamd::MArgs& a) {
    unsigned t = ((unsigned)group << Gm::LG) + (Gm::LG ? tt : 0);
    valid = (int)t < a.ntiles && mine;
    if ((int)t >= a.ntiles) t = 0;
    base = goff;
    int64_t st[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) st[u] = a.nl_stride[u];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const unsigned q = t / D;
      base += (int64_t)(t - q * D) * st[u];
      t = q;
    }
    for (int u = 4; u < a.nnl; ++u) {
      const unsigned q = t / D;
      base += (int64_t)(t - q * D) * a.nl_stride[u];
      t = q;
    }
  }
  // every element of the thread: f(axis-0 digit, LDS offset)
  template <typename F>
  __device__ __forceinline__ void each(F f) const {
    if (!mine) return;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int d = d0 + j * W;
      if ((j + 1) * W <= D || d < D) f(d, lds + d * S0);
    }
  }
  // all of the thread's loads in flight (digit clamped), then the LDS stores
  __device__ __forceinline__ void fetch(const C<T>* __restrict__ src, C<T> (&v)[PER]) const {
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int d = d0 + j * W;
      v[j] = src[base + (int64_t)((j + 1) * W <= D || d < D ? d : 0) * s0];
    }
  }
  __device__ __forceinline__ void put(const C<T> (&v)[PER], C<T>* tile) const {
    if (!mine) return;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int d = d0 + j * W;
      if ((j + 1) * W <= D || d < D) tile[lds + d * S0] = mk<T>(v[j].re, im * v[j].im);
    }
  }
  __device__ __forceinline__ void store(const C<T>* tile, C<T>* __restrict__ dst) const {
    if (valid) each([&](int d, int o) { dst[base + (int64_t)d * s0] = mk<T>(tile[o].re, im * tile[o].im); });
  }
  // The group's tiles to a state whose mode order may differ: the same walk
  // over the tile axes in the output's order, so that neighbouring threads
  // write neighbouring amplitudes along the output's fastest local mode.
  __device__ __forceinline__ void store_permuted(int group, const sfamd::MArgs& a, const C<T>* tile,
                                                 C<T>* __restrict__ dst) const {
    unsigned t = ((unsigned)group << Gm::LG) + (Gm::LG ? tt : 0);
    if ((int)t >= a.ntiles || !mine) return;
    unsigned r = (threadIdx.x >> Gm::LG) - d0 * I;
    int64_t to = 0;
    int o = tt * Gm::TS;
#pragma unroll
    for (int u = K - 1; u >= 1; --u) {
      const unsigned q = div_d<D>(r), d = r - q * D;
      o += (int)__umul24(d, a.out_lds[u]);
      to += (int64_t)d * a.out_stride[u];
      r = q;
    }
    for (int u = 0; u < a.nnl; ++u) {
      const unsigned q = t / D;
      to += (int64_t)(t - q * D) * a.out_nl_stride[u];
      t = q;
    }
    const int64_t g0 = a.out_stride[0];
    const int l0 = a.out_lds[0];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int d = d0 + j * W;
      if ((j + 1) * W <= D || d < D) dst[to + (int64_t)d * g0] = tile[o + d * l0];
    }
  }
};

// ---- operators ------------------------------------------------------------
// this lane's entries of the operator image at img: entry (mb, t) of the lane
// is row group rp(c) / 2's amplitude 2 mb + rp(c) % 2, column group g's
// amplitude t
template <typename T, typename Gm>
__device__ __forceinline__ void load_image(const C<T>* __restrict__ img, C<T> (&v)[Gm::NE]) {
  const unsigned lane = threadIdx.x & 63;
  const unsigned off = (lane >> 4) * 8 + Mx<T>::rp(lane & 15);
#pragma unroll
  for (int i = 0; i < Gm::NE; ++i) v[i] = img[off + i * 32];
}

// acc = operator x for this lane's column (x: the lane group's P amplitudes)
template <typename T, typename Gm>
__device__ __forceinline__ void apply_image(const C<T> (&v)[Gm::NE], const C<T> (&x)[Gm::P],
                                            typename Mx<T>::acc4 (&acc)[Gm::MB]) {
  const int part = Mx<T>::part(threadIdx.x & 15);
#pragma unroll
  for (int mb = 0; mb < Gm::MB; ++mb) acc[mb] = typename Mx<T>::acc4{(T)0, (T)0, (T)0, (T)0};
#pragma unroll
  for (int t = 0; t < Gm::P; ++t) {
#pragma unroll
    for (int mb = 0; mb < Gm::MB; ++mb) {
      const C<T> e = v[mb * Gm::P + t];
      acc[mb] = Mx<T>::mma(part ? e.im : e.re, x[t].re, acc[mb]);
    }
#pragma unroll
    for (int mb = 0; mb < Gm::MB; ++mb) {
      const C<T> e = v[mb * Gm::P + t];
      acc[mb] = Mx<T>::mma(part ? e.re : -e.im, x[t].im, acc[mb]);
    }
  }
}

// the lane group's amplitude q from the accumulators
template <typename T, int MB>
__device__ __forceinline__ C<T> acc_amp(const typename Mx<T>::acc4 (&acc)[MB], int q) {
  const typename Mx<T>::acc4 v = acc[q >> 1];
  return (q & 1) ? mk<T>(v[2], v[3]) : mk<T>(v[0], v[1]);
}

// ---- one gate -------------------------------------------------------------
using Gate = sfamd::MGate;

// Touch every gate's descriptor while the tile loads are in flight: read at
// their first use, the 64-byte lines cost a cache miss in each gate's chain
// (6 modes, cutoff 8, complex64: forward stages 7.2 -> 6.3 us on average).
template <typename Gm>
__device__ __forceinline__ void warm_gates(const sfamd::MArgs& a) {
  int x = 0;
  for (int gi = wave_index(); gi < a.ngates; gi += Gm::NW) x |= a.g[gi].kind;
  if (a.permuted) x |= a.out_lds[0] | (int)a.out_nl_stride[0];
  __asm__ volatile("" ::"s"(x));
}

// The lane's place in item `item` (block * operators + operator) of a gate:
// the LDS offset of its column's amplitude k = grp P + q is lo + q ds, plus
// `wrap` where the second digit, (p - k) mod D or for S2 (k + p) mod D, wraps
// around.
// Slots past amplitude D - 1 (in the last lane groups) read amplitude D - 1,
// which the operators' zero columns and a zero weight in the parameter sums
// leave out (zeros selected after each read cost 2 vector instructions per
// amplitude: 3 modes, cutoff 9, density matrix, complex128 1797 -> 1759 us).  Everything but the gate's strides is the same for all gates,
// so the compiler computes it once per kernel.
template <typename Gm, bool TWO>
struct Place {
  static constexpr int D = Gm::D, P = Gm::P;
  int base, lo, ds, wrap, p, last;  // last: amplitude from whose successor on the second digit wraps
  bool valid;
  __device__ __forceinline__ Place(int item, const Gate& g) {
    const int lane = threadIdx.x & 63;
    const int blk = TWO ? item / D : item;
    p = TWO ? item - blk * D : 0;
    constexpr int NC = Gm::cols(TWO), NCX = TWO ? Gm::K - 2 : Gm::K - 1;
    unsigned f = blk * 16 + (lane & 15);
    valid = NC % 16 == 0 || f < NC;
    if (!valid) f = NC - 1;
    ds = g.ds;
    wrap = g.wrap;
    last = TWO ? (p ^ g.a0) + (g.a0 & D) : 0;  // p, or D - 1 - p where the difference is conserved
    base = p * g.l1;
#pragma unroll
    for (int u = NCX - 1; u >= 0; --u) {
      const unsigned q = div_d<D>(f);
      base += (int)__umul24(f - q * D, g.cs[u]);
      f = q;
    }
    if (Gm::LG) base += (int)(f * Gm::TS);
    lo = base + __mul24((lane >> 4) * P, ds);
  }
  __device__ __forceinline__ int grp() const { return (threadIdx.x & 63) >> 4; }
  __device__ __forceinline__ bool has(int q) const { return 3 * P + q < D || grp() * P + q < D; }
  __device__ __forceinline__ int at(int q) const {
    if (3 * P + q < D) return lo + q * ds + (TWO && grp() * P + q > last ? wrap : 0);
    const int k = grp() * P + q < D ? grp() * P + q : D - 1;
    return base + k * ds + (TWO && k > last ? wrap : 0);
  }
};

template <typename T, typename Gm, bool TWO>
__device__ __forceinline__ void read_fiber(const C<T>* tile, const Place<Gm, TWO>& pl, C<T> (&x)[Gm::P]) {
#pragma unroll
  for (int q = 0; q < Gm::P; ++q) x[q] = tile[pl.at(q)];
}

template <typename T, typename Gm, bool TWO>
__device__ __forceinline__ void write_fiber(C<T>* tile, const Place<Gm, TWO>& pl,
                                            const typename Mx<T>::acc4 (&acc)[Gm::MB]) {
  if (!pl.valid) return;
#pragma unroll
  for (int q = 0; q < Gm::P; ++q)
    if (pl.has(q)) tile[pl.at(q)] = acc_amp<T>(acc, q);
}

// a wave's first operator of the gate whose image starts at table + off
template <typename T, typename Gm>
__device__ __forceinline__ const C<T>* first_image(const C<T>* table, int off, bool two) {
  return table + off + (two ? wave_index() % Gm::D * Gm::IMG : 0);
}

// One gate with operators forward, src -> dst (the same tile: in place).
// `op` holds the wave's first operator.
template <typename T, typename Gm, bool TWO>
__device__ __forceinline__ void heavy_fwd(const Gate& g, const C<T>* __restrict__ table, const C<T>* src,
                                          C<T>* dst, const C<T> (&op)[Gm::NE]) {
  constexpr int N = Gm::items(TWO), J = Gm::per_wave(TWO);
  // a beamsplitter's later items take other operators unless the waves are a
  // multiple of the operators
  constexpr bool kReload = TWO && J > 1 && Gm::NW % Gm::D != 0;
  const int wave = wave_index();
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int item = wave + j * Gm::NW;
    if ((j + 1) * Gm::NW <= N || item < N) {
      const Place<Gm, TWO> pl(item, g);
      C<T> x[Gm::P];
      typename Mx<T>::acc4 acc[Gm::MB];
      if (kReload && j > 0) {
        C<T> other[Gm::NE];
        load_image<T, Gm>(table + g.fwd + pl.p * Gm::IMG, other);
        read_fiber<T, Gm, TWO>(src, pl, x);
        apply_image<T, Gm>(other, x, acc);
      } else {
        read_fiber<T, Gm, TWO>(src, pl, x);
        apply_image<T, Gm>(op, x, acc);
      }
      write_fiber<T, Gm, TWO>(dst, pl, acc);
    }
  }
}

// rotation or Kerr gate on the thread's elements, in place (ph: its phases in LDS)
template <typename T, typename Gm>
__device__ __forceinline__ void diag_fwd(const Gate& g, const Walk<T, Gm>& wk, const C<T>* ph, C<T>* tile) {
  if (g.a0 == 0) {
    wk.each([&](int d, int o) { tile[o] = cmul(ph[d], tile[o]); });
  } else {
    const C<T> w = ph[__builtin_amdgcn_ubfe(wk.digits, 5 * g.a0, 5)];
    wk.each([&](int, int o) { tile[o] = cmul(w, tile[o]); });
  }
}

// the phases of the stage's rotation and Kerr gates into LDS (one contiguous region of the table)
template <typename T, typename Gm>
__device__ __forceinline__ void copy_phases(const sfamd::MArgs& a, const C<T>* __restrict__ table, C<T>* ph) {
  const C<T>* src = table + a.phases;
  for (int i = threadIdx.x; i < a.ndiag * Gm::D; i += Gm::NT) ph[i] = src[i];
}

template <int D, int K, int LG>
using StageGeo = Geo<D, K, LG, sfamd::mst_waves(D, K, LG)>;

// The gate loops are unrolled by two with two register sets for the operators:
// a gate (also a rotation or Kerr gate) first issues the loads of the next
// operators into the other set, so they are in flight over the whole gate and
// no register copies, which would wait for them, carry them around the loop.

// a gate forward; `op` holds its first operator, `next` receives that of the next gate with operators
template <typename T, typename Gm>
__device__ __forceinline__ void gate_fwd(const Gate& g, const C<T>* __restrict__ table, const Walk<T, Gm>& wk,
                                         const C<T>* ph, const C<T>* src, C<T>* dst, const C<T> (&op)[Gm::NE],
                                         C<T> (&next)[Gm::NE]) {
  load_image<T, Gm>(first_image<T, Gm>(table, g.nfwd, g.two & 2), next);
  if (g.kind <= SFAMD_OP_KERR)
    diag_fwd<T, Gm>(g, wk, ph + g.fwd, dst);
  else if (g.two & 1)
    heavy_fwd<T, Gm, true>(g, table, src, dst, op);
  else
    heavy_fwd<T, Gm, false>(g, table, src, dst, op);
  __syncthreads();
}

template <typename T, typename Gm>
__global__ void __launch_bounds__(Gm::NT)
k_mst_fwd(const C<T>* __restrict__ in, C<T>* __restrict__ out, const C<T>* __restrict__ table, sfamd::MArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  // layout: [tiles of the group][phases]
  C<T>* tile = reinterpret_cast<C<T>*>(smem);
  C<T>* ph = tile + Gm::GS;
  const int last = a.ngates - 1;
  const TileRange tr = xcd_tiles((a.ntiles + Gm::TT - 1) >> Gm::LG, a.grid);
  Walk<T, Gm> wk(a);
  copy_phases<T, Gm>(a, table, ph);
  // (the next group's loads in flight over this one's gates measured slower: they
  // cost the registers of a second workgroup per CU)
  for (int grp = tr.first; grp < tr.end; grp += tr.step) {
    C<T> opA[Gm::NE], opB[Gm::NE];
    {
      C<T> v[Walk<T, Gm>::PER];
      wk.at(grp, a);
      wk.fetch(in, v);
      load_image<T, Gm>(first_image<T, Gm>(table, a.h0_fwd, a.h0_two), opA);
      warm_gates<Gm>(a);
      wk.put(v, tile);
    }
    __syncthreads();
    for (int gi = 0; gi <= last; gi += 2) {
      gate_fwd<T, Gm>(a.g[gi], table, wk, ph, tile, tile, opA, opB);
      if (gi == last) break;
      gate_fwd<T, Gm>(a.g[gi + 1], table, wk, ph, tile, tile, opB, opA);
    }
    if (a.permuted)
      wk.store_permuted(grp, a, tile, out);
    else
      wk.store(tile, out);
    __syncthreads();
  }
}

// the operators of one adjoint item: G^H and, where two sets of both fit the
// registers, dG/dp0^H
template <typename T, typename Gm>
struct AdjOp {
  static constexpr bool kBoth = Gm::NE * sizeof(C<T>) <= 32;
  C<T> h[Gm::NE], d[kBoth ? Gm::NE : 1];
  __device__ __forceinline__ void load(const C<T>* __restrict__ table, int off, bool two) {
    const C<T>* img = first_image<T, Gm>(table, off, two);
    load_image<T, Gm>(img, h);
    if constexpr (kBoth) load_image<T, Gm>(img + (two ? Gm::D : 1) * Gm::IMG, d);
  }
};

// One gate with operators backward: lam in place; xt = its input tile, followed
// by its output tile; `op` holds the wave's first operators.  `between` runs
// while the LDS reads are in flight.
template <typename T, typename Gm, bool TWO, typename F>
__device__ __forceinline__ void heavy_adj(const Gate& g, const C<T>* __restrict__ table, const C<T>* xt,
                                          C<T>* lam, const AdjOp<T, Gm>& op, double& g0, double& g1, F between) {
  constexpr int N = Gm::items(TWO), J = Gm::per_wave(TWO);
  constexpr bool kReload = TWO && J > 1 && Gm::NW % Gm::D != 0;
  const int wave = wave_index();
  const C<T>* himg = table + g.adj;
  const C<T>* dimg = himg + (TWO ? Gm::D : 1) * Gm::IMG;
  const T wi = (T)0.5 * (T)(2 - ((g.two >> 4) & 7)), wo = (T)0.5 * (T)(2 - ((g.two >> 7) & 7));
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int item = wave + j * Gm::NW;
    if ((j + 1) * Gm::NW <= N || item < N) {
      const Place<Gm, TWO> pl(item, g);
      constexpr bool kOwnD = !AdjOp<T, Gm>::kBoth;  // dG/dp0^H loaded here
      C<T> der[Gm::NE];
      if (kOwnD || (kReload && j > 0)) load_image<T, Gm>(dimg + pl.p * Gm::IMG, der);
      C<T> l[Gm::P], x[Gm::P], po[Gm::P];
      typename Mx<T>::acc4 acc[Gm::MB], mu[Gm::MB];
      read_fiber<T, Gm, TWO>(lam, pl, l);
      read_fiber<T, Gm, TWO>(xt, pl, x);
      read_fiber<T, Gm, TWO>(xt + Gm::GS, pl, po);
      if (j == 0) between();
      if (kReload && j > 0) {
        C<T> other[Gm::NE];
        load_image<T, Gm>(himg + pl.p * Gm::IMG, other);
        apply_image<T, Gm>(other, l, acc);
        apply_image<T, Gm>(der, l, mu);
      } else {
        apply_image<T, Gm>(op.h, l, acc);
        if constexpr (kOwnD)
          apply_image<T, Gm>(der, l, mu);
        else
          apply_image<T, Gm>(op.d, l, mu);
      }
      T s0 = (T)0, s1 = (T)0;
#pragma unroll
      for (int q = 0; q < Gm::P; ++q) {
        // (slots past D - 1: acc and mu are zero, l and po are not)
        const T k = pl.has(q) ? (T)(pl.grp() * Gm::P + q) : (T)0;
        s1 += k * (wi * im_conj_mul(acc_amp<T>(acc, q), x[q]) + wo * im_conj_mul(l[q], po[q]));
        s0 += re_conj_mul(acc_amp<T>(mu, q), x[q]);
      }
      write_fiber<T, Gm, TWO>(lam, pl, acc);
      if (pl.valid) {
        g0 += (double)s0;
        g1 += (double)s1;
      }
    }
  }
}

// The per-lane parameter sums of the last GATES gates, reduced over the wave together
// and added to the wave's slots while the next gate's LDS reads are in flight.  Two gates
// at once halve the reductions' latency, which is in every gate's chain (6 modes, cutoff 8, 4
// layers, complex64, one gradient 1060 -> 1038 us; 10 modes 3, 2 layers, complex128 855 ->
// 811).  Where registers are short the second pair of sums spills: 5 modes 10, complex64, 40
// gates 321 -> 331 us, 5 modes 14, complex128, 2 layers 2146 -> 2282 (mst_sums).
template <int GATES>
struct Sums {
  double g0[GATES], g1[GATES];
  int gi = -1;  // the first gate; a second one is gi - 1
  template <typename Gm>
  __device__ __forceinline__ void flush(double* gsl, bool first) {
    if (gi < 0) return;
    const int lane = threadIdx.x & 63;
    double g;
    int at = gi;
    bool owner;
    if constexpr (GATES == 2) {
      g = wave_sum_four(g0[0], g0[1], g1[0], g1[1]);
      at -= (lane >> 4) & 1;
      owner = (lane & 15) == 15 && at >= 0;
    } else {
      g = wave_sum_pair(g0[0], g1[0]);
      owner = (lane & 31) == 31;
    }
    if (owner) {  // each wave owns its slots: deterministic
      double* slot = gsl + (at * 2 + (lane >> 5)) * Gm::NW + wave_index();
      slot[0] = first ? g : slot[0] + g;
    }
  }
};

// gate gi backward; `at`: the tile of its output, moved to that of its input; `first`: the workgroup's first
// group; SLOT: its place among the gates whose sums are reduced together; the first flushes those before
template <typename T, typename Gm, int SLOT, int GATES>
__device__ __forceinline__ void gate_adj(const Gate& g, int gi, const C<T>* __restrict__ table,
                                         const Walk<T, Gm>& wk, const C<T>* ph, C<T>*& at, C<T>* lam, double* gsl,
                                         bool first, Sums<GATES>& sum, const AdjOp<T, Gm>& op, AdjOp<T, Gm>& next) {
  next.load(table, g.padj, g.two & 4);
  double g0 = 0.0, g1 = 0.0;
  if (g.kind <= SFAMD_OP_KERR) {
    const C<T>* w0 = ph + g.fwd;
    const int kd = (int)__builtin_amdgcn_ubfe(wk.digits, 5 * g.a0, 5);
    wk.each([&](int d, int o) {
      const int k = g.a0 == 0 ? d : kd;
      const C<T> w = cconj(w0[k]), l = lam[o], x = at[o];
      g0 -= (double)(g.kind == SFAMD_OP_KERR ? k * k : k) * ((double)l.re * x.im - (double)l.im * x.re);
      lam[o] = cmul(w, l);
      at[o] = cmul(w, x);
    });
    if (SLOT == 0) sum.template flush<Gm>(gsl, first);
  } else {
    const bool two = g.two & 1;
    const int N = Gm::items(two);
    auto flush = [&]() {
      if (SLOT == 0) sum.template flush<Gm>(gsl, first);
    };
    if (wave_index() >= N) flush();
    if (two)
      heavy_adj<T, Gm, true>(g, table, at - Gm::GS, lam, op, g0, g1, flush);
    else
      heavy_adj<T, Gm, false>(g, table, at - Gm::GS, lam, op, g0, g1, flush);
    at -= Gm::GS;
  }
  sum.g0[SLOT] = g0;
  sum.g1[SLOT] = g1;
  if (SLOT == 0) {
    if (GATES == 2) sum.g0[GATES - 1] = sum.g1[GATES - 1] = 0.0;
    sum.gi = gi;
  }
  __syncthreads();
}

// waves per SIMD that the adjoint kernel's registers must allow
template <typename T, typename Gm>
constexpr int adj_waves() {
  return (sfamd::mst_two_groups(Gm::D, sizeof(T) == 4 ? SFAMD_C64 : SFAMD_C128) && Gm::LG == 0 && Gm::NW == 8) ? 4
                                                                                                    : (Gm::NW + 3) / 4;
}

// gates whose sums are reduced together (see Sums): one where the adjoint kernel has no register left
template <typename T, typename Gm>
constexpr int mst_sums() {
  return Gm::D <= 8 || (Gm::D <= 12 && sizeof(T) == 8) ? 2 : 1;
}

template <typename T, typename Gm>
__global__ void __launch_bounds__(Gm::NT, (adj_waves<T, Gm>()))
k_mst_adj(const C<T>* __restrict__ psi_in, const C<T>* __restrict__ lam_out, C<T>* __restrict__ lam_in,
          const C<T>* __restrict__ table, sfamd::MArgs a, double* __restrict__ partial, int nwg) {
  constexpr int NW = Gm::NW, NT = Gm::NT;
  extern __shared__ __align__(16) unsigned char smem[];
  // layout: [lam group][nheavy + 1 psi groups][phases][grad slots [ngates][2][waves]]
  C<T>* lam = reinterpret_cast<C<T>*>(smem);
  C<T>* psi = lam + Gm::GS;
  C<T>* ph = psi + (a.nheavy + 1) * Gm::GS;
  double* gsl = reinterpret_cast<double*>(ph + ((a.ndiag * Gm::D + 1) & ~1));
  const int last = a.ngates - 1;
  const TileRange tr = xcd_tiles((a.ntiles + Gm::TT - 1) >> Gm::LG, a.grid);
  Walk<T, Gm> wk(a);
  copy_phases<T, Gm>(a, table, ph);
  for (int idx = threadIdx.x; idx < a.ngates * 2 * NW; idx += NT) gsl[idx] = 0.0;
  for (int grp = tr.first; grp < tr.end; grp += tr.step) {
    C<T>* at = psi;
    {
      C<T> opA[Gm::NE], opB[Gm::NE];
      {
        C<T> v[Walk<T, Gm>::PER], w[Walk<T, Gm>::PER];
        wk.at(grp, a);
        wk.fetch(psi_in, v);
        wk.fetch(lam_out, w);
        load_image<T, Gm>(first_image<T, Gm>(table, a.h0_fwd, a.h0_two), opA);
        warm_gates<Gm>(a);
        if (Gm::LG && !wk.valid) {  // a tile past the last one adds nothing to the gradients
#pragma unroll
          for (int j = 0; j < Walk<T, Gm>::PER; ++j) v[j] = w[j] = mk<T>(0, 0);
        }
        wk.put(v, psi);
        wk.put(w, lam);
      }
      __syncthreads();
      // recompute the stage forward, keeping the input of every gate with operators
      for (int gi = 0; gi <= last; gi += 2) {
        C<T>* to = at + (a.g[gi].kind <= SFAMD_OP_KERR ? 0 : Gm::GS);
        gate_fwd<T, Gm>(a.g[gi], table, wk, ph, at, to, opA, opB);
        at = to;
        if (gi == last) break;
        to = at + (a.g[gi + 1].kind <= SFAMD_OP_KERR ? 0 : Gm::GS);
        gate_fwd<T, Gm>(a.g[gi + 1], table, wk, ph, at, to, opB, opA);
        at = to;
      }
    }
    AdjOp<T, Gm> opA, opB;
    opA.load(table, a.hl_adj, a.hl_two);
    constexpr int kGates = mst_sums<T, Gm>();
    Sums<kGates> sum;
    for (int gi = last; gi >= 0; gi -= 2) {
      gate_adj<T, Gm, 0>(a.g[gi], gi, table, wk, ph, at, lam, gsl, grp == tr.first, sum, opA, opB);
      if (gi == 0) break;
      gate_adj<T, Gm, kGates - 1>(a.g[gi - 1], gi - 1, table, wk, ph, at, lam, gsl, grp == tr.first, sum, opB, opA);
    }
    sum.template flush<Gm>(gsl, grp == tr.first);
    wk.store(lam, lam_in);
    __syncthreads();  // the tiles are free for the next group's loads
  }
  __syncthreads();
  // one partial per workgroup and gate parameter, at
  // partial[((op * 2 + side) * 2 + slot) * nwg + blockIdx.x]; the gradient
  // reduction reads the launch's gridDim.x columns
  for (int idx = threadIdx.x; idx < 2 * a.ngates; idx += NT) {
    const int gi = idx >> 1, slot = idx & 1;
    double s = 0.0;
    for (int w = 0; w < NW; ++w) s += gsl[idx * NW + w];
    partial[((int64_t)a.g[gi].op * 4 + a.side * 2 + slot) * nwg + blockIdx.x] = s;
  }
}

// ---- dispatch ---------------------------------------------------------------
// dynamic LDS above the default per-launch limit needs an opt-in per kernel
template <typename F>
int allow_lds(F kernel, size_t lds) {
  if (lds <= 65536) return 0;
  return (int)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)lds);
}

template <typename T>
constexpr int dtype_of() {
  return sizeof(T) == 4 ? SFAMD_C64 : SFAMD_C128;
}

template <typename T, int D, int K, int LG>
int launch_mst_fwd(const void* in, void* out, const void* table, const sfamd::MArgs& a, int grid, hipStream_t s) {
  using Gm = StageGeo<D, K, LG>;
  if constexpr ((int64_t)Gm::GS * (int64_t)sizeof(C<T>) > sfamd::kMstLds) {
    return SFAMD_E_ARG;
  } else {
    const size_t lds = (size_t)sfamd::mst_lds_fwd(D, K, LG, a.ndiag, dtype_of<T>());
    RET_IF(allow_lds(k_mst_fwd<T, Gm>, lds));
    sfamd::MArgs b = a;
    b.grid = grid;
    hipLaunchKernelGGL((k_mst_fwd<T, Gm>), dim3(grid), dim3(Gm::NT), lds, s, (const C<T>*)in, (C<T>*)out,
                       (const C<T>*)table, b);
    return (int)hipGetLastError();
  }
}

template <typename T, int D, int K, int LG>
int launch_mst_adj(const void* psi, const void* lo, void* li, const void* table, const sfamd::MArgs& a, int grid,
                   double* partial, int nwg, hipStream_t s) {
  using Gm = StageGeo<D, K, LG>;
  // no adjoint kernel where not even one gate's tiles fit the LDS
  if constexpr (3 * (int64_t)Gm::GS * (int64_t)sizeof(C<T>) > sfamd::kMstLds) {
    return SFAMD_E_ARG;
  } else {
    const size_t lds = (size_t)sfamd::mst_lds_adj(D, K, LG, a.ndiag, a.nheavy, dtype_of<T>());
    RET_IF(allow_lds(k_mst_adj<T, Gm>, lds));
    sfamd::MArgs b = a;
    b.grid = grid;
    hipLaunchKernelGGL((k_mst_adj<T, Gm>), dim3(grid), dim3(Gm::NT), lds, s, (const C<T>*)psi, (const C<T>*)lo,
                       (C<T>*)li, (const C<T>*)table, b, partial, nwg);
    return (int)hipGetLastError();
  }
}

// f(integral constants K, LG) for the kernel of (K, lgt), SFAMD_E_ARG if none exists;
// ADJ: the groups of a plan with an adjoint
template <int V>
struct Int {
  static constexpr int v = V;
};
template <int D, int K, bool ADJ, typename F>
int mst_with_group(int lgt, F f) {
  if (lgt == 0) return f(Int<K>(), Int<0>());
  if constexpr (ADJ ? sfamd::mst_group_fills(D, K, 1) : sfamd::mst_group_ok(D, K, 1))
    if (lgt == 1) return f(Int<K>(), Int<1>());
  if constexpr (ADJ ? sfamd::mst_group_fills(D, K, 2) : sfamd::mst_group_ok(D, K, 2))
    if (lgt == 2) return f(Int<K>(), Int<2>());
  return SFAMD_E_ARG;
}
template <int D, bool ADJ, typename F>
int mst_with(int K, int lgt, F f) {
  if (K == 3) return mst_with_group<D, 3, ADJ>(lgt, f);
  if constexpr (sfamd::mst_tile(D, 4) <= sfamd::kMstMaxTile)
    if (K == 4) return mst_with_group<D, 4, ADJ>(lgt, f);
  if constexpr (sfamd::mst_tile(D, 5) <= sfamd::kMstMaxTile)
    if (K == 5) return mst_with_group<D, 5, ADJ>(lgt, f);
  if constexpr (sfamd::mst_tile(D, 6) <= sfamd::kMstMaxTile)
    if (K == 6) return mst_with_group<D, 6, ADJ>(lgt, f);
  return SFAMD_E_ARG;
}

template <typename T, int D>
int mst_fwd_k(int K, const void* in, void* out, const void* table, const sfamd::MArgs& a, int grid, hipStream_t s) {
  return mst_with<D, false>(K, a.lgt, [&](auto k, auto lg) {
    return launch_mst_fwd<T, D, decltype(k)::v, decltype(lg)::v>(in, out, table, a, grid, s);
  });
}

template <typename T, int D>
int mst_adj_k(int K, const void* psi, const void* lo, void* li, const void* table, const sfamd::MArgs& a, int grid,
              double* partial, int nwg, hipStream_t s) {
  return mst_with<D, true>(K, a.lgt, [&](auto k, auto lg) {
    return launch_mst_adj<T, D, decltype(k)::v, decltype(lg)::v>(psi, lo, li, table, a, grid, partial, nwg, s);
  });
}

}  // namespace

// Defines sfamd::mst_fwd_d<d> / mst_adj_d<d>, the launchers of cutoff d (both
// dtypes, every K the tile limit allows); each mstage_dNN_MM.hip translation
// unit instantiates a range of cutoffs so the kernels compile in parallel.
#define SFAMD_MST_DEFINE_D(d)                                                                                   \
  namespace sfamd {                                                                                             \
  int mst_fwd_d##d(int K, const void* in, void* out, const void* table, const MArgs& a, int grid, int dtype,     \
                   hipStream_t s) {                                                                             \
    if (dtype == SFAMD_C64) return mst_fwd_k<float, d>(K, in, out, table, a, grid, s);                          \
    return mst_fwd_k<double, d>(K, in, out, table, a, grid, s);                                                 \
  }                                                                                                             \
  int mst_adj_d##d(int K, const void* psi, const void* lo, void* li, const void* table, const MArgs& a, int grid, \
                   double* partial, int nwg, int dtype, hipStream_t s) {                                        \
    if (dtype == SFAMD_C64) return mst_adj_k<float, d>(K, psi, lo, li, table, a, grid, partial, nwg, s);        \
    return mst_adj_k<double, d>(K, psi, lo, li, table, a, grid, partial, nwg, s);                               \
  }                                                                                                             \
  }
