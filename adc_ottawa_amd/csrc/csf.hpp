// The 1h1p<->2h2p coupling of the INT form applied to the CSF vectors
// themselves (no pair tensors); see csf.hip for the kernels.
#pragma once

#include <algorithm>

#include "csf_index.hpp"
#include "gemm.hpp"
#include "kernels.hpp"

// Lambdas of the kernels: inlined at every call, so that what they capture stays in registers.
#define ADC2G_INLINE __attribute__((always_inline))

namespace adc2g {

// Largest nocc of the CSF kernels: the up kernel holds one accumulator block
// per occupied orbital (32 x 8 registers in FP64).
constexpr int CSF_OMAX = 32;

// Sizes of one pass, passed by value.  P pairs (128 bytes of T) make a chunk;
// the pairs a < b fill nch chunks, the diagonal pairs a = b nchd more.
struct CsfGeo {
  int o, v, nv;
  int npo, nch, nchd;
  int64_t npv, off1, off2, off3, off4, off5, ldx, ldw;
};

template <class T>
constexpr int csf_pairs() { return 128 / (int)sizeof(T); }

template <class T>
inline CsfGeo csf_geo(const DimsK& d, int nv, int64_t ldx, int64_t ldw) {
  constexpr int P = csf_pairs<T>();
  CsfGeo g;
  g.o = d.o; g.v = d.v; g.nv = nv;
  g.npo = (int)d.npo; g.npv = d.npv;
  g.nch = (int)((d.npv + P - 1) / P);
  g.nchd = (d.v + P - 1) / P;
  g.off1 = d.off1; g.off2 = d.off2; g.off3 = d.off3; g.off4 = d.off4; g.off5 = d.off5;
  g.ldx = ldx; g.ldw = ldw;
  return g;
}

// a wave-uniform value that went through VALU instructions (a division), back in an SGPR
__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }

// Elements of the virtual operand: 2 o slabs of v rows of 128 bytes for each
// chunk, o for each diagonal chunk, and 16 rows that whole-tile loads may
// read past the last slab.
template <class T>
inline size_t csf_v_elems(const DimsK& d) {
  const CsfGeo g = csf_geo<T>(d, 1, 0, 0);
  return ((size_t)(2 * g.nch + g.nchd) * d.o * d.v + 16) * csf_pairs<T>();
}
// Occupied operand (FP64): [set][a][OM], sets = pairs k<l of t4, k of t2, pairs of t5.
inline int csf_om(int o) { return o <= 16 ? 16 : 32; }
inline size_t csf_o_elems(const DimsK& d) {
  return (size_t)(2 * d.npo + d.o) * ((d.v + 15) / 16 * 16) * csf_om(d.o);
}

// Operands from the integral blocks V[a][c][(b,l)] = (ac|bl), O[k][m][(b,l)] = (km|bl).
template <class T>
void launch_csf_build_v(const double* V, const DimsK& d, T* out, hipStream_t st);
void launch_csf_build_o(const double* O, const DimsK& d, double* out, hipStream_t st);

// Launch shapes and workspace (bytes) of the partial 1h1p sums.
struct CsfPlan {
  int dw, dg, dns, dnb, ds;  // down: waves, row groups, column splits, 16-column blocks, K splits
  int uw, uvpb, ug;          // up: waves, vectors per workgroup, groups
  int nt, sl;                // occupied: 16-virtual tiles, set slices
  int thin;                  // workgroups of the pass that does both directions, 0: separate passes
  size_t down_bytes, occ_bytes, t2_bytes;
};
CsfPlan csf_plan(const DimsK& d, int nv);
inline size_t ws_round(size_t bytes) { return (bytes + 255) / 256 * 256; }
// The largest workspaces of passes of 1..nv vectors (fewer vectors can mean
// more K splits, and more bytes).
struct CsfBytes {
  size_t down = 0, occ = 0, t2 = 0;
  size_t total() const { return ws_round(down) + ws_round(occ) + ws_round(t2); }
};
CsfBytes csf_workspace(const DimsK& d, int nv);

// W2 = D x2 + occupied up term (when up); partials of the occupied down term
// into `part` and the k-major copy T2 of -sqrt2 (t2, t1) (when down).
void launch_csf_occ(const CsfGeo& g, const CsfPlan& p, const double* X, const double* Oc, const double* eps,
                    double* W, double* part, double* T2, bool up, bool down, hipStream_t st);
// Partials of the virtual down term; zeros: csf_zeros(d) zeros.
template <class T>
void launch_csf_down(const CsfGeo& g, const CsfPlan& p, const double* X, const double* T2, const double* zeros,
                     const T* V, typename Mma<T>::Acc* part, hipStream_t st);
// W1 += both partials.
template <class Acc>
void launch_csf_reduce(const CsfGeo& g, const CsfPlan& p, int ndown, const Acc* down, const double* occ, double* W,
                       hipStream_t st);
// W2 += virtual up term.
template <class T>
void launch_csf_up(const CsfGeo& g, const CsfPlan& p, const double* X, const double* zeros, const T* V, double* W,
                   hipStream_t st);
// Both virtual terms (thin plans): W2 += the up term, partials of the down term.
template <class T>
void launch_csf_thin(const CsfGeo& g, const CsfPlan& p, const double* X, const double* T2, const double* zeros,
                     const T* V, double* W, typename Mma<T>::Acc* part, hipStream_t st);
inline size_t csf_zeros(const DimsK& d) {
  return (size_t)std::max<int64_t>(d.npv + d.v, d.n1 + 16 * d.o) + 64;
}

}  // namespace adc2g
