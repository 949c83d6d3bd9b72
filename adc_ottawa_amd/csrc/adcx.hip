// ADC(2)-x: the first-order 2h2p-2h2p block (get_offdiag_adc2ext_save,
// source/adclib/get_matrix.f90:2435-2893, element functions C_1_1 ..
// C_4ii_4ii of source/adclib/adc_ph.f90:1102-1645; diagonal of
// get_diag_adc2ext_direct) added to the ADC(2)-s sigma-vector.
//
// In pair space, with Z the closed-shell pair tensor of a CSF 2h2p vector
// (the t5 amplitudes weighted by 1/3, the norm ratio of the CSF states) and
// T = 2Z - XZ, (XZ)(c,b,k,l) = Z(b,c,k,l):
//   G(c,b,k,l) = 1/2 sum_de (cd|be) T(d,e,k,l) + 1/2 sum_mn (km|ln) T(c,b,m,n)
//              + sum_dm [2 (ck|dm) - (cd|km)] T(d,b,m,l)
//              - sum_dm [(cl|dm) T(d,b,m,k) + (cd|lm) T(d,b,k,m)],
// and the block is the CSF projection of G (again with 1/3 on t5).
//
// The ring terms are matrix products over n1 = o v:
//   G1[(c,k)][(b,l)] = A1 T1,          A1 = 2 (ck|dm) - (cd|km),  T1[(d,m)][(b,l)] = T(d,b,m,l)
//   G2[(c,l)][(b,k)] = OV T1 + VO T3,  T3[(d,m)][(b,k)] = T(d,b,k,m)
// (T1 also serves the (cl|dm) term: T(d,b,m,k) = T(b,d,k,m), the pair
// symmetry of Z).
//
// The ladder terms split over the parts of T symmetric (+) and antisymmetric
// (-) in the virtual pair, which by the pair symmetry are the same in the
// occupied pair, so that only d <= e, c <= b and k <= l (< for -) remain:
//   S+-(cb;kl) = G(c,b,k,l) +- G(b,c,k,l)
//              = 1/2 sum_{d<=e} Kpm(cb;de) Tpm(de;kl) + (oo|oo) likewise,
//   Kpm(cb;de) = (cd|be) +- (ce|bd).
// T+ and T- are the CSFs themselves (T+ = sqrt2 x4, -2 x2, x3, -sqrt2 x1 for
// the pairs of t4, t2, t3, t1; T- = x5 up to a factor), and S+- enter their
// CSFs directly.  That is 2 (v^2/2)^2 o^2 operations for the (vv|vv) term of a
// vector instead of the 2 v^4 o^2 of the unsymmetrised matrix (which took
// 17.6 of the 25.4 ms of 4 vectors at o=14, v=150), and half its storage.
//
// FP64.
#include "handle.hpp"

#include <algorithm>
#include <cmath>

namespace adc2g {

namespace {

constexpr double AX_SQ2 = 1.4142135623730951;
constexpr double AX_ISQ2 = 0.7071067811865476;
constexpr double AX_SQ32 = 1.2247448713915890;

__device__ __forceinline__ int64_t ax_pair(int64_t lo, int64_t hi, int64_t n) {
  return lo * n - lo * (lo + 1) / 2 + (hi - lo - 1);
}

// p -> (lo, hi), lo < hi < n, the inverse of ax_pair
__device__ __forceinline__ void ax_unpair(int64_t p, int64_t n, int& lo, int& hi) {
  const double b = 2.0 * (double)n - 1.0;
  int a = (int)floor(0.5 * (b - sqrt(fmax(b * b - 8.0 * (double)p, 0.0))));
  a = max(a, 0);
  while (a > 0 && (int64_t)a * (2 * n - a - 1) / 2 > p) --a;
  while ((int64_t)(a + 1) * (2 * n - a - 2) / 2 <= p) ++a;
  lo = a;
  hi = (int)(p - (int64_t)a * (2 * n - a - 1) / 2) + a + 1;
}

// Z(c,b,k,l) of the full vector x (t5 weighted by 1/3)
__device__ double ax_z(const double* __restrict__ x, const DimsK& d, int c, int b, int k, int l) {
  const int o = d.o, v = d.v;
  if (c == b) {
    if (k == l) return -AX_SQ2 * x[d.off1 + (int64_t)k * v + c];
    return x[d.off3 + ax_pair(min(k, l), max(k, l), o) * v + c];
  }
  const int64_t pab = ax_pair(min(c, b), max(c, b), v);
  if (k == l) return -x[d.off2 + pab * o + k];
  const int64_t q = ax_pair(min(k, l), max(k, l), o) * d.npv + pab;
  const double s4 = AX_ISQ2 * x[d.off4 + q], s5 = (AX_SQ32 / 3.0) * x[d.off5 + q];
  return ((c < b) == (k < l)) ? s4 + s5 : s4 - s5;
}

__device__ __forceinline__ double ax_t(const double* x, const DimsK& d, int c, int b, int k, int l) {
  return 2.0 * ax_z(x, d, c, b, k, l) - ax_z(x, d, b, c, k, l);
}

// T1 and T3 for the nb vectors of a chunk (vector j = blockIdx.y), stored
// transposed -- contiguous over the contraction index:
//   T1t[j][(b,l)][(d,m)] = T(d,b,m,l), T3t[j][(b,k)][(d,m)] = T(d,b,k,m)
// (one element per thread, for nocc > 64; launch_pack_t otherwise)
__global__ void ax_layouts_kernel(const double* __restrict__ X, int64_t ldx, DimsK d, double* __restrict__ T1,
                                  double* __restrict__ T3) {
  const int o = d.o;
  const int j = blockIdx.y;
  const double* x = X + ldx * j;
  const int64_t n1 = d.n1, nn = n1 * n1;
  for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < nn;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int64_t q = idx / n1, r = idx - q * n1;
    const int dd = (int)(r / o), m = (int)(r - (int64_t)dd * o);
    const int b = (int)(q / o), l = (int)(q - (int64_t)b * o);
    T1[j * nn + idx] = ax_t(x, d, dd, b, m, l);
    T3[j * nn + idx] = ax_t(x, d, dd, b, l, m);
  }
}

// Tp[(j, k<=l)][d<=e] and Tm[(j, k<l)][d<e] of the vectors of a chunk, rows of
// ldp and ldm elements (zeros at their ends): pairs k < l first, then k = l;
// pairs d < e first, then d = e.
__global__ void ax_pm_kernel(const double* __restrict__ X, int64_t ldx, int nb, DimsK d, int64_t ldp, int64_t ldm,
                             double* __restrict__ Tp, double* __restrict__ Tm) {
  const int o = d.o, v = d.v;
  const int64_t so = d.npo + o;
  const int64_t row = blockIdx.y + (int64_t)gridDim.y * blockIdx.z;
  if (row >= so * nb) return;
  const int64_t j = row / so, kl = row - j * so;
  const double* x = X + ldx * j;
  double* tp = Tp + row * ldp;
  double* tm = Tm + (j * d.npo + kl) * ldm;
  for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < ldp; p += (int64_t)gridDim.x * blockDim.x) {
    double val = 0.0;
    if (kl < d.npo) {
      if (p < d.npv) val = AX_SQ2 * x[d.off4 + kl * d.npv + p];
      else if (p < d.npv + v) val = x[d.off3 + kl * v + p - d.npv];
      if (p < ldm) tm[p] = p < d.npv ? x[d.off5 + kl * d.npv + p] : 0.0;
    } else {
      const int64_t k = kl - d.npo;
      if (p < d.npv) val = -2.0 * x[d.off2 + p * o + k];
      else if (p < d.npv + v) val = -AX_SQ2 * x[d.off1 + k * v + p - d.npv];
    }
    tp[p] = val;
  }
}

// Kp[(c<=b)][(d<=e)], Km[(c<b)][(d<e)] from I[c][d][b][e] = (cd|be)
__global__ void ax_kpm_kernel(const double* __restrict__ I, DimsK d, int64_t ldp, int64_t ldm,
                              double* __restrict__ Kp, double* __restrict__ Km) {
  const int v = d.v;
  const int64_t r = blockIdx.y + (int64_t)gridDim.y * blockIdx.z;
  if (r >= d.npv + v) return;
  int c, b;
  if (r < d.npv) ax_unpair(r, v, c, b);
  else c = b = (int)(r - d.npv);
  for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < ldp; p += (int64_t)gridDim.x * blockDim.x) {
    double kp = 0.0, km = 0.0;
    if (p < d.npv + v) {
      int dd, e;
      if (p < d.npv) ax_unpair(p, v, dd, e);
      else dd = e = (int)(p - d.npv);
      const double g1 = I[(((int64_t)c * v + dd) * v + b) * v + e], g2 = I[(((int64_t)c * v + e) * v + b) * v + dd];
      kp = g1 + g2;
      km = g1 - g2;
    }
    Kp[r * ldp + p] = kp;
    if (r < d.npv && p < ldm) Km[r * ldm + p] = p < d.npv ? km : 0.0;
  }
}

// Columns of the matrices of the occupied ladder: whole blocks of ax_ladder_kernel.
constexpr int AX_LADDER_ROWS = 64;
__host__ __device__ __forceinline__ int ax_ladder_ld(int64_t n) {
  return (int)((n + AX_LADDER_ROWS - 1) / AX_LADDER_ROWS) * AX_LADDER_ROWS;
}

// Op[(m<=n)][(k<=l)] = (km|ln) + (kn|lm) (m < n), (km|lm) (m = n); Om with a
// minus sign and no equal pairs: rows of ax_ladder_ld elements, zero rows and
// columns up to as many.  oooo[(m,n)][(k,l)] = (km|ln).
__global__ void ax_opm_kernel(const double* __restrict__ oooo, DimsK d, double* __restrict__ Op,
                              double* __restrict__ Om) {
  const int o = d.o;
  const int64_t so = d.npo + o, lp = ax_ladder_ld(so), lm = ax_ladder_ld(d.npo);
  for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < lp * lp;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int64_t q = idx / lp, r = idx - q * lp;
    double p = 0.0, x = 0.0;
    if (r < so && q < so) {
      int k, l, m, n;
      if (r < d.npo) ax_unpair(r, o, k, l);
      else k = l = (int)(r - d.npo);
      if (q < d.npo) ax_unpair(q, o, m, n);
      else m = n = (int)(q - d.npo);
      const double g1 = oooo[(((int64_t)m * o + n) * o + k) * o + l], g2 = oooo[(((int64_t)n * o + m) * o + k) * o + l];
      p = m == n ? g1 : g1 + g2;
      x = r < d.npo && q < d.npo ? g1 - g2 : 0.0;
    }
    Op[idx] = p;
    if (r < lm && q < lm) Om[q * lm + r] = x;
  }
}

// ring part of G(c,b,k,l) of vector j
__device__ __forceinline__ double ax_g(const double* G1, const double* G2, const DimsK& d, int j, int c, int b, int k,
                                       int l) {
  const int o = d.o;
  const int64_t n1 = d.n1, base = (int64_t)j * n1 * n1;
  return G1[base + ((int64_t)c * o + k) * n1 + (int64_t)b * o + l] -
         G2[base + ((int64_t)c * o + l) * n1 + (int64_t)b * o + k];
}

// 2h2p configuration J (0-based within the 2h2p part) -> type 1..5 and (a, b, k, l)
__device__ __forceinline__ int ax_decode(int64_t J, const DimsK& d, int& a, int& b, int& k, int& l) {
  const int o = d.o, v = d.v;
  const int64_t c1 = (int64_t)o * v, c2 = d.npv * o, c3 = d.npo * v, c4 = d.npo * d.npv;
  if (J < c1) {
    k = l = (int)(J / v);
    a = b = (int)(J - (int64_t)k * v);
    return 1;
  }
  J -= c1;
  if (J < c2) {
    k = l = (int)(J % o);
    ax_unpair(J / o, v, a, b);
    return 2;
  }
  J -= c2;
  if (J < c3) {
    a = b = (int)(J % v);
    ax_unpair(J / v, o, k, l);
    return 3;
  }
  J -= c3;
  const int t = (J < c4) ? 4 : 5;
  if (t == 5) J -= c4;
  ax_unpair(J % d.npv, v, a, b);
  ax_unpair(J / d.npv, o, k, l);
  return t;
}

// w[off1 + J] += (M22 x)_J of the ring terms (the CSF projection of G, 1/3 on
// t5), vector j = blockIdx.y (for nocc > 64; launch_unpack_g otherwise)
__global__ void ax_project_kernel(const double* __restrict__ G1, const double* __restrict__ G2, DimsK d,
                                  double* __restrict__ W, int64_t ldw) {
  const int64_t n2 = d.ndim - d.n1;
  const int j = blockIdx.y;
  double* w = W + ldw * j;
  for (int64_t J = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; J < n2; J += (int64_t)gridDim.x * blockDim.x) {
    int a, b, k, l;
    const int t = ax_decode(J, d, a, b, k, l);
    double val;
    if (t == 1) {
      val = -AX_SQ2 * ax_g(G1, G2, d, j, a, a, k, k);
    } else if (t == 2) {
      val = -(ax_g(G1, G2, d, j, a, b, k, k) + ax_g(G1, G2, d, j, b, a, k, k));
    } else if (t == 3) {
      val = ax_g(G1, G2, d, j, a, a, k, l) + ax_g(G1, G2, d, j, a, a, l, k);
    } else {
      const double g1 = ax_g(G1, G2, d, j, a, b, k, l), g2 = ax_g(G1, G2, d, j, b, a, k, l);
      const double g3 = ax_g(G1, G2, d, j, a, b, l, k), g4 = ax_g(G1, G2, d, j, b, a, l, k);
      val = (t == 4) ? AX_ISQ2 * (g1 + g2 + g3 + g4) : (AX_SQ32 / 3.0) * (g1 - g2 - g3 + g4);
    }
    w[d.off1 + J] += val;
  }
}

// The occupied ladder added to the virtual one in S+ (PLUS) or S-, and both to
// the CSFs: w4 += sqrt2 S+, w3 += S+, w2 -= S+, w1 -= S+ / sqrt2, w5 += S-
// (already in units of x5); rows as in ax_pm_kernel, ld elements each.  A
// workgroup takes 16 columns p and 64 rows kl on FP64 MFMA, its four waves every
// fourth run of 16 pairs mn (one wave alone is a chain of (o/2)^2 / 8 round trips to
// the L2); T is read along p and the matrix along kl, whole cache lines both, and
// S is read once.  As products of their own (three launches of few workgroups) the
// occupied terms and the addition took 67 us of the 200 of one vector at o=12,
// v=24; this kernel 8.5.
constexpr int AX_MB = AX_LADDER_ROWS / 16;
static_assert(AX_MB == 4, "one block of rows for each wave at the end");

template <bool PLUS>
__device__ __forceinline__ void ax_ladder(const double* __restrict__ T, const double* __restrict__ O,
                                          const double* __restrict__ S, const DimsK& d, int64_t ld, int chunk,
                                          double* __restrict__ W, int64_t ldw,
                                          double (*red)[AX_MB][4][64]) {  // [wave][block][register][lane]
  typedef Mma<double> MT;
  typedef MT::v4 v4;
  constexpr int MB = AX_MB;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, li = lane & 15, gq = lane >> 4;
  const int64_t npv = d.npv;
  const int n = (int)(PLUS ? d.npo + d.o : d.npo), lo = ax_ladder_ld(n);
  const int64_t j = blockIdx.y, p = (int64_t)blockIdx.x * 16 + li;
  const int kl0 = chunk * AX_LADDER_ROWS;
  if (p - li >= ld) return;  // the whole workgroup (ld is a multiple of 16)
  const double* t = T + j * n * ld + p;
  const double* a = O + kl0 + li;
  v4 acc[MB];
#pragma unroll
  for (int m = 0; m < MB; ++m) acc[m] = (v4){0, 0, 0, 0};
  for (int k = wv * 16; k < n; k += 64) {
    double b[4], x[4][MB];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int mn = k + 4 * s + gq;  // (rows past n: zeros)
      b[s] = t[min(mn, n - 1) * ld];
      b[s] = mn < n ? b[s] : 0.0;
#pragma unroll
      for (int m = 0; m < MB; ++m) x[s][m] = a[(int64_t)mn * lo + m * 16];
    }
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int m = 0; m < MB; ++m) acc[m] = MT::mma(x[s][m], b[s], acc[m]);
  }
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wv][m][r][lane] = acc[m][r];
  __syncthreads();
  const int o = d.o, v = d.v;
  if (p >= (PLUS ? npv + v : npv)) return;
  const double* s0 = S + j * n * ld + p;
  double* w = W + ldw * j;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int64_t kl = kl0 + wv * 16 + MT::row(lane, r);
    if (kl >= n) continue;
    const double occ = (red[0][wv][r][lane] + red[1][wv][r][lane]) + (red[2][wv][r][lane] + red[3][wv][r][lane]);
    if (!PLUS) {
      w[d.off5 + kl * npv + p] += s0[kl * ld] + occ;
      continue;
    }
    // (T+ of c = b is not doubled)
    const double s = s0[kl * ld] + (p < npv ? 0.5 : 1.0) * occ;
    if (kl < d.npo) {
      if (p < npv) w[d.off4 + kl * npv + p] += AX_SQ2 * s;
      else w[d.off3 + kl * v + p - npv] += s;
    } else {
      const int64_t k = kl - d.npo;
      if (p < npv) w[d.off2 + p * o + k] -= s;
      else w[d.off1 + k * v + p - npv] -= AX_ISQ2 * s;
    }
  }
}

// workgroups (columns, vector, rows): the first cp of the rows S+, the others S-
__global__ void __launch_bounds__(256)
ax_ladder_kernel(const double* __restrict__ Tp, const double* __restrict__ Op, const double* __restrict__ Sp,
                 const double* __restrict__ Tm, const double* __restrict__ Om, const double* __restrict__ Sm, DimsK d,
                 int64_t ldp, int64_t ldm, int cp, double* __restrict__ W, int64_t ldw) {
  __shared__ double red[4][AX_MB][4][64];
  const int z = blockIdx.z;
  if (z < cp) ax_ladder<true>(Tp, Op, Sp, d, ldp, z, W, ldw, red);
  else ax_ladder<false>(Tm, Om, Sm, d, ldm, z - cp, W, ldw, red);
}

struct AxMats {
  const double *vvvv, *oooo, *ov, *vo, *a1;
};

// pair-space matrix element of the operator acting on T (the G formula)
__device__ double ax_kpp(const AxMats& M, const DimsK& d, int c, int b, int k, int l, int dd, int e, int m, int n) {
  const int o = d.o, v = d.v;
  const int64_t n1 = d.n1;
  double r = 0.0;
  if (k == m && l == n) r += 0.5 * M.vvvv[(((int64_t)c * v + dd) * v + b) * v + e];
  if (c == dd && b == e) r += 0.5 * M.oooo[(((int64_t)m * o + n) * o + k) * o + l];
  if (b == e) {
    if (n == l) r += M.a1[((int64_t)c * o + k) * n1 + (int64_t)dd * o + m];
    if (n == k) r -= M.ov[((int64_t)c * o + l) * n1 + (int64_t)dd * o + m];
    if (m == k) r -= M.vo[((int64_t)c * o + l) * n1 + (int64_t)dd * o + n];
  }
  return r;
}

// diagonal of the block: sum over the (at most 4) pair positions x, y of the
// configuration's pair tensor P of P[x] P[y] (2 K''[x,y] - K''[x,Xy])
__global__ void ax_diag_kernel(AxMats M, DimsK d, double* __restrict__ diag) {
  const int64_t n2 = d.ndim - d.n1;
  for (int64_t J = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; J < n2; J += (int64_t)gridDim.x * blockDim.x) {
    int a, b, k, l;
    const int t = ax_decode(J, d, a, b, k, l);
    int pc[4], pb[4], pk[4], pl[4];
    double pw[4];
    int np;
    double nt = 1.0;
    if (t == 1) {
      np = 1;
      pc[0] = a; pb[0] = a; pk[0] = k; pl[0] = k; pw[0] = -AX_SQ2;
    } else if (t == 2) {
      np = 2;
      pc[0] = a; pb[0] = b; pk[0] = k; pl[0] = k; pw[0] = -1.0;
      pc[1] = b; pb[1] = a; pk[1] = k; pl[1] = k; pw[1] = -1.0;
    } else if (t == 3) {
      np = 2;
      pc[0] = a; pb[0] = a; pk[0] = k; pl[0] = l; pw[0] = 1.0;
      pc[1] = a; pb[1] = a; pk[1] = l; pl[1] = k; pw[1] = 1.0;
    } else {
      np = 4;
      const double s = (t == 4) ? AX_ISQ2 : AX_SQ32;
      const double x = (t == 4) ? AX_ISQ2 : -AX_SQ32;
      if (t == 5) nt = 1.0 / 3.0;
      pc[0] = a; pb[0] = b; pk[0] = k; pl[0] = l; pw[0] = s;
      pc[1] = b; pb[1] = a; pk[1] = l; pl[1] = k; pw[1] = s;
      pc[2] = b; pb[2] = a; pk[2] = k; pl[2] = l; pw[2] = x;
      pc[3] = a; pb[3] = b; pk[3] = l; pl[3] = k; pw[3] = x;
    }
    double sum = 0.0;
    for (int i = 0; i < np; ++i)
      for (int j = 0; j < np; ++j) {
        const double kk = 2.0 * ax_kpp(M, d, pc[i], pb[i], pk[i], pl[i], pc[j], pb[j], pk[j], pl[j]) -
                          ax_kpp(M, d, pc[i], pb[i], pk[i], pl[i], pb[j], pc[j], pk[j], pl[j]);
        sum += pw[i] * pw[j] * kk;
      }
    diag[J] = nt * nt * sum;
  }
}

// out[i0][k][j][i3] = in[i0][j][k][i3]: in of shape (n0, nb, na, n3), out of
// shape (n0, na, nb, n3) -- the two middle indices swapped
__global__ void ax_swap_mid_kernel(const double* __restrict__ in, int64_t n0, int64_t na, int64_t nb, int64_t n3,
                                   double* __restrict__ out) {
  const int64_t total = n0 * na * nb * n3;
  for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    int64_t r = idx;
    const int64_t i3 = r % n3; r /= n3;
    const int64_t j = r % nb; r /= nb;   // output index order: [i][j'][k'][i3] with j' over nb
    const int64_t k = r % na; r /= na;
    const int64_t i0 = r;
    // idx = ((i0*na + k)*nb + j)*n3 + i3 is out[i0][k][j][i3] = in[i0][j][k][i3]
    out[idx] = in[((i0 * nb + j) * na + k) * n3 + i3];
  }
}

__global__ void ax_axpby_kernel(int64_t n, double a, const double* __restrict__ x, double b,
                                const double* __restrict__ y, double* __restrict__ z) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    z[i] = a * x[i] + b * y[i];
}

__global__ void ax_add_kernel(int64_t n, double s, const double* __restrict__ x, double* __restrict__ y) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    y[i] += s * x[i];
}

// rows padded to whole K tiles of the products
inline int64_t ax_ld(int64_t n) { return (n + 15) / 16 * 16; }

// C (M x N, ldc) = alpha A (M x K, lda) Bt^T + beta C with Bt N x K (ldbt): both
// operands contiguous along K (the vector loads and the wide tiles)
void ax_gemm_bt(Handle& H, int M, int N, int K, const double* A, int64_t lda, const double* Bt, int64_t ldbt,
                double* C, int64_t ldc, double alpha, double beta, hipStream_t s) {
  GemmArgs g;
  g.M = M; g.N = N; g.K = K;
  g.A = A; g.sam = lda; g.sak = 1;
  g.B = Bt; g.sbk = 1; g.sbn = ldbt;
  g.map.C = C; g.map.scm = ldc; g.map.scn = 1; g.map.alpha = alpha; g.map.beta = beta;
  gemm(g, Prec::F64, H.gws, s);
}


}  // namespace

void Handle::enable_adcx(bool on) {
  ARG_CHECK(!parent, "ADC(2)-x is switched on the full operator, before its views are made");
  ARG_CHECK(nviews == 0, "switch ADC(2)-x before making views (their diagonal is taken at creation)");
  if (on == adcx) return;
  HIP_CHECK(hipSetDevice(device));
  const int o = d.o, v = d.v, naux = d.naux;
  const int64_t n1 = d.n1, n2 = d.ndim - d.n1, vv = (int64_t)v * v, oo = (int64_t)o * o;
  if (on && !ax_d2.get()) {
    // (ck|dm) and (cd|km) as n1 x n1 matrices, A1 = 2 OV - VO
    ax_ov.alloc((size_t)n1 * n1);
    ax_vo.alloc((size_t)n1 * n1);
    ax_a1.alloc((size_t)n1 * n1);
    {
      GemmArgs g;
      g.M = (int)n1; g.N = (int)n1; g.K = naux;
      g.A = Bov.get(); g.sam = 1; g.sak = n1;
      g.B = Bov.get(); g.sbk = n1; g.sbn = 1;
      g.map.C = ax_ov.get(); g.map.scm = n1; g.map.scn = 1;
      gemm(g, Prec::F64, gws, st);
    }
    {
      DevBuf<double> J;  // [(c,d)][(k,m)] = (cd|km)
      J.alloc((size_t)vv * oo);
      GemmArgs g;
      g.M = (int)vv; g.N = (int)oo; g.K = naux;
      g.A = Bvv.get(); g.sam = 1; g.sak = vv;
      g.B = Boo.get(); g.sbk = oo; g.sbn = 1;
      g.map.C = J.get(); g.map.scm = oo; g.map.scn = 1;
      gemm(g, Prec::F64, gws, st);
      // [c][d][k][m] -> [c][k][d][m]
      hipLaunchKernelGGL(ax_swap_mid_kernel, dim3(grid_for(vv * oo)), dim3(256), 0, st, J.get(), (int64_t)v,
                         (int64_t)o, (int64_t)v, (int64_t)o, ax_vo.get());
      HIP_CHECK(hipGetLastError());
      HIP_CHECK(hipStreamSynchronize(st));
    }
    hipLaunchKernelGGL(ax_axpby_kernel, dim3(grid_for(n1 * n1)), dim3(256), 0, st, n1 * n1, 2.0, ax_ov.get(), -1.0,
                       ax_vo.get(), ax_a1.get());
    HIP_CHECK(hipGetLastError());
    // I[(c,d)][(b,e)] = (cd|be): its symmetric and antisymmetric parts and,
    // with it, the diagonal of the block
    DevBuf<double> I;
    I.alloc((size_t)vv * vv);
    {
      GemmArgs g;
      g.M = (int)vv; g.N = (int)vv; g.K = naux;
      g.A = Bvv.get(); g.sam = 1; g.sak = vv;
      g.B = Bvv.get(); g.sbk = vv; g.sbn = 1;
      g.map.C = I.get(); g.map.scm = vv; g.map.scn = 1;
      gemm(g, Prec::F64, gws, st);
    }
    const int64_t sv = d.npv + v, ldp = ax_ld(sv), ldm = ax_ld(d.npv);
    ax_kp.alloc((size_t)sv * ldp);
    ax_km.alloc((size_t)d.npv * ldm);
    hipLaunchKernelGGL(ax_kpm_kernel, dim3((unsigned)std::min<int64_t>((ldp + 255) / 256, 64), 4096,
                                           (unsigned)((sv + 4095) / 4096)),
                       dim3(256), 0, st, I.get(), dk, ldp, ldm, ax_kp.get(), ax_km.get());
    HIP_CHECK(hipGetLastError());
    // (km|ln) as [(m,n)][(k,l)]
    DevBuf<double> ax_oooo;
    ax_oooo.alloc((size_t)oo * oo);
    {
      DevBuf<double> Q;  // [(k,m)][(l,n)] = (km|ln)
      Q.alloc((size_t)oo * oo);
      GemmArgs g;
      g.M = (int)oo; g.N = (int)oo; g.K = naux;
      g.A = Boo.get(); g.sam = 1; g.sak = oo;
      g.B = Boo.get(); g.sbk = oo; g.sbn = 1;
      g.map.C = Q.get(); g.map.scm = oo; g.map.scn = 1;
      gemm(g, Prec::F64, gws, st);
      // [k][m][l][n] -> [m][n][k][l]: two steps, swap(m,l) then transpose pairs
      DevBuf<double> R;
      R.alloc((size_t)oo * oo);
      // R[k][l][m][n] = Q[k][m][l][n]
      hipLaunchKernelGGL(ax_swap_mid_kernel, dim3(grid_for(oo * oo)), dim3(256), 0, st, Q.get(), (int64_t)o,
                         (int64_t)o, (int64_t)o, (int64_t)o, R.get());
      HIP_CHECK(hipGetLastError());
      // ax_oooo[(m,n)][(k,l)] = R[(k,l)][(m,n)]: a transpose of the oo x oo matrix
      launch_transpose<double, double>(R.get(), oo, oo, ax_oooo.get(), st);
      HIP_CHECK(hipStreamSynchronize(st));
    }
    const int64_t lp = ax_ladder_ld(d.npo + o), lm = ax_ladder_ld(d.npo);
    ax_op.alloc((size_t)lp * lp);
    ax_om.alloc((size_t)lm * lm);
    hipLaunchKernelGGL(ax_opm_kernel, dim3(grid_for(lp * lp)), dim3(256), 0, st, ax_oooo.get(), dk, ax_op.get(),
                       ax_om.get());
    HIP_CHECK(hipGetLastError());
    ax_d2.alloc((size_t)n2);
    AxMats M{I.get(), ax_oooo.get(), ax_ov.get(), ax_vo.get(), ax_a1.get()};
    hipLaunchKernelGGL(ax_diag_kernel, dim3(grid_for(n2)), dim3(256), 0, st, M, dk, ax_d2.get());
    HIP_CHECK(hipGetLastError());
    HIP_CHECK(hipStreamSynchronize(st));
  }
  // the ADC(2)-x diagonal: hii of the 2h2p configurations plus the block's
  hipLaunchKernelGGL(ax_add_kernel, dim3(grid_for(n2)), dim3(256), 0, st, n2, on ? 1.0 : -1.0, ax_d2.get(),
                     hii.get() + n1);
  HIP_CHECK(hipGetLastError());
  HIP_CHECK(hipStreamSynchronize(st));
  adcx = on;
}

void Handle::adcx_apply(const double* X, int64_t ldx, double* W, int64_t ldw, int nvec, hipStream_t s) {
  ARG_CHECK(!scratch, "the no-allocation sigma-vector does not include the ADC(2)-x block");
  const int o = d.o, v = d.v;
  const int64_t n1 = d.n1, nn = n1 * n1;
  const int64_t sv = d.npv + v, so = d.npo + o, ldp = ax_ld(sv), ldm = ax_ld(d.npv);
  // vectors per chunk: about six n1 x n1 arrays per vector within about 4 GB
  const int64_t per_vec = 6 * nn * (int64_t)sizeof(double);
  const int cap = (int)std::max<int64_t>(1, std::min<int64_t>(16, ((int64_t)4 << 30) / per_vec));
  const int nbmax = std::min(nvec, cap);
  ax_t1.alloc((size_t)nbmax * nn);
  ax_t3.alloc((size_t)nbmax * nn);
  ax_g1.alloc((size_t)nbmax * nn);
  ax_g2.alloc((size_t)nbmax * nn);
  ax_tp.alloc((size_t)nbmax * so * ldp);
  ax_tm.alloc((size_t)nbmax * d.npo * ldm);
  ax_sp.alloc((size_t)nbmax * so * ldp);
  ax_sm.alloc((size_t)nbmax * d.npo * ldm);
  const PairLayout lay = pair_layout_vec_major(dk);
  for (int j0 = 0; j0 < nvec; j0 += nbmax) {
    const int nb = std::min(nbmax, nvec - j0);
    const double* x = X + ldx * j0;
    double* w = W + ldw * j0;
    if (!launch_pack_t(x, ldx, nb, dk, ax_t1.get(), ax_t3.get(), lay, s)) {
      hipLaunchKernelGGL(ax_layouts_kernel, dim3(grid_for(nn), nb), dim3(256), 0, s, x, ldx, dk, ax_t1.get(),
                         ax_t3.get());
      HIP_CHECK(hipGetLastError());
    }
    auto ring = [&](const double* A, const double* T, double* G, double beta) {
      GemmArgs g;
      g.M = (int)n1; g.N = (int)n1; g.K = (int)n1; g.batch = nb;
      g.A = A; g.sam = n1; g.sak = 1; g.sab = 0;
      g.B = T; g.sbk = 1; g.sbn = n1; g.sbb = nn;
      g.map.C = G; g.map.scm = n1; g.map.scn = 1; g.map.scb = nn; g.map.beta = beta;
      gemm(g, Prec::F64, gws, s);
    };
    ring(ax_a1.get(), ax_t1.get(), ax_g1.get(), 0.0);
    ring(ax_ov.get(), ax_t1.get(), ax_g2.get(), 0.0);
    ring(ax_vo.get(), ax_t3.get(), ax_g2.get(), 1.0);
    if (!launch_unpack_g(ax_g1.get(), ax_g2.get(), w, ldw, nb, dk, lay, s)) {
      hipLaunchKernelGGL(ax_project_kernel, dim3(grid_for(d.ndim - n1), nb), dim3(256), 0, s, ax_g1.get(),
                         ax_g2.get(), dk, w, ldw);
      HIP_CHECK(hipGetLastError());
    }
    // ladder: rows (vector, kl), columns cb; T and K contiguous along de
    const unsigned ry = (unsigned)std::min<int64_t>(nb * so, 32768);
    const dim3 rows((unsigned)std::min<int64_t>((ldp + 255) / 256, 64), ry, (unsigned)((nb * so + ry - 1) / ry));
    hipLaunchKernelGGL(ax_pm_kernel, rows, dim3(256), 0, s, x, ldx, nb, dk, ldp, ldm, ax_tp.get(), ax_tm.get());
    HIP_CHECK(hipGetLastError());
    ax_gemm_bt(*this, (int)(nb * so), (int)sv, (int)ldp, ax_tp.get(), ldp, ax_kp.get(), ldp, ax_sp.get(), ldp, 0.5,
               0.0, s);
    ax_gemm_bt(*this, (int)(nb * d.npo), (int)d.npv, (int)ldm, ax_tm.get(), ldm, ax_km.get(), ldm, ax_sm.get(), ldm,
               1.0, 0.0, s);
    const int cp = ax_ladder_ld(so) / AX_LADDER_ROWS, cm = ax_ladder_ld(d.npo) / AX_LADDER_ROWS;
    hipLaunchKernelGGL(ax_ladder_kernel, dim3((unsigned)(ldp / 16), (unsigned)nb, (unsigned)(cp + cm)), dim3(256), 0, s,
                       ax_tp.get(), ax_op.get(), ax_sp.get(), ax_tm.get(), ax_om.get(), ax_sm.get(), dk, ldp, ldm, cp,
                       w, ldw);
    HIP_CHECK(hipGetLastError());
  }
}

}  // namespace adc2g
