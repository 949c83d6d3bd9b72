// INT-form coupling on the CSF vectors: operand layouts, the occupied term
// and the sum of the 1h1p partials (the virtual contractions are in
// csf_virt.hpp).
//
// With x the CSF amplitudes (index maps in kernels.hip) and, for a <= b,
//   V4[l][c][ab] = ((ac|bl) + (bc|al)) / sqrt2   (a < b),   V4[l][c][aa] = (ac|al)
//   V5[l][c][ab] = sqrt(3/2) ((ac|bl) - (bc|al))
//   O4[kl][m][b] = ((km|bl) + (lm|bk)) / sqrt2,  O2[k][m][b] = -(km|bk)
//   O5[kl][m][b] = sqrt(3/2) ((km|bl) - (lm|bk))
// the coupling needs no pair tensor: for k < l
//   w4[kl][ab] = sum_c V4[l][c][ab] x(c,k) + V4[k][c][ab] x(c,l)
//                - sum_m x(a,m) O4[kl][m][b] + x(b,m) O4[kl][m][a]
//   w5[kl][ab] = the same with V5, O5 and a minus sign on each second term
//   w2[ab][k]  = -sqrt2 sum_c V4[k][c][ab] x(c,k) - sum_m x(a,m) O2[k][m][b] + x(b,m) O2[k][m][a]
// t3 and t1 are the a = b entries of the t4 and t2 forms (occupied part times
// 1/sqrt2), and the down terms are the transposes.  The pair of rows (k, l)
// and (l, k) of a CSF is thus two entries of one product over the virtual
// index, so the vectors are read and written in their own order: the pair
// tensor form moved n1^2 elements three times per direction beside them.  20
// vectors at o=16, v=200: FP64 5.70 -> 3.81 ms, FP32 3.91 -> 2.59 ms; 7 vectors
// at o=13, v=117: 0.61 -> 0.39 ms; two at o=16, v=200: 0.92 -> 0.58 ms; one at
// o=5, v=36: 67 -> 38 us.
#include "csf.hpp"

#include <algorithm>

namespace adc2g {

namespace {

constexpr double SQ2 = 1.4142135623730951;
constexpr double ISQ2 = 0.7071067811865476;
constexpr double SQ32 = 1.2247448713915890;  // sqrt(3/2)

__device__ __forceinline__ int64_t row_start(int64_t a, int64_t v) { return a * v - a * (a + 1) / 2 - a - 1; }

// p = pair number of a < b among n
__device__ __forceinline__ void unpair(int64_t p, int64_t n, int& lo, int& hi) {
  const double nn = (double)(2 * n - 1);
  int64_t a = (int64_t)floor((nn - sqrt(fmax(nn * nn - 8.0 * (double)p, 0.0))) * 0.5);
  if (a < 0) a = 0;
  if (a > n - 2) a = n - 2;
  while (a > 0 && row_start(a, n) + a + 1 > p) --a;
  while (a + 1 < n - 1 && row_start(a + 1, n) + a + 2 <= p) ++a;
  lo = (int)a;
  hi = (int)(p - row_start(a, n));
}

// One workgroup per (chunk, RB virtual rows c): the (ac|bl), (bc|al) of its
// pairs are read along l, combined, turned in LDS and written as whole
// 128-byte rows.  Within a row the 16-byte pieces are permuted by c & 7, so
// that 16-byte LDS reads of one piece of eight consecutive rows touch all
// banks after a linear copy of the rows into LDS.
template <class T>
__global__ void __launch_bounds__(256) csf_build_v_kernel(const double* __restrict__ V, CsfGeo g, int RB,
                                                           T* __restrict__ out) {
  constexpr int P = csf_pairs<T>(), EV = 16 / (int)sizeof(T);
  extern __shared__ char smraw[];
  T* sm = (T*)smraw;  // [slab][RB][P]
  __shared__ int pa[P], pb[P];
  const int o = g.o, v = g.v;
  const int ch = blockIdx.x;
  const bool diag = ch >= g.nch;
  const int c0 = blockIdx.y * RB;
  const int64_t p0 = (int64_t)(diag ? ch - g.nch : ch) * P;
  if (threadIdx.x < P) {
    const int64_t p = p0 + threadIdx.x;
    int a = -1, b = -1;
    if (diag) {
      if (p < v) a = b = (int)p;
    } else if (p < g.npv) {
      unpair(p, v, a, b);
    }
    pa[threadIdx.x] = a;
    pb[threadIdx.x] = b;
  }
  __syncthreads();
  const int64_t n1 = (int64_t)o * v;
  const int per = P * o;
  for (int t = threadIdx.x; t < RB * per; t += 256) {
    const int r = t / per, pl = t - r * per, p = pl / o, l = pl - p * o;
    const int a = pa[p], b = pb[p], c = c0 + r;
    double x4 = 0.0, x5 = 0.0;
    if (a >= 0 && c < v) {
      const double g1 = V[((int64_t)a * v + c) * n1 + (int64_t)b * o + l];
      if (diag) {
        x4 = g1;
      } else {
        const double g2 = V[((int64_t)b * v + c) * n1 + (int64_t)a * o + l];
        x4 = ISQ2 * (g1 + g2);
        x5 = SQ32 * (g1 - g2);
      }
    }
    const int pos = (((p / EV) ^ (c & 7)) * EV) + p % EV;
    sm[(l * RB + r) * P + pos] = (T)x4;
    if (!diag) sm[((o + l) * RB + r) * P + pos] = (T)x5;
  }
  __syncthreads();
  const int slabs = diag ? o : 2 * o;
  const int64_t u0 = diag ? (int64_t)g.nch * 2 * o + (int64_t)(ch - g.nch) * o : (int64_t)ch * 2 * o;
  for (int t = threadIdx.x; t < slabs * RB * P; t += 256) {
    const int s = t / (RB * P), rp = t - s * RB * P, r = rp / P;
    if (c0 + r < v) out[((u0 + s) * v + c0) * P + rp] = sm[t];
  }
}

__global__ void csf_build_o_kernel(const double* __restrict__ O, DimsK d, int om, double* __restrict__ out) {
  const int o = d.o, v = d.v, vp = (v + 15) / 16 * 16;
  const int64_t n1 = d.n1;
  const int64_t total = (2 * d.npo + o) * (int64_t)vp * om;
  for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int m = (int)(idx % om);
    const int b = (int)((idx / om) % vp);
    int64_t s = idx / ((int64_t)om * vp);
    double x = 0.0;
    if (m < o && b < v) {
      if (s >= d.npo && s < d.npo + o) {
        const int k = (int)(s - d.npo);
        x = -O[((int64_t)k * o + m) * n1 + (int64_t)b * o + k];
      } else {
        const bool five = s >= d.npo + o;
        int k, l;
        unpair(five ? s - d.npo - o : s, o, k, l);
        const double g1 = O[((int64_t)k * o + m) * n1 + (int64_t)b * o + l];
        const double g2 = O[((int64_t)l * o + m) * n1 + (int64_t)b * o + k];
        x = five ? SQ32 * (g1 - g2) : ISQ2 * (g1 + g2);
      }
    }
    out[idx] = x;
  }
}

// Occupied term, both directions, and the 2h2p diagonal, in FP64 at every
// GEMM precision.  Bound by the vectors: x2 is read once and W2 written once
// (1.64 GB for 20 vectors at o=16, v=200), 2 o products per element and
// direction on FP64 MFMA.  One wave owns a 16 x 16 tile of virtuals (a, b),
// a <= b, for VG vectors and a slice of the sets (the pairs k < l of t4/t3,
// the k of t2/t1, the pairs of t5); the 1h1p sums over the sets stay in its
// registers.  The x tile is loaded with b along the lanes (128-byte runs);
// as an MFMA operand it is then its own transpose, which gives the sum over
// a; the sum over b, and the down operands, take x and O through LDS.  The
// loads of a set are issued before the products and stores of the set before
// it: loads and stores retire in order, so a load issued after the stores
// would wait for them too.  The four waves of a workgroup take neighbouring b
// tiles set by set together: a run of 16 pairs starts anywhere in a cache
// line, and the line's other part is the neighbour's.
template <int OM, int VG>
struct OccSet {
  static constexpr int KK = OM / 4;
  double x[VG][4];
  double a[KK], b[KK];            // O of the a and b tiles: row li, m = KK*gq + e
  uint32_t base, dbase, stride;   // positions of the entries in a vector (uniform)
  double ekl;
  int five, two;
};

template <int OM, int VG, bool UP, bool DOWN>
__global__ void __launch_bounds__(256, OM == 16 && VG == 1 ? 3 : 2)
csf_occ_kernel(CsfGeo g, int nt, int sl, const double* __restrict__ X, const double* __restrict__ Oc,
               const double* __restrict__ eps, double* __restrict__ W, double* __restrict__ part,
               double* __restrict__ T2) {
  typedef double v4 __attribute__((ext_vector_type(4)));
  typedef OccSet<OM, VG> Set;
  constexpr int KK = OM / 4;   // K steps over the occupied index (up)
  constexpr int NJ = OM / 16;  // 16-column blocks of the occupied index (down)
  constexpr int OR = OM + 2;   // LDS row of an O block (16-byte aligned)
  __shared__ double tr[4][VG][16 * 17];
  __shared__ __attribute__((aligned(16))) double to[4][2][16 * OR];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, gq = lane >> 4;
  const int o = g.o, v = g.v;
  // blockIdx.x: vector group fastest (the workgroups of one tile share the
  // set operands), then slice, then tiles
  const int vgs = (g.nv + VG - 1) / VG;
  int w = xcd_tile(blockIdx.x, gridDim.x);
  const int vg = uniform(w % vgs);
  w = uniform(w / vgs);
  const int slice = uniform(w % sl);
  w = uniform(w / sl);
  // four consecutive tiles of the list (ta, tb >= ta), tb fastest
  const int ntile = nt * (nt + 1) / 2;
  const int tix = min(w * 4 + wv, ntile - 1);
  const bool active = w * 4 + wv < ntile;
  int ta = 0, tb = tix;
  while (tb >= nt - ta) tb -= nt - ta++;
  tb += ta;
  ta = uniform(ta);
  tb = uniform(tb);
  const int v0 = vg * VG, nvec = min(VG, g.nv - v0);
  const int ns = 2 * g.npo + o;
  const int s_begin = uniform(ns * slice / sl), s_end = uniform(ns * (slice + 1) / sl);
  const int vp = nt * 16;
  const bool dtile = ta == tb;

  // x1 of the a and b virtuals: operand entry (row li, m = KK*gq + s) of step s
  double xa[VG][KK], xb[VG][KK];
  if (UP) {
#pragma unroll
    for (int j = 0; j < VG; ++j)
#pragma unroll
      for (int s = 0; s < KK; ++s) {
        const int m = KK * gq + s;
        const int a = ta * 16 + li, b = tb * 16 + li;
        const double* x = X + g.ldx * (v0 + min(j, nvec - 1));
        xa[j][s] = (m < o && a < v) ? x[(int64_t)a * o + m] : 0.0;
        xb[j][s] = (m < o && b < v) ? x[(int64_t)b * o + m] : 0.0;
      }
  }
  v4 ya[VG][NJ], yb[VG][NJ];
#pragma unroll
  for (int j = 0; j < VG; ++j)
#pragma unroll
    for (int n = 0; n < NJ; ++n) {
      ya[j][n] = (v4){0, 0, 0, 0};
      yb[j][n] = (v4){0, 0, 0, 0};
    }
  // the lane's four tile entries: a = ta*16 + 4 r + gq, b = tb*16 + li
  const int b = tb * 16 + li;
  const double eb = b < v ? eps[o + b] : 0.0;
  uint32_t pv[4];
  double ea[4];
  bool ok[4], dg[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int a = ta * 16 + 4 * r + gq;
    ok[r] = active && b < v && a <= b;
    dg[r] = a == b;
    pv[r] = !ok[r] ? 0u : (dg[r] ? (uint32_t)a : (uint32_t)(row_start(a, v) + b));
    ea[r] = (a < v ? eps[o + a] : 0.0) + eb;
  }
  const double* xv[VG];
#pragma unroll
  for (int j = 0; j < VG; ++j) xv[j] = X + g.ldx * (v0 + min(j, nvec - 1));
  double* wj[VG];
#pragma unroll
  for (int j = 0; j < VG; ++j) wj[j] = W + g.ldw * (v0 + min(j, nvec - 1));

  int k = 0, l = 1, q = 0;  // occupied pair of the next set to load
  if (s_begin < g.npo || s_begin > g.npo + o) {
    q = s_begin < g.npo ? s_begin : s_begin - g.npo - o;
    unpair(q, o, k, l);
  }
  k = uniform(k);
  l = uniform(l);
  q = uniform(q);
  const uint32_t npv = (uint32_t)g.npv, off1 = (uint32_t)g.off1, off2 = (uint32_t)g.off2, off3 = (uint32_t)g.off3,
                 off4 = (uint32_t)g.off4, off5 = (uint32_t)g.off5;
  int k_last = k, l_last = l, q_last = q;
  int sn = s_begin;  // next set to load
  auto load = [&](Set& S) ADC2G_INLINE {
    const bool two = sn >= g.npo && sn < g.npo + o, five = sn >= g.npo + o;
    if (sn == g.npo + o) { k = 0; l = 1; q = 0; }
    const int ka = two ? sn - g.npo : k, la = two ? sn - g.npo : l;
    const uint32_t base = two ? off2 + ka : (five ? +off5 : +off4) + q * npv;
    const uint32_t stride = two ? o : 1;
    const uint32_t dbase = two ? off1 + ka * v : off3 + q * v;
    S.five = five ? 1 : 0;
    S.two = two ? 1 : 0;
    S.base = base;
    S.dbase = dbase;
    S.stride = stride;
    S.ekl = eps[ka] + eps[la];
    uint32_t at[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) at[r] = dg[r] ? dbase + pv[r] : base + pv[r] * stride;
#pragma unroll
    for (int j = 0; j < VG; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) S.x[j][r] = xv[j][at[r]];  // (entries outside read entry 0 of the set)
    const double* Oa = Oc + ((int64_t)sn * vp + ta * 16) * OM;
    const double* Ob = Oc + ((int64_t)sn * vp + tb * 16) * OM;
#pragma unroll
    for (int e = 0; e < KK; ++e) {
      S.a[e] = Oa[li * OM + KK * gq + e];
      S.b[e] = Ob[li * OM + KK * gq + e];
    }
    if (!two) {
      ++q;
      if (++l >= o) { ++k; l = k + 1; }
    }
    ++sn;
  };
  // The results of a set are stored after the loads of the set after the next
  // have been issued and those of the next have landed: every wait for loads
  // also waits for the stores issued before them, which by then are a whole
  // set old.
  double val[VG][4];
  uint32_t s_base = 0, s_dbase = 0, s_stride = 0;
  int s_five = 0;
  auto store = [&]() ADC2G_INLINE {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const uint32_t at = dg[r] ? s_dbase + pv[r] : s_base + pv[r] * s_stride;
      if (ok[r] && !(s_five && dg[r])) {
#pragma unroll
        for (int j = 0; j < VG; ++j)
          if (j < nvec) wj[j][at] = val[j][r];
      }
    }
  };
  auto landed = [&](Set& S) ADC2G_INLINE {
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int j = 0; j < VG; ++j) asm volatile("" : "+v"(S.x[j][r]));
#pragma unroll
    for (int e = 0; e < KK; ++e) asm volatile("" : "+v"(S.a[e]), "+v"(S.b[e]));
  };
  auto in_ = [&](const Set& S, int r) ADC2G_INLINE { return ok[r] && !(S.five && dg[r]); };
  auto use = [&](Set& S) ADC2G_INLINE {
    const double sg = S.five ? -1.0 : 1.0;
#pragma unroll
    for (int e = 0; e < KK; ++e) S.a[e] *= sg;
    if (DOWN) {
#pragma unroll
      for (int e = 0; e < KK; ++e) {
        to[wv][0][li * OR + KK * gq + e] = S.a[e];
        to[wv][1][li * OR + KK * gq + e] = S.b[e];
      }
#pragma unroll
      for (int j = 0; j < VG; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          // (the 1h1p sums take a diagonal entry once from each side)
          S.x[j][r] = in_(S, r) ? S.x[j][r] : 0.0;
          tr[wv][j][(4 * r + gq) * 17 + li] = dtile && dg[r] ? ISQ2 * S.x[j][r] : S.x[j][r];
        }
      __builtin_amdgcn_wave_barrier();
      if (S.two) {  // uniform: o of the 2 npo + o sets
#pragma unroll
        for (int j = 0; j < VG; ++j) {
          double* t2 = T2 + ((int64_t)(v0 + j) * o + (S.base - off2)) * (g.npv + v);
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (ok[r] && j < nvec) t2[dg[r] ? npv + pv[r] : pv[r]] = -SQ2 * S.x[j][r];
        }
      }
    }
    if (UP) {
#pragma unroll
      for (int j = 0; j < VG; ++j) {
        v4 acc = (v4){0, 0, 0, 0}, acc2 = (v4){0, 0, 0, 0};
#pragma unroll
        for (int e = 0; e < KK; ++e) {
          acc = Mma<double>::mma(xa[j][e], S.b[e], acc);
          acc2 = Mma<double>::mma(S.a[e], xb[j][e], acc2);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const double sum = acc[r] + acc2[r];
          val[j][r] = (ea[r] - S.ekl) * S.x[j][r] - (dg[r] ? ISQ2 * sum : sum);
        }
      }
      s_base = S.base;
      s_dbase = S.dbase;
      s_stride = S.stride;
      s_five = S.five;
    }
    if (DOWN) {
      double oa[NJ][4], ob[NJ][4];  // row m = 16 n + li of the a = 4 e + gq (b) virtual
#pragma unroll
      for (int n = 0; n < NJ; ++n)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          oa[n][e] = to[wv][0][(4 * e + gq) * OR + n * 16 + li];
          ob[n][e] = to[wv][1][(4 * e + gq) * OR + n * 16 + li];
        }
#pragma unroll
      for (int j = 0; j < VG; ++j) {
        const double* t = tr[wv][j];
        double xr[4];  // x(a = li, b = 4 e + gq)
#pragma unroll
        for (int e = 0; e < 4; ++e) xr[e] = t[li * 17 + 4 * e + gq];
        if (dtile) {
#pragma unroll
          for (int r = 0; r < 4; ++r) S.x[j][r] *= dg[r] ? ISQ2 : 1.0;
        }
#pragma unroll
        for (int n = 0; n < NJ; ++n)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            yb[j][n] = Mma<double>::mma(oa[n][e], S.x[j][e], yb[j][n]);
            ya[j][n] = Mma<double>::mma(ob[n][e], xr[e], ya[j][n]);
          }
      }
    }
  };
  // the last set is loaded again rather than none, so that the number of
  // loads in flight does not depend on where the loop ends
  auto next = [&](Set& S) ADC2G_INLINE {
    if (sn >= s_end) {
      sn = s_end - 1;
      k = k_last;
      l = l_last;
      q = q_last;
    }
    k_last = k;
    l_last = l;
    q_last = q;
    load(S);
  };
  if (s_begin < s_end) {
    Set A, B;
    next(A);
    bool first = true;
    for (int s = s_begin; s < s_end; s += 2) {
      next(B);
      landed(A);
      __syncthreads();
      if (UP && !first) store();
      use(A);
      next(A);
      landed(B);
      __syncthreads();
      if (UP) store();
      if (s + 1 < s_end) use(B);
      first = s + 1 >= s_end;
    }
    if (UP && !first) store();
  }
  if (DOWN && active) {
    // slot (of the nt that add up to a tile): the other tile's number
    const int64_t n1 = (int64_t)o * v;
#pragma unroll
    for (int j = 0; j < VG; ++j) {
      if (j >= nvec) break;
#pragma unroll
      for (int n = 0; n < NJ; ++n) {
        // row k of the lane's register r, column li of the tile
        const int a = ta * 16 + li, bb = tb * 16 + li;
        double* pa = part + (((int64_t)slice * nt + tb) * g.nv + v0 + j) * n1;
        double* pb = part + (((int64_t)slice * nt + ta) * g.nv + v0 + j) * n1;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int kk = n * 16 + 4 * r + gq;
          if (kk >= o) continue;
          if (dtile) {
            if (a < v) pa[(int64_t)kk * v + a] = -(ya[j][n][r] + yb[j][n][r]);
          } else {
            if (a < v) pa[(int64_t)kk * v + a] = -ya[j][n][r];
            if (bb < v) pb[(int64_t)kk * v + bb] = -yb[j][n][r];
          }
        }
      }
    }
  }
}

// W1[a o + k] += the partials of both terms, in a fixed order: eight threads
// a sum, each over every eighth partial.
template <class Acc>
__global__ void __launch_bounds__(256) csf_reduce_kernel(CsfGeo g, int ds, const Acc* __restrict__ down, int no,
                                                         const double* __restrict__ occ, double* __restrict__ W) {
  __shared__ double red[8][32];
  const int64_t n1 = (int64_t)g.o * g.v, total = n1 * g.nv;
  const int x = threadIdx.x & 31, y = threadIdx.x >> 5;
  const int64_t idx = (int64_t)blockIdx.x * 32 + x;
  double s = 0.0;
  if (idx < total) {
    // idx = (vec, k, a)
    double s0 = 0.0, s1 = 0.0;
    int e = y;
    for (; e + 8 < ds; e += 16) {
      s0 += (double)down[(int64_t)e * total + idx];
      s1 += (double)down[(int64_t)(e + 8) * total + idx];
    }
    if (e < ds) s0 += (double)down[(int64_t)e * total + idx];
    for (int f = y; f < no; f += 8) s1 += occ[(int64_t)f * total + idx];
    s = s0 + s1;
  }
  red[y][x] = s;
  __syncthreads();
  if (y == 0 && idx < total) {
    double t = 0.0;
#pragma unroll
    for (int e = 0; e < 8; ++e) t += red[e][x];
    const int64_t row = idx / g.v;
    const int a = (int)(idx - row * g.v);
    const int64_t vec = row / g.o;
    const int k = (int)(row - vec * g.o);
    W[g.ldw * vec + (int64_t)a * g.o + k] += t;
  }
}

template <int OM, int VG>
void occ_launch(const CsfGeo& g, const CsfPlan& p, const double* X, const double* Oc, const double* eps, double* W,
                double* part, double* T2, bool up, bool down, hipStream_t st) {
  const int tiles = (p.nt * (p.nt + 1) / 2 + 3) / 4;
  const dim3 grid((unsigned)(tiles * p.sl * ((g.nv + VG - 1) / VG)));
  if (up && down)
    hipLaunchKernelGGL((csf_occ_kernel<OM, VG, true, true>), grid, dim3(256), 0, st, g, p.nt, p.sl, X, Oc, eps, W, part, T2);
  else if (up)
    hipLaunchKernelGGL((csf_occ_kernel<OM, VG, true, false>), grid, dim3(256), 0, st, g, p.nt, p.sl, X, Oc, eps, W,
                       part, T2);
  else
    hipLaunchKernelGGL((csf_occ_kernel<OM, VG, false, true>), grid, dim3(256), 0, st, g, p.nt, p.sl, X, Oc, eps, W,
                       part, T2);
  HIP_CHECK(hipGetLastError());
}

}  // namespace

template <class T>
void launch_csf_build_v(const double* V, const DimsK& d, T* out, hipStream_t st) {
  const CsfGeo g = csf_geo<T>(d, 1, 0, 0);
  const int rb = d.o <= 16 ? 8 : 4;  // 32 KiB of LDS
  const size_t lds = (size_t)2 * d.o * rb * 128;
  hipLaunchKernelGGL((csf_build_v_kernel<T>), dim3(g.nch + g.nchd, (d.v + rb - 1) / rb), dim3(256), lds, st, V, g, rb,
                     out);
  HIP_CHECK(hipGetLastError());
  // the rows that whole-tile loads read past the end
  const size_t n = csf_v_elems<T>(d);
  HIP_CHECK(hipMemsetAsync(out + n - 16 * csf_pairs<T>(), 0, 16 * 128, st));
}

void launch_csf_build_o(const double* O, const DimsK& d, double* out, hipStream_t st) {
  hipLaunchKernelGGL(csf_build_o_kernel, dim3(grid_for((int64_t)csf_o_elems(d))), dim3(256), 0, st, O, d, csf_om(d.o),
                     out);
  HIP_CHECK(hipGetLastError());
}

// vectors a wave of the occupied kernel takes together
static int csf_occ_vectors(int o, int nv) { return o <= 16 && nv > 1 ? 2 : 1; }

CsfPlan csf_plan(const DimsK& d, int nv) {
  CsfPlan p;
  const int o = d.o, v = d.v;
  const int rows = nv * o, waves = (rows + 15) / 16;
  // down: rows in groups of dw waves (4, or fewer when there are no more),
  // columns in equal splits of at most 13 blocks of 16, K split so that about
  // two workgroups per CU are in flight, each with three slabs or more: with
  // fewer the sum over the splits grows, with more the chain of a workgroup does
  // (whole product with at least 1, 2, 3, 4, 8 slabs, FP64: o=4, v=24, 20 vectors
  // 40.6, 41.0, 42.3, 43.2, 47.8 us; o=5, v=36, 20 vectors 53.5, 50.3, 50.6, 51.9,
  // 56.4; o=8, v=60, one vector 54.4, 53.6, 52.1, 52.6, 57.3)
  const int nb = (v + 15) / 16;
  p.dns = (nb + 12) / 13;
  p.dnb = (nb + p.dns - 1) / p.dns;
  p.dns = (nb + p.dnb - 1) / p.dnb;
  p.dw = std::min(4, waves);
  if (waves > 4 && waves <= 8) p.dw = (waves + 1) / 2;
  p.dg = (waves + p.dw - 1) / p.dw;
  const CsfGeo g8 = csf_geo<double>(d, nv, 0, 0), g4 = csf_geo<float>(d, nv, 0, 0);
  const int64_t tiles = std::min((int64_t)(2 * g8.nch + g8.nchd), (int64_t)(2 * g4.nch + g4.nchd)) * o;
  p.ds = (int)std::max<int64_t>(1, std::min<int64_t>(tiles / 3, 512 / ((int64_t)p.dg * p.dns)));
  // one pass for both directions where the rows fit two 16-row blocks and a
  // slab's columns the registers, and every workgroup has work for two rounds
  // also with the fewer chunks of FP32, that is from v = 128 on (o=16, v=200:
  // one vector 0.29 ms against 0.26 + 0.27 in two passes, two vectors 0.49
  // against 0.33 + 0.30; o=5, v=36, 83 chunks: 17 us against 15).  A whole
  // product of one vector, one pass against two, FP64 and FP32: o=16, v=128 147
  // against 220 and 134 against 148 us, o=3, v=128 55 against 57 and 50 against
  // 51; o=5, v=112 70 against 65 and 66 against 60
  const int items = 2 * g4.nch + g4.nchd;
  p.thin = (o <= 16 && rows <= 32 && v <= 208 && items >= 512) ? 256 : 0;
  p.down_bytes = (size_t)std::max(p.ds, p.thin) * rows * v * sizeof(double);
  // up: whole vectors per workgroup, the number of waves that pads least; no
  // more vectors than leave each CU a workgroup (64 vectors, FP64: o=2, v=4 53 ->
  // 29 us, o=2, v=16 58 -> 36; pair tensors took 53 and 67)
  const int wmax = o <= 16 ? 8 : 4;
  const int groups = std::min(nv, std::max(1, 256 / (2 * g8.nch + g8.nchd))), cap = (nv + groups - 1) / groups;
  double best = 1e300;
  for (int w : {4, 8, 6, 2, 1}) {
    if (w > wmax || 16 * w < o) continue;
    const int vpb = std::min(cap, 16 * w / o), grp = (nv + vpb - 1) / vpb;
    const double cost = (double)grp * w * (w == 6 ? 1.05 : 1.0);
    if (cost < best) {
      best = cost;
      p.uw = w;
      p.uvpb = vpb;
      p.ug = grp;
    }
  }
  p.nt = nb;
  // occupied: slices of the sets so that the workgroups come in whole rounds
  // of two per CU (three with one vector each: their registers); the fewest
  // slices among equals, at most 32 and, where those leave the round unfilled,
  // 64 (one vector, FP32: o=32, v=33 167 -> 136 us, o=30, v=60 182 -> 155; pair
  // tensors took 138 and 176)
  const int vgl = csf_occ_vectors(o, nv), vgs = (nv + vgl - 1) / vgl;
  const int64_t slots = o <= 16 && vgl == 1 ? 768 : 512;
  const int64_t wgs = (int64_t)(nb * (nb + 1) / 2 + 3) / 4 * vgs;
  double beff = 0.0;
  p.sl = 1;
  for (int sl = 1; sl <= 64 && sl <= (int)(2 * d.npo + o + 3) / 4; ++sl) {
    const int64_t n = wgs * sl;
    if ((n > 2048 && sl > 1) || (n > slots && sl > 32)) break;
    const double eff = (double)n / (double)((n + slots - 1) / slots * slots);
    if (eff > 1.03 * beff) {
      beff = eff;
      p.sl = sl;
    }
  }
  p.occ_bytes = (size_t)p.sl * nb * nv * o * v * sizeof(double);
  p.t2_bytes = (size_t)nv * o * (size_t)(d.npv + v) * sizeof(double);
  return p;
}

CsfBytes csf_workspace(const DimsK& d, int nv) {
  CsfBytes b;
  for (int n = 1; n <= nv; ++n) {
    const CsfPlan p = csf_plan(d, n);
    b.down = std::max(b.down, p.down_bytes);
    b.occ = std::max(b.occ, p.occ_bytes);
    b.t2 = std::max(b.t2, p.t2_bytes);
  }
  return b;
}

void launch_csf_occ(const CsfGeo& g, const CsfPlan& p, const double* X, const double* Oc, const double* eps,
                    double* W, double* part, double* T2, bool up, bool down, hipStream_t st) {
  if (g.o <= 16 && csf_occ_vectors(g.o, g.nv) == 1)
    occ_launch<16, 1>(g, p, X, Oc, eps, W, part, T2, up, down, st);
  else if (g.o <= 16)
    occ_launch<16, 2>(g, p, X, Oc, eps, W, part, T2, up, down, st);
  else
    occ_launch<32, 1>(g, p, X, Oc, eps, W, part, T2, up, down, st);
}

template <class Acc>
void launch_csf_reduce(const CsfGeo& g, const CsfPlan& p, int ndown, const Acc* down, const double* occ, double* W,
                       hipStream_t st) {
  const int64_t total = (int64_t)g.o * g.v * g.nv;
  hipLaunchKernelGGL((csf_reduce_kernel<Acc>), dim3((unsigned)((total + 31) / 32)), dim3(256), 0, st, g, ndown, down,
                     p.sl * p.nt, occ, W);
  HIP_CHECK(hipGetLastError());
}

template void launch_csf_build_v<double>(const double*, const DimsK&, double*, hipStream_t);
template void launch_csf_build_v<float>(const double*, const DimsK&, float*, hipStream_t);
template void launch_csf_reduce<double>(const CsfGeo&, const CsfPlan&, int, const double*, const double*, double*,
                                        hipStream_t);
template void launch_csf_reduce<float>(const CsfGeo&, const CsfPlan&, int, const float*, const double*, double*,
                                       hipStream_t);

}  // namespace adc2g
