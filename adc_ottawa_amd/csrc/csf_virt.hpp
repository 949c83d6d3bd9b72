// Virtual contractions of the CSF form (see csf.hip for the operands), one
// template for FP64 and FP32 MFMA; instantiated in csf_f64.hip, csf_f32.hip.
//
// Layout of the virtual operand: for each chunk of P = 128 bytes of pairs, the
// slabs (t4, l), (t5, l) (diagonal chunks: (t4, l) only), each v rows c of P
// pairs.  Both directions read it: down, a slab is one K tile (the pairs) of
// all output columns c; up, 16 rows of every slab of a (chunk, type) are one K
// tile (c) of all output columns (l, pair).  Either way whole runs of 128-byte
// rows go to LDS by direct 16-byte loads, and the waves own the rows (vector,
// k) of the product, so that every wave has the same number of MFMAs whatever
// v is (the 16-column blocks of v = 200, 13, do not split evenly over 4 or 8
// waves).
#pragma once

#include "csf.hpp"

namespace adc2g {

namespace csfv {

constexpr double SQ2 = 1.4142135623730951;

__device__ __forceinline__ int64_t po_index(int lo, int hi, int n) {
  return (int64_t)lo * n - (int64_t)lo * (lo + 1) / 2 + (hi - lo - 1);
}

// 1 KiB of global memory to LDS, 16 bytes a lane, both sides contiguous: `base`
// and `off` are uniform, so that the address takes no VALU instruction.  (An
// FP64 MFMA holds the VALU of its SIMD: the address and masking arithmetic
// of a K tile comes out of the MFMA time of both waves there.  With 63 VALU
// instructions to 52 MFMAs the down kernel kept the MFMAs 74 % busy, with two
// waves as with one.)
typedef __amdgpu_buffer_rsrc_t Rsrc;
__device__ __forceinline__ Rsrc lds_source(const char* base) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, 0x7fffffff, 0x00027000);
}
__device__ __forceinline__ void lds_copy(Rsrc base, int off, char* dst, int lane16) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(base, (__attribute__((address_space(3))) void*)dst, 16, lane16, off, 0, 0);
}

// all direct loads of this wave have landed, and every wave's have after the barrier
__device__ __forceinline__ void lds_ready() {
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
  __syncthreads();
}

// ---- down: part[split][(vec,k)][c] = sum over the split's slabs (chunk, t, l)
// and pairs p of x_t(kl, p) V_t[l][c][p].  The row (vec, k) of a slab reads
// the CSFs of the pair (k, l) -- t5 with a minus sign for k > l -- or, for
// k = l, T2, the k-major copy of -sqrt2 times t2 and t1 (t4 slabs), and
// nothing (t5 slabs); in the diagonal chunks t3 and t1 take their places.  K
// order within a slab: lane group g holds the pairs g*KS .. g*KS + KS-1, step
// s its s-th.  Where each row of a slab starts is looked up in LDS (`tab`, one
// address per (t, l) and row; rows that read nothing point to zeros), so that
// a slab's operand costs one address and its loads.
template <class T, int NB>
__global__ void __launch_bounds__(512, NB > 5 ? 2 : 3)
down_kernel(CsfGeo g, int ds, int dg, int dns, const double* __restrict__ X, const double* __restrict__ T2,
            const double* __restrict__ zeros, const T* __restrict__ V, typename Mma<T>::Acc* __restrict__ part) {
  typedef Mma<T> MT;
  typedef typename MT::v4 v4;
  constexpr int KS = 32 / (int)sizeof(T);  // pairs per lane and slab
  constexpr int P = 4 * KS;
  __shared__ __attribute__((aligned(1024))) char s0[NB * 2048];
  __shared__ __attribute__((aligned(1024))) char s1[NB * 2048];
  extern __shared__ uint64_t tab[];  // [(t, l)][row]
  const int lane = threadIdx.x & 63, nw = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, gq = lane >> 4;
  const int o = g.o, v = g.v;
  int w = xcd_tile(blockIdx.x, gridDim.x);
  const int grp = uniform(w % dg);
  w = uniform(w / dg);
  const int ks = uniform(w / dns);
  const int n0 = (w - ks * dns) * NB * 16;
  const int rows = g.nv * o;
  const int row = (grp * nw + wave) * 16 + li;
  const bool live = row < rows;
  const int vec = live ? row / o : 0, k = live ? row - vec * o : 0;
  const double* xv = X + g.ldx * vec;
  const double* t2v = T2 + (int64_t)(vec * o + k) * (g.npv + v);
  const int u_all = (2 * g.nch + g.nchd) * o;
  const int u_begin = uniform((int)((int64_t)u_all * ks / ds)), u_end = uniform((int)((int64_t)u_all * (ks + 1) / ds));
  const int64_t slab = (int64_t)v * 128;
  const char* vsrc = (const char*)V + (int64_t)n0 * 128;
  const int nrow8 = min(NB * 2, ((v + 15) / 16 * 16 - n0) / 8);
  const int nch = g.nch, npv = (int)g.npv;

  // the slab whose operand is loaded next: chunk, index (t, l) within it
  const int u_off = 2 * nch * o;
  int diag = u_begin >= u_off ? 1 : 0;
  const int per0 = diag ? o : 2 * o;
  int c = uniform((diag ? u_begin - u_off : u_begin) / per0);
  int tl = (diag ? u_begin - u_off : u_begin) - c * per0;
  // each wave fills and reads the entries of its own rows
  auto fill = [&](int dg1) ADC2G_INLINE {
    for (int i = gq; i < (dg1 ? o : 2 * o); i += 4) {
      const int t = i >= o ? 1 : 0, l = i - t * o;
      const double* e = zeros;
      if (live) {
        if (l == k) {
          if (dg1) e = t2v + g.npv;
          else if (!t) e = t2v;
        } else {
          const int64_t q = po_index(min(k, l), max(k, l), o);
          e = xv + (dg1 ? g.off3 + q * v : (t ? g.off5 : g.off4) + q * g.npv);
        }
      }
      tab[i * (nw * 16) + wave * 16 + li] = (uint64_t)e;
    }
    __builtin_amdgcn_wave_barrier();
  };
  fill(diag);
  const uint64_t* my = tab + wave * 16 + li;
  const int tstep = nw * 16;
  // operand of a slab: the lane's KS values as loaded, and what the slab is
  double xr[KS];
  int x_t = 0, x_l = 0, x_left = 0;  // type, l, pairs that count (>= P but in the last chunk)
  uint64_t entry = my[tl * tstep];
  uint64_t at = (uint64_t)(c * P + gq * KS) * 8;
  typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));
  auto load_x = [&]() ADC2G_INLINE {
    x_t = tl >= o ? 1 : 0;
    x_l = tl - x_t * o;
    x_left = (diag ? v : npv) - c * P;
    const double* e = (const double*)(entry + at);
    if (x_left >= P) {
#pragma unroll
      for (int s = 0; s < KS; s += 2) {
        const d2u y = *(const d2u*)(e + s);
        xr[s] = y[0];
        xr[s + 1] = y[1];
      }
    } else {  // the row ends in this chunk: no read past it
#pragma unroll
      for (int s = 0; s < KS; ++s) xr[s] = *(const double*)(gq * KS + s < x_left ? (uint64_t)(e + s) : entry);
    }
    // the entry of the slab after
    if (++tl == (diag ? o : 2 * o)) {
      tl = 0;
      if (++c == nch && !diag) {
        c = 0;
        diag = 1;
        fill(1);
      }
      at = (uint64_t)(c * P + gq * KS) * 8;
    }
    entry = my[tl * tstep];
  };
  auto operand = [&](T (&a)[KS]) ADC2G_INLINE {
    if (x_left < P) {
#pragma unroll
      for (int s = 0; s < KS; ++s) xr[s] = gq * KS + s < x_left ? xr[s] : 0.0;
    }
    if (x_t) {
      const bool neg = x_l < k;
#pragma unroll
      for (int s = 0; s < KS; ++s) xr[s] = neg ? -xr[s] : xr[s];
    }
#pragma unroll
    for (int s = 0; s < KS; ++s) a[s] = (T)xr[s];
  };
  const int lane16 = lane * 16;
  auto dma = [&](int u, char* buf) ADC2G_INLINE {
    const Rsrc src = lds_source(vsrc + u * slab);
    // (blocks past the last virtual are skipped: their columns are not stored)
    for (int i = wave; i < nrow8; i += nw) lds_copy(src, i * 1024, buf + i * 1024, lane16);
  };
  v4 acc[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) acc[j] = (v4){0, 0, 0, 0};
  // FP32: sums of 8 slabs (256 products) are added up apart, so that a sum
  // has no more roundings in a row than the splits of a plain product have
  constexpr bool TWO = sizeof(T) == 4;
  v4 sum[TWO ? NB : 1];
#pragma unroll
  for (int j = 0; j < (TWO ? NB : 1); ++j) sum[j] = (v4){0, 0, 0, 0};
  // 16-byte pieces 2 gq and 2 gq + 1 of row li of each block (pieces permuted by the row)
  const int pa = li * 128 + (((2 * gq) ^ (li & 7)) << 4), pb = li * 128 + (((2 * gq + 1) ^ (li & 7)) << 4);
  // Blocks in groups; the LDS reads of a group are issued behind the first MFMA
  // of the group before it, those of a slab's first group ahead of the next
  // slab's loads (an MFMA that waits for a read just issued idles the pipe)
  typedef T th __attribute__((ext_vector_type(KS / 2)));
  constexpr int NG = NB < 6 ? 1 : (NB + 2) / 4;
  constexpr int GS = (NB + NG - 1) / NG;  // blocks gr*NB/NG .. of group gr, at most GS
  th blo[2][GS], bhi[2][GS];
  auto read = [&](const char* buf, int gr) ADC2G_INLINE {
#pragma unroll
    for (int j = 0; j < GS; ++j) {
      const int blk = gr * NB / NG + j;
      if (blk < (gr + 1) * NB / NG) {
        blo[gr & 1][j] = *(const th*)(buf + blk * 2048 + pa);
        bhi[gr & 1][j] = *(const th*)(buf + blk * 2048 + pb);
      }
    }
  };
  if (u_begin < u_end) {
    load_x();
    dma(u_begin, s0);
    lds_ready();
    int u = u_begin;
    auto step = [&](const char* cur, char* nxt) ADC2G_INLINE {
      read(cur, 0);
      T a[KS];
      operand(a);
      if (u + 1 < u_end) {
        load_x();
        dma(u + 1, nxt);
      }
#pragma unroll
      for (int gr = 0; gr < NG; ++gr) {
#pragma unroll
        for (int s = 0; s < KS; ++s)
#pragma unroll
          for (int j = 0; j < GS; ++j) {
            if (s == 0 && j == 1) {  // behind the MFMA that waits for this group's reads
              __builtin_amdgcn_sched_barrier(0);
              if (gr + 1 < NG) read(cur, gr + 1);
              __builtin_amdgcn_sched_barrier(0);
            }
            const int blk = gr * NB / NG + j;
            if (blk < (gr + 1) * NB / NG)
              acc[blk] =
                  MT::mma(a[s], s < KS / 2 ? blo[gr & 1][j][s % (KS / 2)] : bhi[gr & 1][j][s % (KS / 2)], acc[blk]);
          }
        __builtin_amdgcn_sched_barrier(0);
      }
      if (TWO && ((u - u_begin) & 7) == 7) {
#pragma unroll
        for (int j = 0; j < (TWO ? NB : 1); ++j) {
          sum[j] += acc[j];
          acc[j] = (v4){0, 0, 0, 0};
        }
      }
      lds_ready();
      ++u;
    };
    while (u < u_end) {
      step(s0, s1);
      if (u < u_end) step(s1, s0);
    }
  }
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    if (TWO) acc[j] += sum[TWO ? j : 0];
    const int cc = n0 + j * 16 + li;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int rr = (grp * nw + wave) * 16 + MT::row(lane, r);
      if (rr < rows && cc < v) part[((int64_t)ks * rows + rr) * v + cc] = acc[j][r];
    }
  }
}

// ---- up: W2 += the CSF combinations of H[(vec,k)][(l,p)] = sum_c x(c,k) V_t[l][c][p].
// One workgroup: the pairs p of one (chunk, type), every l, whole vectors.  The
// accumulators of a wave are 16 rows (vec,k) of all (l, p); (k,l) and (l,k)
// meet in LDS, a few vectors at a time, and W2 -- holding D x2 + the occupied
// term -- is updated in runs of P pairs.
template <class T, int NL>
__global__ void __launch_bounds__(NL <= 16 ? 512 : 256, NL <= 16 ? 2 : 1)
up_kernel(CsfGeo g, int vpb, int ug, const double* __restrict__ X, const double* __restrict__ zeros,
          const T* __restrict__ V, double* __restrict__ W) {
  typedef Mma<T> MT;
  typedef typename MT::v4 v4;
  typedef typename MT::Acc Acc;
  constexpr int PB = 8 / (int)sizeof(T);  // 16-pair blocks per chunk; lane li holds pairs PB*li ..
  constexpr int P = 16 * PB;
  constexpr int KT = CSF_UP_ROWS;         // rows c per K tile
  constexpr int ARR = NL * KT * 128;
  typedef T tv __attribute__((ext_vector_type(PB)));
  __shared__ __attribute__((aligned(1024))) char s0[ARR];
  __shared__ __attribute__((aligned(1024))) char s1[ARR];
  __shared__ __attribute__((aligned(1024))) char s2[ARR];
  __shared__ unsigned char tk[NL * (NL - 1) / 2 + 1], tl[NL * (NL - 1) / 2 + 1];
  const int lane = threadIdx.x & 63, nw = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, gq = lane >> 4;
  const int o = g.o, v = g.v;
  const int w = xcd_tile(blockIdx.x, gridDim.x);
  const int grp = uniform(w % ug), pan = uniform(w / ug);
  const bool diag = pan >= 2 * g.nch;
  const int ch = diag ? pan - 2 * g.nch : pan >> 1;
  const bool five = !diag && (pan & 1);
  const int vec0 = grp * vpb, nvec = min(vpb, g.nv - vec0);
  const int rows = nvec * o;
  const int row = wave * 16 + li;
  const bool live = row < rows;
  const int vec = live ? row / o : 0, k = live ? row - vec * o : 0;
  // the lane's next x1 value (rows past the last vector read zeros)
  const char* xp = (const char*)(live ? X + g.ldx * (vec0 + vec) + k : zeros) + (int64_t)csf_up_first(gq, v) * o * 8;
  const int64_t slab = (int64_t)v * 128;
  const char* src0 =
      (const char*)V + (diag ? (int64_t)2 * g.nch * o + (int64_t)ch * o : (int64_t)ch * 2 * o + (five ? o : 0)) * slab;

  for (int kk = threadIdx.x; kk < o; kk += blockDim.x) {
    int q = (int)po_index(kk, kk + 1, o);
    for (int ll = kk + 1; ll < o; ++ll, ++q) {
      tk[q] = (unsigned char)kk;
      tl[q] = (unsigned char)ll;
    }
  }
  const Rsrc src = lds_source(src0);
  const int lane16 = lane * 16, slab32 = v * 128;
  auto dma = [&](int c0, char* buf) ADC2G_INLINE {
    for (int l = wave; l < o; l += nw) lds_copy(src, l * slab32 + c0 * 128, buf + l * 1024, lane16);
  };
  double xr[2];
  const int64_t xhalf = (int64_t)csf_up_half(v) * o * 8, xstep = (int64_t)o * KT * 8;
  auto load_x = [&]() ADC2G_INLINE {  // (rows c past the last virtual are masked in operand)
    xr[0] = *(const double*)xp;
    xr[1] = *(const double*)(xp + xhalf);
    xp += xstep;
  };
  v4 acc[NL][PB];
#pragma unroll
  for (int l = 0; l < NL; ++l)
#pragma unroll
    for (int j = 0; j < PB; ++j) acc[l][j] = (v4){0, 0, 0, 0};
  // Three buffers, and the one barrier of a tile in the middle of its MFMAs:
  // there tile c0 + KT has landed and every wave is done with tile c0 - KT,
  // whose buffer takes c0 + 2 KT.  The LDS reads of a group of LG columns l are
  // issued behind the first MFMA of the group before it.
  constexpr int LG = NL % 8 == 0 ? 8 : (NL % 6 == 0 ? 6 : (NL % 10 == 0 ? 10 : NL / 2));
  constexpr int NG = NL / LG;
  tv b[2][LG];
  auto read = [&](const char* buf, int x) ADC2G_INLINE {  // x = group of step s, s * NG + group
    const int s = x / NG, g0 = (x % NG) * LG;
    // row c = 4 s + gq, 8 bytes at li * 8 (16-byte pieces permuted by the row)
    const int at = (4 * s + gq) * 128 + ((((li >> 1) ^ (4 * s + gq)) << 4) | ((li & 1) << 3));
#pragma unroll
    for (int l = 0; l < LG; ++l) b[x & 1][l] = *(const tv*)(buf + (g0 + l) * (KT * 128) + at);
  };
  T a[2];
  auto operand = [&](int c0, T (&to)[2]) ADC2G_INLINE {
#pragma unroll
    for (int s = 0; s < 2; ++s) to[s] = (T)xr[s];
    if (c0 + KT > v) {
#pragma unroll
      for (int s = 0; s < 2; ++s) to[s] = c0 + 4 * s + gq < v ? to[s] : (T)0;
    }
  };
  int c0 = 0;
  dma(0, s0);
  load_x();
  operand(0, a);
  if (KT < v) {
    dma(KT, s1);
    load_x();
  }
  lds_ready();
  read(s0, 0);
  auto step = [&](const char* cur, const char* nxt, char* nn) ADC2G_INLINE {
    T an[2];
#pragma unroll
    for (int x = 0; x < 2 * NG; ++x) {
      const int s = x / NG, g0 = (x % NG) * LG;
#pragma unroll
      for (int l = 0; l < LG; ++l) {
        if (l == 1 || LG == 1) {  // behind the MFMA that waits for this group's reads
          __builtin_amdgcn_sched_barrier(0);
          if (x + 1 < 2 * NG)
            read(cur, x + 1);
          else
            read(nxt, 0);
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int j = 0; j < PB; ++j) acc[g0 + l][j] = MT::mma(a[s], b[x & 1][l][j], acc[g0 + l][j]);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (x == NG - 1) {
        lds_ready();
        operand(c0 + KT, an);
        if (c0 + 2 * KT < v) {
          dma(c0 + 2 * KT, nn);
          load_x();
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int s = 0; s < 2; ++s) a[s] = an[s];
    c0 += KT;
  };
  while (c0 < v) {
    step(s0, s1, s2);
    if (c0 < v) step(s1, s2, s0);
    if (c0 < v) step(s2, s0, s1);
  }
  __syncthreads();

  // H of whole vectors through LDS, a third of the rows k in each buffer; for
  // more than 24 orbitals in two halves of the pairs
  constexpr int PH = NL > 24 ? 2 : 1, PP = P / PH;
  const int hk = (o + 2) / 3;
  const int third = hk * o * PP;  // elements of a vector in each buffer
  const int nvp = ARR / (third * (int)sizeof(Acc));
  auto base = [&](int kk) ADC2G_INLINE -> Acc* {
    Acc* e = (Acc*)s0;
    e = kk < hk ? e : (Acc*)s1 - hk * o * PP;
    return kk < 2 * hk ? e : (Acc*)s2 - 2 * hk * o * PP;
  };
  for (int b0 = 0; b0 < nvec; b0 += nvp) {
    const int nb = min(nvp, nvec - b0);
    for (int ph = 0; ph < PH; ++ph) {
      const int p0 = ch * P + ph * PP;
      const int64_t lim = (diag ? (int64_t)v : g.npv) - p0;
      const int np = (int)max((int64_t)0, min((int64_t)PP, lim));
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int rr = wave * 16 + MT::row(lane, r);
        const int vv = rr / o, kk = rr - vv * o;
        if (vv < b0 || vv >= b0 + nb || (PH == 2 && (li >> 3) != ph)) continue;
        Acc* e = base(kk) + kk * o * PP + (vv - b0) * third;
#pragma unroll
        for (int l = 0; l < NL; ++l)
          if (l < NL - 1 || o == NL)  // NL = o, or o + 1 with an unused last block
#pragma unroll
            for (int j = 0; j < PB; ++j) e[l * PP + PB * (li & (16 / PH - 1)) + j] = acc[l][j][r];
      }
      __syncthreads();
      const int p = threadIdx.x & (PP - 1);
      const int y = threadIdx.x / PP, ny = blockDim.x / PP;
      for (int vv = 0; vv < nb; ++vv) {
        double* wv = W + g.ldw * (vec0 + b0 + vv);
        auto at = [&](int kk, int ll, int pp) ADC2G_INLINE {
          return (double)base(kk)[vv * third + (kk * o + ll) * PP + pp];
        };
        double* wq = wv + (diag ? g.off3 : (five ? g.off5 : g.off4)) + p0 + p;
        const int64_t sq = diag ? (int64_t)v : g.npv;
        // t2, or t1: (pair, k) with k fastest, or (k, pair); the first value is
        // loaded ahead of the pairs of t4, t5 or t3
        const int n2 = five ? 0 : np * o;
        auto at2 = [&](int t, int& kk, int& pp) ADC2G_INLINE -> double* {
          if (diag) {
            kk = t / np;
            pp = t - kk * np;
            return wv + g.off1 + (int64_t)kk * v + p0 + pp;
          }
          pp = t / o;
          kk = t - pp * o;
          return wv + g.off2 + (int64_t)p0 * o + t;
        };
        int k2 = 0, p2 = 0;
        double* w2 = n2 > 0 ? at2(min((int)threadIdx.x, n2 - 1), k2, p2) : wv;
        double old2 = *w2;
        if (p < np)
          for (int q0 = y; q0 < g.npo; q0 += 8 * ny) {
            double old[8];  // eight loads of W in flight
#pragma unroll
            for (int e = 0; e < 8; ++e) old[e] = wq[min(q0 + e * ny, g.npo - 1) * sq];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              const int q = q0 + e * ny;
              if (q >= g.npo) break;
              const int kk = tk[q], ll = tl[q];
              const double h1 = at(kk, ll, p), h2 = at(ll, kk, p);
              wq[q * sq] = old[e] + (five ? h1 - h2 : h1 + h2);
            }
          }
        for (int t = threadIdx.x; t < n2; t += blockDim.x) {
          if (t != (int)threadIdx.x) {
            w2 = at2(t, k2, p2);
            old2 = *w2;
          }
          *w2 = old2 - SQ2 * at(k2, k2, p2);
        }
      }
      __syncthreads();
    }
  }
}

// ---- both directions in one pass over the operand, for at most 32 rows
// (vec,k): a few vectors read the operand faster than they use it (1 GB for
// o=16, v=200 in FP64, against 0.1 ms of MFMAs for one vector), and both
// directions read the same one.  One workgroup a CU takes (chunk, type) after
// (chunk, type); its waves take the l of one by turns, each streaming its slabs
// through two LDS slots of its own (no barrier in the slab loop), with the
// down sums of all columns and the H of its l in registers.  The down sums of
// the four waves are added at the end, the H exchanged in LDS after each
// (chunk, type) as in the up kernel.
template <class T, int NB, int NS, int TM>
__global__ void __launch_bounds__(256, 1)
thin_kernel(CsfGeo g, const double* __restrict__ X, const double* __restrict__ T2, const double* __restrict__ zeros,
            const T* __restrict__ V, double* __restrict__ W, typename Mma<T>::Acc* __restrict__ part) {
  typedef Mma<T> MT;
  typedef typename MT::v4 v4;
  typedef typename MT::Acc Acc;
  constexpr int KS = 32 / (int)sizeof(T), P = 4 * KS, PB = 8 / (int)sizeof(T);
  constexpr int SB = (NB + NS - 1) / NS;  // blocks s*NB/NS .. of slab part s, at most SB
  constexpr int NLW = 4;                  // l of a wave: wave, wave + 4, ...
  constexpr int R = 16 * TM;
  static_assert(NS % 2 == 0, "slab parts alternate between two slots");
  typedef T th __attribute__((ext_vector_type(KS / 2)));
  typedef T tv __attribute__((ext_vector_type(PB)));
  __shared__ __attribute__((aligned(1024))) char r0[4][SB * 2048];
  __shared__ __attribute__((aligned(1024))) char r1[4][SB * 2048];
  __shared__ T x1s[NB * 16 * R];
  __shared__ Acc hx[16 * 16 * P];
  __shared__ unsigned char tk[120], tl[120];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, gq = lane >> 4;
  const int o = g.o, v = g.v, rows = g.nv * o;
  const int nb = (v + 15) / 16;
  const int items = 2 * g.nch + g.nchd;
  const int wg = xcd_tile(blockIdx.x, gridDim.x);
  const int it0 = uniform((int)((int64_t)items * wg / gridDim.x)), it1 = uniform((int)((int64_t)items * (wg + 1) / gridDim.x));
  const int64_t slab = (int64_t)v * 128;
  const int lane16 = lane * 16;

  for (int kk = threadIdx.x; kk < o; kk += 256) {
    int q = (int)po_index(kk, kk + 1, o);
    for (int ll = kk + 1; ll < o; ++ll, ++q) {
      tk[q] = (unsigned char)kk;
      tl[q] = (unsigned char)ll;
    }
  }
  for (int t = threadIdx.x; t < NB * 16 * R; t += 256) {
    const int c = t / R, rr = t - c * R;
    const int vv = rr / o, kk = rr - vv * o;
    x1s[t] = (rr < rows && c < v) ? (T)X[g.ldx * vv + (int64_t)c * o + kk] : (T)0;
  }
  int vec[TM], kr[TM];
  bool live[TM];
#pragma unroll
  for (int m = 0; m < TM; ++m) {
    const int row = m * 16 + li;
    live[m] = row < rows;
    vec[m] = live[m] ? row / o : 0;
    kr[m] = live[m] ? row - vec[m] * o : 0;
  }
  __syncthreads();
  const int nl = wave < o ? (o - wave + 3) / 4 : 0;

  // (chunk, type) `it`: is it diagonal, t5, and its first slab
  auto decode = [&](int it, int& diag, int& t, int& ch) ADC2G_INLINE {
    diag = it >= 2 * g.nch ? 1 : 0;
    ch = diag ? it - 2 * g.nch : it >> 1;
    t = diag ? 0 : it & 1;
  };
  auto dma = [&](int it, int il, int s, char* buf) ADC2G_INLINE {
    int diag, t, ch;
    decode(it, diag, t, ch);
    const int64_t u = (diag ? (int64_t)2 * g.nch * o + (int64_t)ch * o : (int64_t)ch * 2 * o + t * o) + wave + 4 * il;
    const Rsrc src = lds_source((const char*)V + u * slab);
    const int b0 = s * NB / NS, b1 = min((s + 1) * NB / NS, nb);
    for (int i = 2 * b0; i < 2 * b1; ++i) lds_copy(src, i * 1024, buf + (i - 2 * b0) * 1024, lane16);
  };
  double xr[TM][KS];
  int left = 0, five = 0, lx = 0;
  auto load_x = [&](int it, int il) ADC2G_INLINE {
    int diag, t, ch;
    decode(it, diag, t, ch);
    const int l = wave + 4 * il;
    left = (diag ? v : (int)g.npv) - ch * P;
    five = t;
    lx = l;
#pragma unroll
    for (int m = 0; m < TM; ++m) {
      const int k = kr[m];
      const double* e = zeros;
      if (live[m]) {
        if (l == k) {
          const double* t2v = T2 + (int64_t)(vec[m] * o + k) * (g.npv + v);
          e = diag ? t2v + g.npv : (t ? zeros : t2v);
        } else {
          const int64_t q = po_index(min(k, l), max(k, l), o);
          e = X + g.ldx * vec[m] + (diag ? g.off3 + q * v : (t ? g.off5 : g.off4) + q * g.npv);
        }
      }
      e += ch * P;
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const int p = gq * KS + s;
        xr[m][s] = e[p < left ? p : 0];
      }
    }
  };
  v4 sacc[TM][NB];
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int j = 0; j < NB; ++j) sacc[m][j] = (v4){0, 0, 0, 0};
  v4 h[NLW][TM][PB];
  const int pa = li * 128 + (((2 * gq) ^ (li & 7)) << 4), pb = li * 128 + (((2 * gq + 1) ^ (li & 7)) << 4);
  const int pu = (((li >> 1) << 4) | ((li & 1) << 3));

  const int npo = g.npo;
  if (nl > 0 && it0 < it1) {
    load_x(it0, 0);
    dma(it0, 0, 0, r0[wave]);
  }
  for (int it = it0; it < it1; ++it) {
    int diag, t, ch;
    decode(it, diag, t, ch);
#pragma unroll
    for (int il = 0; il < NLW; ++il) {
#pragma unroll
      for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int j = 0; j < PB; ++j) h[il][m][j] = (v4){0, 0, 0, 0};
      if (il < nl) {
        T a[TM][KS];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this part (and the rows) have landed
          __builtin_amdgcn_wave_barrier();
          if (s == 0) {
#pragma unroll
            for (int m = 0; m < TM; ++m) {
              const double sg = five && lx < kr[m] ? -1.0 : 1.0;
#pragma unroll
              for (int e = 0; e < KS; ++e) a[m][e] = gq * KS + e < left ? (T)(sg * xr[m][e]) : (T)0;
            }
          }
          char* nxt = (s & 1) ? r0[wave] : r1[wave];
          if (s + 1 < NS) {
            dma(it, il, s + 1, nxt);
          } else {
            const int il2 = il + 1 < nl ? il + 1 : 0, it2 = il + 1 < nl ? it : it + 1;
            if (it2 < it1) {
              load_x(it2, il2);
              dma(it2, il2, 0, nxt);
            }
          }
          const char* cur = (s & 1) ? r1[wave] : r0[wave];
#pragma unroll
          for (int jj = 0; jj < SB; ++jj) {
            const int j = s * NB / NS + jj;
            if (j < (s + 1) * NB / NS && j < nb) {
              const char* blk = cur + jj * 2048;
              const th lo = *(const th*)(blk + pa), hi = *(const th*)(blk + pb);
#pragma unroll
              for (int e = 0; e < KS; ++e)
#pragma unroll
                for (int m = 0; m < TM; ++m)
                  sacc[m][j] = MT::mma(a[m][e], e < KS / 2 ? lo[e % (KS / 2)] : hi[e % (KS / 2)], sacc[m][j]);
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const int c = 4 * e + gq;
                const tv b = *(const tv*)(blk + c * 128 + (pu ^ ((c & 7) << 4)));
#pragma unroll
                for (int m = 0; m < TM; ++m) {
                  const T x = x1s[(j * 16 + c) * R + m * 16 + li];
#pragma unroll
                  for (int q = 0; q < PB; ++q) h[il][m][q] = MT::mma(x, b[q], h[il][m][q]);
                }
              }
            }
          }
        }
      }
    }
    // exchange, one vector at a time: hx[k][l][p]
    const int p0 = ch * P;
    const int np = min(P, (diag ? v : (int)g.npv) - p0);
    for (int vv = 0; vv < g.nv; ++vv) {
      __syncthreads();
#pragma unroll
      for (int m = 0; m < TM; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int rr = m * 16 + MT::row(lane, r);
          const int kk = rr - vv * o;
          if (kk < 0 || kk >= o) continue;
#pragma unroll
          for (int il = 0; il < NLW; ++il)
            if (il < nl)
#pragma unroll
              for (int q = 0; q < PB; ++q) hx[(kk * o + wave + 4 * il) * P + PB * li + q] = h[il][m][q][r];
        }
      __syncthreads();
      double* wv = W + g.ldw * vv;
      const int p = threadIdx.x & (P - 1), y = threadIdx.x / P;
      constexpr int NY = 256 / P;
      if (p < np) {
        double* wq = wv + (diag ? g.off3 : (t ? g.off5 : g.off4)) + p0 + p;
        const int64_t sq = diag ? (int64_t)v : g.npv;
        for (int q0 = y; q0 < npo; q0 += 8 * NY) {
          double old[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) old[e] = wq[min(q0 + e * NY, npo - 1) * sq];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const int q = q0 + e * NY;
            if (q >= npo) break;
            const int kk = tk[q], ll = tl[q];
            const double h1 = (double)hx[(kk * o + ll) * P + p], h2 = (double)hx[(ll * o + kk) * P + p];
            wq[q * sq] = old[e] + (t ? h1 - h2 : h1 + h2);
          }
        }
      }
      if (!t)
        for (int i = threadIdx.x; i < np * o; i += 256) {
          const int kk = diag ? i / np : i % o, pp = diag ? i % np : i / o;
          double* w2 = diag ? wv + g.off1 + (int64_t)kk * v + p0 + pp : wv + g.off2 + (int64_t)p0 * o + i;
          *w2 -= SQ2 * (double)hx[(kk * o + kk) * P + pp];
        }
    }
  }
  // down sums of the four waves, 16 rows at a time through the first slot
  static_assert(NB * 16 * 16 * (int)sizeof(Acc) <= (int)sizeof(hx), "the sums fit the exchange buffer");
#pragma unroll
  for (int m = 0; m < TM; ++m) {
    for (int w = 0; w < 4; ++w) {
      __syncthreads();
      if (wave == w) {
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            Acc* e = hx + MT::row(lane, r) * (NB * 16) + j * 16 + li;
            *e = (w == 0 ? (Acc)0 : *e) + sacc[m][j][r];
          }
      }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 16 * v; i += 256) {
      const int rr = i / v, c = i - rr * v;
      if (m * 16 + rr < rows) part[((int64_t)wg * rows + m * 16 + rr) * v + c] = hx[rr * (NB * 16) + c];
    }
  }
}

template <class T, int NB>
void down_launch(const CsfGeo& g, const CsfPlan& p, const double* X, const double* T2, const double* zeros, const T* V,
                 typename Mma<T>::Acc* part, hipStream_t st) {
  if constexpr (NB > 1) {
    if (p.dnb < NB) {
      down_launch<T, NB - 1>(g, p, X, T2, zeros, V, part, st);
      return;
    }
  }
  hipLaunchKernelGGL((down_kernel<T, NB>), dim3((unsigned)(p.ds * p.dg * p.dns)), dim3(64 * p.dw),
                     (size_t)2 * g.o * p.dw * 16 * sizeof(uint64_t), st, g, p.ds, p.dg, p.dns, X, T2, zeros, V, part);
  HIP_CHECK(hipGetLastError());
}

template <class T, int NL>
void up_launch(const CsfGeo& g, const CsfPlan& p, const double* X, const double* zeros, const T* V, double* W,
               hipStream_t st) {
  if constexpr (NL > 2) {
    if (g.o <= NL - 2) {
      up_launch<T, NL - 2>(g, p, X, zeros, V, W, st);
      return;
    }
  }
  hipLaunchKernelGGL((up_kernel<T, NL>), dim3((unsigned)((2 * g.nch + g.nchd) * p.ug)), dim3(64 * p.uw), 0, st, g,
                     p.uvpb, p.ug, X, zeros, V, W);
  HIP_CHECK(hipGetLastError());
}

template <class T, int TM>
void thin_launch(const CsfGeo& g, const CsfPlan& p, const double* X, const double* T2, const double* zeros, const T* V,
                 double* W, typename Mma<T>::Acc* part, hipStream_t st) {
  const dim3 grid((unsigned)p.thin), blk(256);
  const int nb = (g.v + 15) / 16;
  // thin plans start at v = 128 (eight blocks): two vectors, o = 16, FP64 there
  // 237 us, with the parts of 13 blocks 255
  if (nb <= 8)
    hipLaunchKernelGGL((thin_kernel<T, 8, 2, TM>), grid, blk, 0, st, g, X, T2, zeros, V, W, part);
  else
    hipLaunchKernelGGL((thin_kernel<T, 13, 4, TM>), grid, blk, 0, st, g, X, T2, zeros, V, W, part);
  HIP_CHECK(hipGetLastError());
}

}  // namespace csfv

template <class T>
void launch_csf_down(const CsfGeo& g, const CsfPlan& p, const double* X, const double* T2, const double* zeros,
                     const T* V, typename Mma<T>::Acc* part, hipStream_t st) {
  csfv::down_launch<T, 13>(g, p, X, T2, zeros, V, part, st);
}

template <class T>
void launch_csf_up(const CsfGeo& g, const CsfPlan& p, const double* X, const double* zeros, const T* V, double* W,
                   hipStream_t st) {
  csfv::up_launch<T, CSF_OMAX>(g, p, X, zeros, V, W, st);
}

template <class T>
void launch_csf_thin(const CsfGeo& g, const CsfPlan& p, const double* X, const double* T2, const double* zeros,
                     const T* V, double* W, typename Mma<T>::Acc* part, hipStream_t st) {
  if (g.nv * g.o <= 16)
    csfv::thin_launch<T, 1>(g, p, X, T2, zeros, V, W, part, st);
  else
    csfv::thin_launch<T, 2>(g, p, X, T2, zeros, V, W, part, st);
}

}  // namespace adc2g
