// Device code of the mixed-radix passes (ddx_mixed.h).
#pragma once

#include "ddx_mixed.h"

namespace ddx {

// p[i] from a base that is uniform over the wavefront: the byte offset fits 32
// bits (checked on the host), so the load takes the base from scalar
// registers and one vector register of offset (OFF unsigned long: arrays of
// 4 GB and more).
template <typename T, typename OFF>
__device__ __forceinline__ cpx<T> ld_off(const cpx<T>* __restrict__ p, OFF i) {
  return *reinterpret_cast<const cpx<T>*>(reinterpret_cast<const char*>(p) + (size_t)(i * (OFF)sizeof(cpx<T>)));
}
template <typename T, typename OFF>
__device__ __forceinline__ cpx<T>* at_off(cpx<T>* p, OFF i) {
  return reinterpret_cast<cpx<T>*>(reinterpret_cast<char*>(p) + (size_t)(i * (OFF)sizeof(cpx<T>)));
}

// --- composite DFTs -----------------------------------------------------------

// n = A B with A, B coprime: the prime-factor map needs no twiddles.  Input
// index (B n1 + A n2) mod n; output k with k = k1 mod A, k = k2 mod B.
template <int D, int A, int B, typename T>
__device__ __forceinline__ void dft_pfa(cpx<T>* v) {
  constexpr int N = A * B;
  cpx<T> t[B][A];
#pragma unroll
  for (int n2 = 0; n2 < B; ++n2) {
#pragma unroll
    for (int n1 = 0; n1 < A; ++n1) t[n2][n1] = v[(B * n1 + A * n2) % N];
    dft<D, A>(t[n2]);
  }
#pragma unroll
  for (int k1 = 0; k1 < A; ++k1) {
    cpx<T> u[B];
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) u[n2] = t[n2][k1];
    dft<D, B>(u);
#pragma unroll
    for (int k2 = 0; k2 < B; ++k2) {
      int k = k1;
#pragma unroll
      for (int q = 0; q < B; ++q)
        if (k % B != k2) k += A;
      v[k] = u[k2];
    }
  }
}

// 9 = 3 x 3 with the twiddles W9^1, W9^2, W9^4
template <int D, typename T>
__device__ __forceinline__ void dft9(cpx<T>* v) {
  const T c1 = T(0.76604444311897803520), s1 = T(0.64278760968653932632);
  const T c2 = T(0.17364817766693034885), s2 = T(0.98480775301220805937);
  const T c4 = T(-0.93969262078590838405), s4 = T(0.34202014332566873304);
  cpx<T> t[3][3];
#pragma unroll
  for (int n2 = 0; n2 < 3; ++n2) {
#pragma unroll
    for (int n1 = 0; n1 < 3; ++n1) t[n2][n1] = v[3 * n1 + n2];
    dft3<D>(t[n2]);
  }
  t[1][1] = t[1][1] * mk(c1, T(D) * s1);
  t[1][2] = t[1][2] * mk(c2, T(D) * s2);
  t[2][1] = t[2][1] * mk(c2, T(D) * s2);
  t[2][2] = t[2][2] * mk(c4, T(D) * s4);
#pragma unroll
  for (int k1 = 0; k1 < 3; ++k1) {
    cpx<T> u[3] = {t[0][k1], t[1][k1], t[2][k1]};
    dft3<D>(u);
#pragma unroll
    for (int k2 = 0; k2 < 3; ++k2) v[k1 + 3 * k2] = u[k2];
  }
}

template <int D, int R, typename T>
__device__ __forceinline__ void mdft(cpx<T>* v) {
  if constexpr (R == 6) dft_pfa<D, 2, 3>(v);
  else if constexpr (R == 9) dft9<D>(v);
  else if constexpr (R == 10) dft_pfa<D, 2, 5>(v);
  else if constexpr (R == 12) dft_pfa<D, 4, 3>(v);
  else if constexpr (R == 15) dft_pfa<D, 3, 5>(v);
  else dft<D, R>(v);
}

// Leg r (>= 1) multiplied by W^(r e), each from its own table entry: powers
// formed from one entry by a product tree made the 192^3 x rows 6 % faster
// (the table reads share the L1 with the data) at 1.4 to 1.7 times the FP64
// rounding error of a step.
template <int D, int R, typename T>
__device__ __forceinline__ void mix_legs(cpx<T>* v, const cpx<T>* __restrict__ tw, int e) {
#pragma unroll
  for (int r = 1; r < R; ++r) {
    const cpx<T> w = ld_off(tw, (unsigned)(r * e));
    v[r] = v[r] * mk(w.x, D < 0 ? w.y : -w.y);
  }
}

// body<R>() for the radix r (uniform)
#define MIX_RADIX(r, CALL)      \
  switch (r) {                  \
    case 1: CALL(1); break;     \
    case 2: CALL(2); break;     \
    case 3: CALL(3); break;     \
    case 4: CALL(4); break;     \
    case 5: CALL(5); break;     \
    case 6: CALL(6); break;     \
    case 8: CALL(8); break;     \
    case 9: CALL(9); break;     \
    case 10: CALL(10); break;   \
    case 12: CALL(12); break;   \
    case 15: CALL(15); break;   \
    default: CALL(16); break;   \
  }

#define MIX_RADIX12(r, CALL)    \
  switch (r) {                  \
    case 1: CALL(1); break;     \
    case 2: CALL(2); break;     \
    case 3: CALL(3); break;     \
    case 4: CALL(4); break;     \
    case 5: CALL(5); break;     \
    case 6: CALL(6); break;     \
    case 8: CALL(8); break;     \
    case 9: CALL(9); break;     \
    case 10: CALL(10); break;   \
    default: CALL(12); break;   \
  }

#define MIX_RADIX10(r, CALL)    \
  switch (r) {                  \
    case 1: CALL(1); break;     \
    case 2: CALL(2); break;     \
    case 3: CALL(3); break;     \
    case 4: CALL(4); break;     \
    case 5: CALL(5); break;     \
    case 6: CALL(6); break;     \
    case 8: CALL(8); break;     \
    case 9: CALL(9); break;     \
    default: CALL(10); break;   \
  }

// --- column pass ----------------------------------------------------------------

// The sources of a first pass, read from the arguments once: up to two
// recipe terms coef * (i k)^[kind > 0] * src, k along the column axis
// (kind 1), the slab axis (2) or the row axis (3).
template <typename T>
struct MixSrc {
  const cpx<T>* p[2];
  int kind[2];
  T coef[2];
  double ks;             // the slab's wavenumber
  const double* k_col;
  double kr_inv, kr_kny;
  int in_c, in_rows, ncols;
  long in_rs;
};

template <typename T, bool SPECTRAL>
__device__ __forceinline__ MixSrc<T> mixc_src(const ColArgs<T>& a, int f, long slab) {
  MixSrc<T> s;
  s.in_c = a.in_c;
  s.in_rows = a.in_rows;
  s.ncols = a.ncols;
  s.in_rs = a.in_rs;
  if (SPECTRAL) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const Term tm = a.rec[f].t[t];
      s.p[t] = a.src[tm.src] + slab * a.in_ss;
      s.kind[t] = tm.dim < 0 ? 0 : (tm.dim == 0 ? 1 : (tm.dim == a.row_dim ? 3 : 2));
      s.coef[t] = T(tm.coef);
    }
    const double* ks = a.k_slab;
    s.ks = ks ? ks[slab] : 0.0;
    s.k_col = a.k_col;
    s.kr_inv = a.kr_inv;
    s.kr_kny = a.kr_kny;
  } else {
    s.p[0] = a.in[f] + slab * a.in_ss;
  }
  return s;
}

// First pass: butterfly j of column c reads rows j + r M_0 from global memory
// (rows the 2/3 rule leaves out are zero; NT > 0 forms the recipe's NT
// terms), every load unconditional from a clamped address.
template <typename T, typename OFF, int D, int NT, int R>
__device__ __forceinline__ void mixc_first(const MixSrc<T>& a, const MixPlan& mp, const cpx<T>* __restrict__ tw,
                                           cpx<T>* lds, int c0) {
  constexpr int NTA = NT > 0 ? NT : 1;
  const int W = mp.W, n = mp.n, J = mp.M[0];
  const int total = J << mp.wshift;
  for (int idx = threadIdx.x; idx < total; idx += blockDim.x) {
    const int c = idx & (W - 1), j = idx >> mp.wshift;
    const int col = c0 + c;
    const int colc = col < a.ncols ? col : a.ncols - 1;
    double kc = 0.0;
    if constexpr (NT > 0) kc = a.k_col[colc];
    cpx<T> ld[NTA][R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int m = j + r * J;
      int row = m;
      if (a.in_c >= 0) row = m <= a.in_c ? m : (m >= n - a.in_c ? m - (n - a.in_rows) : 0);
      const OFF off = (OFF)row * (OFF)a.in_rs + (OFF)colc;
#pragma unroll
      for (int t = 0; t < NTA; ++t) ld[t][r] = ld_off(a.p[t], off);
    }
    cpx<T> v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int m = j + r * J;
      const bool ok = a.in_c < 0 || m <= a.in_c || m >= n - a.in_c;
      cpx<T> x;
      if constexpr (NT > 0) {
        x = mk(T(0), T(0));
        // k of the row from its index, as the table has it
        const double kr = ((double)(m <= a.in_c ? m : m - n) * a.kr_inv) * 2.0 * a.kr_kny;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const double kk = a.kind[t] == 3 ? kr : (a.kind[t] == 2 ? a.ks : kc);
          const cpx<T> sv = a.kind[t] ? mul_is(ld[t][r], T(kk)) : ld[t][r];
          x = x + scale(sv, a.coef[t]);
        }
      } else {
        x = ld[0][r];
      }
      v[r] = ok ? x : mk(T(0), T(0));
    }
    mdft<D, R>(v);
    mix_legs<D, R>(v, tw, j);
#pragma unroll
    for (int r = 0; r < R; ++r) lds[((j + r * J) << mp.wshift) + c] = v[r];
  }
}

template <typename T, int D, int R>
__device__ __forceinline__ void mixc_mid(const MixPlan& mp, int p, const cpx<T>* __restrict__ tw, cpx<T>* lds) {
  const int W = mp.W, M = mp.M[p];
  const int total = mix_div(mp.n, mp.dR[p]) << mp.wshift;
  for (int idx = threadIdx.x; idx < total; idx += blockDim.x) {
    const int c = idx & (W - 1), i = idx >> mp.wshift;
    const int q = mix_div(i, mp.dM[p]), j = i - q * M;
    cpx<T>* b = lds + ((q * R * M + j) << mp.wshift) + c;
    cpx<T> v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = b[(r * M) << mp.wshift];
    mdft<D, R>(v);
    mix_legs<D, R>(v, tw, mp.L[p] * j);
#pragma unroll
    for (int r = 0; r < R; ++r) b[(r * M) << mp.wshift] = v[r];
  }
}

// Last pass: leg r of butterfly i is frequency rev(i) + r L, stored where
// the output layout keeps it.
template <typename T, typename OFF, int D, int R>
__device__ __forceinline__ void mixc_last(const ColArgs<T>& a, const MixPlan& mp, const cpx<T>* lds, int f,
                                          long slab, int c0) {
  const int W = mp.W, n = mp.n, P = mp.np, LL = mp.L[P - 1];
  const int total = mix_div(n, mp.dR[P - 1]) << mp.wshift;
  cpx<T>* __restrict__ out = a.out[f] + slab * a.out_ss;
  for (int idx = threadIdx.x; idx < total; idx += blockDim.x) {
    const int c = idx & (W - 1), i = idx >> mp.wshift;
    const int col = c0 + c;
    const cpx<T>* b = lds + ((i * R) << mp.wshift) + c;
    cpx<T> v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = b[r << mp.wshift];
    mdft<D, R>(v);
    int k = 0;
    for (int p = P - 2, q = i; p >= 0; --p) {
      const int t = mix_div(q, mp.dR[p]);
      k += (q - t * mp.R[p]) * mp.L[p];
      q = t;
    }
    if (col >= a.ncols) continue;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int m = k + r * LL;
      int row = m;
      if (a.out_c >= 0) row = m <= a.out_c ? m : (m >= n - a.out_c ? m - (n - a.out_rows) : -1);
      if (row >= 0) st_nt(at_off(out, (OFF)row * (OFF)a.out_rs + (OFF)col), scale(v[r], a.scale), a.nt);
    }
  }
}

// Columns of one tile: entry (m, c) at m W + c, so a wavefront's accesses are
// runs of W consecutive entries whatever the strides (no bank conflicts).
// 192^3 FP64: spectral passes 100 -> 57 us and plain forward passes 51 -> 33
// us against the two-buffer form (3.7 and 4.8 TB/s of their bytes).
template <typename T, typename OFF, int D, bool SPECTRAL>
__global__ void __launch_bounds__(512) mix_col_kernel(const ColArgs<T> a, const MixPlan mp) {
  extern __shared__ __align__(16) unsigned char mix_smem[];
  cpx<T>* lds = reinterpret_cast<cpx<T>*>(mix_smem);
  int f, tile;
  long slab;
  if (!col_unit(a, f, tile, slab)) return;
  const int c0 = tile * mp.W;
  const cpx<T>* __restrict__ tw = a.tw;
  const MixSrc<T> src = mixc_src<T, SPECTRAL>(a, f, slab);
  if constexpr (SPECTRAL) {
    if (a.rec[f].nterm >= 2) {
#define MIX_CALL(R) mixc_first<T, OFF, D, 2, R>(src, mp, tw, lds, c0)
      MIX_RADIX12(mp.R[0], MIX_CALL)
#undef MIX_CALL
    } else {
#define MIX_CALL(R) mixc_first<T, OFF, D, 1, R>(src, mp, tw, lds, c0)
      MIX_RADIX12(mp.R[0], MIX_CALL)
#undef MIX_CALL
    }
  } else {
#define MIX_CALL(R) mixc_first<T, OFF, D, 0, R>(src, mp, tw, lds, c0)
    MIX_RADIX12(mp.R[0], MIX_CALL)
#undef MIX_CALL
  }
  __syncthreads();
  for (int p = 1; p < mp.np - 1; ++p) {
#define MIX_CALL(R) mixc_mid<T, D, R>(mp, p, tw, lds)
    MIX_RADIX(mp.R[p], MIX_CALL)
#undef MIX_CALL
    __syncthreads();
  }
#define MIX_CALL(R) mixc_last<T, OFF, D, R>(a, mp, lds, f, slab, c0)
  MIX_RADIX(mp.R[mp.np - 1], MIX_CALL)
#undef MIX_CALL
}

// --- x rows -----------------------------------------------------------------------

// Sequences of a workgroup: row q / NS of the block, sequence q % NS of the
// row.  First c2r pass: butterfly j of sequence q from the half spectra of
// its two real rows at in + oa and in + ob (addresses clamped, unused values
// zeroed, the k = 0 entry taken as real).  Legs that the 2/3 rule empties for
// every butterfly (two or three of 8 to 10) are not read at all: the
// branches, uniform, cost less than the loads and selects (3 fields of
// 160x144x180, FP64 c2r: 45 -> 40 us; 192^3 hydro x rows 150 -> 146 us).  In
// the column passes they cost more (57 -> 62 us): their loads stay whole.
template <typename T, int R, typename SRC>
__device__ __forceinline__ void mixr_first(const MixRow& mr, const cpx<T>* __restrict__ tw, cpx<T>* buf,
                                           int nq, int cx, const cpx<T>* __restrict__ in, SRC src) {
  const int n = mr.n;
  const int total = nq * mr.J;
  for (int idx = threadIdx.x; idx < total; idx += blockDim.x) {
    const int q = mix_div(idx, mr.dJ), jj = idx - q * mr.J;
    const int n2 = mix_div(jj, mr.dR1), n1 = jj - n2 * mr.R1;
    const int j = n1 * mr.RL + n2;
    unsigned oa, ob;
    bool hasb;
    src(q, oa, ob, hasb);
    cpx<T> la[R], lb[R], v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      la[r] = lb[r] = mk(T(0), T(0));
      if (r * mr.J > cx && (r + 1) * mr.J <= n - cx) continue;   // no entry of this leg is kept
      const int m = j + r * mr.J;
      int k = m < n - m ? m : n - m;
      k = k < cx ? k : cx;
      la[r] = ld_off(in, oa + (unsigned)k);
      lb[r] = ld_off(in, ob + (unsigned)k);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int m = j + r * mr.J;
      const bool keep = m <= cx || m >= n - cx;
      if (r == 0 && m == 0) la[0].y = lb[0].y = T(0);
      // the sign of the mirrored half's imaginary parts
      const T sg = m > cx ? T(-1) : T(1);
      const T ay = la[r].y * sg;
      const T bx = hasb ? lb[r].x : T(0);
      const T by = hasb ? lb[r].y * sg : T(0);
      v[r] = keep ? mk(la[r].x - by, ay + bx) : mk(T(0), T(0));
    }
    mdft<1, R>(v);
    mix_legs<1, R>(v, tw, j);
    cpx<T>* b = buf + q * mr.SS + n2 * mr.S2 + n1 * mr.S1;
#pragma unroll
    for (int r = 0; r < R; ++r) b[r] = v[r];
  }
}

// Middle pass over digit 1: D > 0 multiplies the legs after the DFT (c2r),
// D < 0 before it (r2c)
template <typename T, int D, int R>
__device__ __forceinline__ void mixr_mid(const MixRow& mr, const cpx<T>* __restrict__ tw, cpx<T>* buf, int nq,
                                         int nper, int stride) {
  const int total = nq * mr.TM;
  for (int idx = threadIdx.x; idx < total; idx += blockDim.x) {
    const int q = mix_div(idx, mr.dTM), t = idx - q * mr.TM;
    const int n2 = mix_div(t, mr.dR0), k0 = t - n2 * mr.R0;
    const int s = q / nper * stride + q % nper;
    cpx<T>* b = buf + s * mr.SS + n2 * mr.S2 + k0;
    cpx<T> v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = b[r * mr.S1];
    if (D < 0) mix_legs<D, R>(v, tw, mr.R0 * n2);
    mdft<D, R>(v);
    if (D > 0) mix_legs<D, R>(v, tw, mr.R0 * n2);
#pragma unroll
    for (int r = 0; r < R; ++r) b[r * mr.S1] = v[r];
  }
}

// Last r2c pass over digit 0, in place: entry (n0, n1, n2) is then frequency
// n0 J + n1 RL + n2
template <typename T, int R>
__device__ __forceinline__ void mixr_end(const MixRow& mr, const cpx<T>* __restrict__ tw, cpx<T>* buf, int nq,
                                         int nper, int stride) {
  const int total = nq * mr.J;
  for (int idx = threadIdx.x; idx < total; idx += blockDim.x) {
    const int q = mix_div(idx, mr.dJ), jj = idx - q * mr.J;
    const int n2 = mix_div(jj, mr.dR1), n1 = jj - n2 * mr.R1;
    const int s = q / nper * stride + q % nper;
    cpx<T>* b = buf + s * mr.SS + n2 * mr.S2 + n1 * mr.S1;
    cpx<T> v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = b[r];
    mix_legs<-1, R>(v, tw, n1 * mr.RL + n2);
    mdft<-1, R>(v);
#pragma unroll
    for (int r = 0; r < R; ++r) b[r] = v[r];
  }
}

__device__ __forceinline__ int mixr_entry(const MixRow& mr, int k) {
  const int n0 = mix_div(k, mr.dJ), j = k - n0 * mr.J;
  const int n1 = mix_div(j, mr.dRL), n2 = j - n1 * mr.RL;
  return n2 * mr.S2 + n1 * mr.S1 + n0;
}

// Half spectra of the two real sequences from Z: A = (Z_k + conj Z_{n-k}) / 2,
// B = (Z_k - conj Z_{n-k}) / 2i
template <typename T>
__device__ __forceinline__ void mixr_unpair(const MixRow& mr, const cpx<T>* b, int k, int kx, cpx<T>& A, cpx<T>& B) {
  A = B = mk(T(0), T(0));
  if (k < kx) {
    const cpx<T> zk = b[mixr_entry(mr, k)];
    const cpx<T> zm = conj(b[mixr_entry(mr, k ? mr.n - k : 0)]);
    const cpx<T> s = zk + zm, d = zk - zm;
    A = mk(T(0.5) * s.x, T(0.5) * s.y);
    B = mk(T(0.5) * d.y, T(-0.5) * d.x);
  }
}

template <int PH, int ND> struct MixIO;
template <> struct MixIO<PH_HYDRO, 3> { static constexpr int NIN = 6, NOUT = 3; };
template <> struct MixIO<PH_HYDRO, 2> { static constexpr int NIN = 3, NOUT = 2; };
template <> struct MixIO<PH_BOUSS, 3> { static constexpr int NIN = 10, NOUT = 4; };
template <> struct MixIO<PH_BOUSS, 2> { static constexpr int NIN = 6, NOUT = 3; };
template <> struct MixIO<PH_MHD, 3>   { static constexpr int NIN = 12, NOUT = 6; };
template <> struct MixIO<PH_MHD, 2>   { static constexpr int NIN = 6, NOUT = 3; };

// x rows of the right-hand side: c2r of the field pairs (each pass over all
// pairs of the block's rows), then one thread per last-pass butterfly takes
// every field's x values of its RL positions, forms the products and starts
// the r2c in registers, so x-space data never goes through LDS.
//
// 192^3 FP64 hydro (6 fields in, 3 out, 340 MB): 138 to 146 us on different
// cards against 398 us of the general row kernel, 2.3 to 2.5 TB/s.  VALU issue is busy 55 % of the time (71 k
// lane-instructions per row, a third of them index arithmetic), wavefronts
// wait 55 % of theirs, in phases that six barriers keep apart, so wavefronts
// per SIMD set the time (one card: 3, at 156 registers, 173 us, 4 152 us, 5
// 143 us).  The bounds on the registers below
// are the largest counts without spills that matter (RL 5 and 6 of the 10-
// and 12-field rows spill at three wavefronts; the 2D hydro row keeps five
// with 8 bytes spilled).
template <typename T, int PH, int ND, int RL>
__global__ void __launch_bounds__(256, (ND == 3 && PH != PH_HYDRO && sizeof(T) == 8)
                                                 ? (RL == 4 ? 3 : 2)
                                                 : (sizeof(T) == 8 && RL == 4 ? 5 : 4))
mix_row_phys(const RowArgs<T> a, const MixRow mr, long nrows) {
  constexpr int NIN = MixIO<PH, ND>::NIN, NOUT = MixIO<PH, ND>::NOUT;
  constexpr int NSI = (NIN + 1) / 2, NSO = (NOUT + 1) / 2;
  extern __shared__ __align__(16) unsigned char mix_smem[];
  cpx<T>* buf = reinterpret_cast<cpx<T>*>(mix_smem);
  const cpx<T>* __restrict__ tw = a.tw;
  const long r0 = (long)blockIdx.x * mr.rows;
  const int cx = a.kx - 1;
  const cpx<T>* __restrict__ in0 = a.in[0];
  auto src = [&](int q, unsigned& oa, unsigned& ob, bool& hasb) {
    const int s = q % NSI;
    long row = r0 + q / NSI;
    row = row < nrows ? row : nrows - 1;
    hasb = NIN % 2 == 0 || 2 * s + 1 < NIN;
    oa = (unsigned)(2 * s) * (unsigned)mr.in_fs + (unsigned)row * (unsigned)a.kxp;
    ob = hasb ? oa + (unsigned)mr.in_fs : oa;
  };
#define MIX_CALL(R) mixr_first<T, R>(mr, tw, buf, mr.rows * NSI, cx, in0, src)
  MIX_RADIX10(mr.R0, MIX_CALL)
#undef MIX_CALL
  __syncthreads();
  if (mr.R1 > 1) {
#define MIX_CALL(R) mixr_mid<T, 1, R>(mr, tw, buf, mr.rows * NSI, NSI, NSI)
    MIX_RADIX10(mr.R1, MIX_CALL)
#undef MIX_CALL
    __syncthreads();
  }
  for (int idx = threadIdx.x; idx < mr.rows * mr.T3; idx += blockDim.x) {
    const int rl = mix_div(idx, mr.dT3), t = idx - rl * mr.T3;
    const int k1 = mix_div(t, mr.dR0), k0 = t - k1 * mr.R0;
    cpx<T>* b = buf + rl * NSI * mr.SS + k1 * mr.S1 + k0;
    T q[2 * NSI][RL], o[2 * NSO][RL];
#pragma unroll
    for (int s = 0; s < NSI; ++s) {
      cpx<T> v[RL];
#pragma unroll
      for (int r = 0; r < RL; ++r) v[r] = b[s * mr.SS + r * mr.S2];
      mdft<1, RL>(v);
#pragma unroll
      for (int r = 0; r < RL; ++r) {
        q[2 * s][r] = v[r].x;
        q[2 * s + 1][r] = v[r].y;
      }
    }
#pragma unroll
    for (int r = 0; r < RL; ++r) {
      T qi[12], oi[6];
#pragma unroll
      for (int f = 0; f < 12; ++f) qi[f] = f < NIN ? q[f < 2 * NSI ? f : 0][r] : T(0);
#pragma unroll
      for (int f = 0; f < 6; ++f) oi[f] = T(0);
      row_physics<T>(PH, ND, a.fpr_inv, qi, oi);
#pragma unroll
      for (int f = 0; f < 2 * NSO; ++f) o[f][r] = f < NOUT ? oi[f] : T(0);
    }
    long row = r0 + rl;
    row = row < nrows ? row : nrows - 1;
#pragma unroll
    for (int f = 0; f < NOUT; ++f)
      if (a.xadd[f]) {
#pragma unroll
        for (int r = 0; r < RL; ++r) o[f][r] += a.xadd[f][row * mr.n + t + r * mr.T3];
      }
#pragma unroll
    for (int p = 0; p < NSO; ++p) {
      cpx<T> v[RL];
#pragma unroll
      for (int r = 0; r < RL; ++r) v[r] = mk(o[2 * p][r], o[2 * p + 1][r]);
      mdft<-1, RL>(v);
#pragma unroll
      for (int r = 0; r < RL; ++r) b[p * mr.SS + r * mr.S2] = v[r];
    }
  }
  __syncthreads();
  if (mr.R1 > 1) {
#define MIX_CALL(R) mixr_mid<T, -1, R>(mr, tw, buf, mr.rows * NSO, NSO, NSI)
    MIX_RADIX10(mr.R1, MIX_CALL)
#undef MIX_CALL
    __syncthreads();
  }
#define MIX_CALL(R) mixr_end<T, R>(mr, tw, buf, mr.rows * NSO, NSO, NSI)
  MIX_RADIX10(mr.R0, MIX_CALL)
#undef MIX_CALL
  __syncthreads();
  cpx<T>* __restrict__ out0 = a.out[0];
  for (int idx = threadIdx.x; idx < mr.rows * NSO * a.kxp; idx += blockDim.x) {
    const int q = idx / a.kxp, k = idx - q * a.kxp;
    const int rl = q / NSO, p = q - rl * NSO;
    const long row = r0 + rl;
    if (row >= nrows) continue;
    cpx<T> A, B;
    mixr_unpair(mr, buf + (rl * NSI + p) * mr.SS, k, a.kx, A, B);
    const unsigned o = (unsigned)(2 * p) * (unsigned)mr.out_fs + (unsigned)row * (unsigned)a.kxp + (unsigned)k;
    st_nt(at_off(out0, o), A, a.nt);
    if (NOUT % 2 == 0 || 2 * p + 1 < NOUT) st_nt(at_off(out0, o + (unsigned)mr.out_fs), B, a.nt);
  }
}

// Plain x-row transforms of one field (blockIdx.y): sequences are row pairs
// (row_pair; GRP: within groups, apart because the division it takes costs
// 2 % of the 3 x 160x144x180 c2r where it is not needed).

template <typename T, int RL, bool GRP>
__global__ void __launch_bounds__(256, 4) mix_row_c2r(const RowArgs<T> a, const MixRow mr, long nrows, int group) {
  extern __shared__ __align__(16) unsigned char mix_smem[];
  cpx<T>* buf = reinterpret_cast<cpx<T>*>(mix_smem);
  const cpx<T>* __restrict__ tw = a.tw;
  const long p0 = (long)blockIdx.x * mr.rows;   // row pairs
  const int f = blockIdx.y;
  const cpx<T>* __restrict__ in = a.in[f];
  auto src = [&](int q, unsigned& oa, unsigned& ob, bool& hasb) {
    long row;
    bool live;
    row_pair(p0 + q, nrows, GRP ? group : 0, row, live, hasb);
    oa = (unsigned)(live ? row : nrows - 1) * (unsigned)a.kxp;
    ob = hasb ? oa + (unsigned)a.kxp : oa;
  };
#define MIX_CALL(R) mixr_first<T, R>(mr, tw, buf, mr.rows, a.kx - 1, in, src)
  MIX_RADIX10(mr.R0, MIX_CALL)
#undef MIX_CALL
  __syncthreads();
  if (mr.R1 > 1) {
#define MIX_CALL(R) mixr_mid<T, 1, R>(mr, tw, buf, mr.rows, 1, 1)
    MIX_RADIX10(mr.R1, MIX_CALL)
#undef MIX_CALL
    __syncthreads();
  }
  T* __restrict__ x = a.xout[f];
  for (int idx = threadIdx.x; idx < mr.rows * mr.T3; idx += blockDim.x) {
    const int rl = mix_div(idx, mr.dT3), t = idx - rl * mr.T3;
    const int k1 = mix_div(t, mr.dR0), k0 = t - k1 * mr.R0;
    const cpx<T>* b = buf + rl * mr.SS + k1 * mr.S1 + k0;
    cpx<T> v[RL];
#pragma unroll
    for (int r = 0; r < RL; ++r) v[r] = b[r * mr.S2];
    mdft<1, RL>(v);
    long row;
    bool live, two;
    row_pair(p0 + rl, nrows, GRP ? group : 0, row, live, two);
    if (!live) continue;
    T* xa = x + row * mr.n + t;
#pragma unroll
    for (int r = 0; r < RL; ++r) {
      xa[r * mr.T3] = v[r].x;
      if (two) xa[mr.n + r * mr.T3] = v[r].y;
    }
  }
}

template <typename T, int RL, bool GRP>
__global__ void __launch_bounds__(256) mix_row_r2c(const RowArgs<T> a, const MixRow mr, long nrows, int group) {
  extern __shared__ __align__(16) unsigned char mix_smem[];
  cpx<T>* buf = reinterpret_cast<cpx<T>*>(mix_smem);
  const cpx<T>* __restrict__ tw = a.tw;
  const long p0 = (long)blockIdx.x * mr.rows;
  const int f = blockIdx.y;
  const T* __restrict__ x = a.xin[f];
  for (int idx = threadIdx.x; idx < mr.rows * mr.T3; idx += blockDim.x) {
    const int rl = mix_div(idx, mr.dT3), t = idx - rl * mr.T3;
    const int k1 = mix_div(t, mr.dR0), k0 = t - k1 * mr.R0;
    long row;
    bool live, two;
    row_pair(p0 + rl, nrows, GRP ? group : 0, row, live, two);
    const T* xa = x + (live ? row : nrows - 1) * mr.n + t;
    const T* xb = x + (two ? row + 1 : nrows - 1) * mr.n + t;
    cpx<T> v[RL];
#pragma unroll
    for (int r = 0; r < RL; ++r) {
      const T x0 = xa[r * mr.T3], x1 = xb[r * mr.T3];
      v[r] = mk(x0, two ? x1 : T(0));
    }
    mdft<-1, RL>(v);
    cpx<T>* b = buf + rl * mr.SS + k1 * mr.S1 + k0;
#pragma unroll
    for (int r = 0; r < RL; ++r) b[r * mr.S2] = v[r];
  }
  __syncthreads();
  if (mr.R1 > 1) {
#define MIX_CALL(R) mixr_mid<T, -1, R>(mr, tw, buf, mr.rows, 1, 1)
    MIX_RADIX10(mr.R1, MIX_CALL)
#undef MIX_CALL
    __syncthreads();
  }
#define MIX_CALL(R) mixr_end<T, R>(mr, tw, buf, mr.rows, 1, 1)
  MIX_RADIX10(mr.R0, MIX_CALL)
#undef MIX_CALL
  __syncthreads();
  cpx<T>* __restrict__ out = a.out[f];
  for (int idx = threadIdx.x; idx < mr.rows * a.kxp; idx += blockDim.x) {
    const int rl = idx / a.kxp, k = idx - rl * a.kxp;
    long row;
    bool live, two;
    row_pair(p0 + rl, nrows, GRP ? group : 0, row, live, two);
    if (!live) continue;
    cpx<T> A, B;
    mixr_unpair(mr, buf + rl * mr.SS, k, a.kx, A, B);
    out[row * a.kxp + k] = A;
    if (two) out[(row + 1) * a.kxp + k] = B;
  }
}

}  // namespace ddx
