// Mixed-radix FFT passes for every grid extent without a size-specialised
// kernel (2^a 3^b 5^c other than 64, 128, 256, 512).
//
// A transform of length n = R_0 R_1 ... R_{P-1} (radices up to 16, three or
// fewer for most extents to 640) runs in place in one LDS buffer.  Write a position as digits
// (d_0, ..., d_{P-1}), d_0 most significant, M_p = R_{p+1} ... R_{P-1} the
// stride of digit p and L_p = R_0 ... R_{p-1}.  Decimation in frequency: pass
// p is a DFT over digit p of each of the n / R_p butterflies, its leg k
// multiplied by W_{n / L_p}^{k j} (j the value of the digits after p), and
// written back where it was read.  The first pass reads from global memory
// and the last one writes to it, so a pass boundary costs one LDS write, one
// barrier and one LDS read, and the buffer holds the transform once: the
// self-sorting form it replaces staged the input and the output in LDS too
// and needed two buffers.  After the last pass digit order is reversed: leg r
// of butterfly i holds frequency rev(i) + r L_{P-1}.
//
// The reversed sequence (decimation in time: legs multiplied first, digits
// P-1 ... 0) takes that order back to the natural one, which is how the
// x-row kernel runs c2r, products and r2c without reordering.
#pragma once

#include "ddx_kernels.h"

namespace ddx {

constexpr int MIX_MAXP = 6;

// i / d for 0 <= i < 2^16, d < 2^16: the high word of i * ceil(2^32 / d)
// (mag 0: d = 1)
inline unsigned mix_mag(int d) { return d <= 1 ? 0u : (unsigned)((0x100000000ull + (unsigned)d - 1) / (unsigned)d); }
__device__ __forceinline__ int mix_div(int i, unsigned mag) {
  return mag ? (int)__umulhi((unsigned)i, mag) : i;
}

struct MixPlan {
  int n, np;
  int R[MIX_MAXP], M[MIX_MAXP], L[MIX_MAXP];
  unsigned dR[MIX_MAXP], dM[MIX_MAXP];   // mix_mag of R and M
  int W, wshift;                         // tile width (a power of two)
};

// An x row: n = R0 R1 RL, digits (d0, d1, dl) at LDS entry dl S2 + d1 S1 + d0.
// Lanes take d0 (or d1) fastest, so S1 odd and S2 = R0 mod 16 spread the
// 16-byte entries of a pass over the banks.
struct MixRow {
  int n, R0, R1, RL;
  int J, T3, TM;      // butterflies of the first, last and middle pass
  int S1, S2, SS;     // strides, entries per sequence
  int rows;           // rows (PHYS) or row pairs (C2R, R2C) per workgroup
  unsigned dJ, dR1, dR0, dRL, dT3, dTM;
  long in_fs, out_fs; // field strides of the half-spectrum arrays (PHYS)
};

// Radix plan of a column pass; false if n does not factor.
bool mix_col_plan(int n, MixPlan* p);
// Plan of an x row with nin fields; false if this path does not apply.
bool mix_row_plan(int n, MixRow* p);

template <typename T> struct ColArgs;
template <typename T> struct RowArgs;

// Launches; false where the path does not apply (nothing launched).
template <typename T>
bool mix_col_launch(hipStream_t s, ColArgs<T>& a, const MixPlan& mp, int nslabs, int nfields, int dir,
                    bool spectral);
// group: rows of which only those of one group may share a transform (the
// members of a batched plan), nrows if all may; it divides nrows.
template <typename T>
bool mix_row_launch(hipStream_t s, const RowArgs<T>& a, const MixRow& mr, long nrows, long group);

}  // namespace ddx
