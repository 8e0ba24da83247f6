// Radix plans of the mixed-radix passes (host code).
#include "ddx_mixed.h"

namespace ddx {

namespace {

const int kRadices[] = {16, 15, 12, 10, 9, 8, 6, 5, 4, 3, 2};

// Factor lists of n in non-increasing radices, at least one of them 12 or
// less; keeps the one with the fewest passes, two or more, then the smallest
// largest radix (fewest registers), then the smallest sum.  A composite n in
// one pass would leave one lane per column with all of it (12^3 hydro step
// 59.5 us in one pass, 49.5 in two; 2000 members of 12 x 50 138 and 113).
void mix_search(int n0, int n, int top, int depth, int* cur, int* best, int* nbest) {
  if (n == 1) {
    if (depth && cur[depth - 1] > 12) return;
    if (depth == 1 && n0 != 2 && n0 != 3 && n0 != 5) return;
    int mb = 0, mc = 0, sb = 0, sc = 0;
    for (int i = 0; i < *nbest; ++i) { mb = best[i] > mb ? best[i] : mb; sb += best[i]; }
    for (int i = 0; i < depth; ++i) { mc = cur[i] > mc ? cur[i] : mc; sc += cur[i]; }
    if (*nbest < 0 || depth < *nbest || (depth == *nbest && (mc < mb || (mc == mb && sc < sb)))) {
      *nbest = depth;
      for (int i = 0; i < depth; ++i) best[i] = cur[i];
    }
    return;
  }
  if (depth == MIX_MAXP) return;
  for (int r : kRadices)
    if (r <= top && n % r == 0) {
      cur[depth] = r;
      mix_search(n0, n / r, r, depth + 1, cur, best, nbest);
    }
}

}  // namespace

bool mix_col_plan(int n, MixPlan* p) {
  int cur[MIX_MAXP], best[MIX_MAXP], nb = -1;
  if (n < 1 || n > 65535) return false;
  mix_search(n, n, 16, 0, cur, best, &nb);
  if (nb < 0) return false;
  while (nb < 2) best[nb++] = 1;   // at least a first and a last pass
  // The first pass takes the largest radix up to 12: with two spectral terms
  // a radix-16 butterfly has 32 loads in flight, 215 registers and two
  // wavefronts per SIMD; with 12 it is 163 and three (192^3 FP64 spectral
  // passes 71 -> 57 us, plain 35 -> 33 us; with 64-bit offsets 169 and two).
  if (best[0] > 12) {
    int i = 0;
    while (best[i] > 12) ++i;
    const int f = best[i];
    for (; i > 0; --i) best[i] = best[i - 1];
    best[0] = f;
  }
  p->n = n;
  p->np = nb;
  int L = 1;
  for (int i = 0; i < nb; ++i) {
    p->R[i] = best[i];
    p->L[i] = L;
    L *= best[i];
    p->M[i] = n / L;
    p->dR[i] = mix_mag(p->R[i]);
    p->dM[i] = mix_mag(p->M[i]);
  }
  p->W = 1;
  p->wshift = 0;
  return true;
}

bool mix_row_plan(int n, MixRow* p) {
  // RL last (4 where it divides n: the products of 12 fields at 4 positions
  // fit the registers); n / RL in one radix if possible, else two, up to 10
  // (the first pass has two loads per leg in flight: with radix 16 the FP64
  // hydro row takes 156 registers, with 10 it fits 96, five wavefronts per
  // SIMD; 192^3 x rows 173 -> 143 us).  Extents without such a plan (576,
  // 640) keep the general row kernel.
  const int rls[3] = {4, 5, 6};
  int bR0 = 0, bR1 = 0, bRL = 0;
  for (int rl : rls) {
    if (n % rl) continue;
    const int q = n / rl;
    int r0 = 0, r1 = 0;
    auto radix = [](int r) {
      if (r == 1) return true;
      for (int k : kRadices)
        if (k == r) return k <= 10;
      return false;
    };
    if (radix(q)) { r0 = q; r1 = 1; }
    else {
      for (int k : kRadices)   // descending: the last hit has the smallest r0 >= r1
        if (k <= 10 && q % k == 0 && radix(q / k) && k >= q / k) { r0 = k; r1 = q / k; }
    }
    if (!r0) continue;
    if (!bRL || (bR1 > 1 && r1 == 1)) { bR0 = r0; bR1 = r1; bRL = rl; }
  }
  if (!bRL) return false;
  p->n = n;
  p->R0 = bR0; p->R1 = bR1; p->RL = bRL;
  p->J = n / bR0;
  p->T3 = bR0 * bR1;
  p->TM = bR0 * bRL;
  p->S1 = bR0 | 1;
  if (bR1 == 1) {
    p->S2 = bR0 | 1;
  } else {
    p->S2 = bR1 * p->S1;
    while (p->S2 % 16 != bR0 % 16) ++p->S2;
  }
  p->SS = bRL * p->S2;
  p->dJ = mix_mag(p->J); p->dR1 = mix_mag(bR1); p->dR0 = mix_mag(bR0); p->dRL = mix_mag(bRL);
  p->dT3 = mix_mag(p->T3); p->dTM = mix_mag(p->TM);
  p->rows = 1;
  p->in_fs = p->out_fs = 0;
  return true;
}

}  // namespace ddx
