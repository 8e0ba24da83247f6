// Mixed-radix x-row passes; built once per real type and dimension
// (DDX_MIX_T, DDX_MIX_ND; DDX_MIX_ND = 0: the plain transforms and the
// dispatch, 1: the plain transforms within groups) so that the parts compile
// side by side.
#include <hip/hip_runtime.h>

#include "ddx_mixed_dev.h"

namespace ddx {

template <typename T, int PH, int ND>
void mix_row_phys_go(hipStream_t s, const RowArgs<T>& a, const MixRow& mr, unsigned blocks, unsigned thr, size_t lds,
                     long nrows);

template <typename T, bool GRP>
void mix_row_plain_go(hipStream_t s, const RowArgs<T>& a, const MixRow& mr, dim3 grid, unsigned thr, size_t lds,
                      long nrows, int group);

#if DDX_MIX_ND < 2

template <typename T, bool GRP>
void mix_row_plain_go(hipStream_t s, const RowArgs<T>& a, const MixRow& mr, dim3 grid, unsigned thr, size_t lds,
                      long nrows, int group) {
  if (a.mode == ROW_C2R) {
    if (mr.RL == 4) hipLaunchKernelGGL((mix_row_c2r<T, 4, GRP>), grid, dim3(thr), lds, s, a, mr, nrows, group);
    else if (mr.RL == 5) hipLaunchKernelGGL((mix_row_c2r<T, 5, GRP>), grid, dim3(thr), lds, s, a, mr, nrows, group);
    else hipLaunchKernelGGL((mix_row_c2r<T, 6, GRP>), grid, dim3(thr), lds, s, a, mr, nrows, group);
  } else {
    if (mr.RL == 4) hipLaunchKernelGGL((mix_row_r2c<T, 4, GRP>), grid, dim3(thr), lds, s, a, mr, nrows, group);
    else if (mr.RL == 5) hipLaunchKernelGGL((mix_row_r2c<T, 5, GRP>), grid, dim3(thr), lds, s, a, mr, nrows, group);
    else hipLaunchKernelGGL((mix_row_r2c<T, 6, GRP>), grid, dim3(thr), lds, s, a, mr, nrows, group);
  }
}

template void mix_row_plain_go<double, DDX_MIX_ND == 1>(hipStream_t, const RowArgs<double>&, const MixRow&, dim3,
                                                        unsigned, size_t, long, int);
template void mix_row_plain_go<float, DDX_MIX_ND == 1>(hipStream_t, const RowArgs<float>&, const MixRow&, dim3,
                                                       unsigned, size_t, long, int);

#endif

#if DDX_MIX_ND > 1

template <typename T, int PH, int ND>
void mix_row_phys_go(hipStream_t s, const RowArgs<T>& a, const MixRow& mr, unsigned blocks, unsigned thr, size_t lds,
                     long nrows) {
  if (mr.RL == 4) hipLaunchKernelGGL((mix_row_phys<T, PH, ND, 4>), dim3(blocks), dim3(thr), lds, s, a, mr, nrows);
  else if (mr.RL == 5) hipLaunchKernelGGL((mix_row_phys<T, PH, ND, 5>), dim3(blocks), dim3(thr), lds, s, a, mr, nrows);
  else hipLaunchKernelGGL((mix_row_phys<T, PH, ND, 6>), dim3(blocks), dim3(thr), lds, s, a, mr, nrows);
}

#define DDX_MIX_INST(PH)                                                                                   \
  template void mix_row_phys_go<DDX_MIX_T, PH, DDX_MIX_ND>(hipStream_t, const RowArgs<DDX_MIX_T>&,         \
                                                           const MixRow&, unsigned, unsigned, size_t, long);
DDX_MIX_INST(PH_HYDRO)
DDX_MIX_INST(PH_BOUSS)
DDX_MIX_INST(PH_MHD)

#elif DDX_MIX_ND == 0

template <typename T>
bool mix_row_launch(hipStream_t s, const RowArgs<T>& a, const MixRow& mr0, long nrows, long group) {
  MixRow mr = mr0;
  const bool phys = a.mode == ROW_PHYS;
  const int nseq = phys ? (a.nin + 1) / 2 : 1;
  if (phys || group % 2 == 0 || group >= nrows) group = 0;   // pairs stay inside the groups by themselves
  // rows, or pairs of rows
  const long units = phys ? nrows : group ? nrows / group * ((group + 1) / 2) : (nrows + 1) / 2;
  const int nf = phys ? 1 : (a.mode == ROW_C2R ? a.nin : a.nout);
  if (phys) {
    // the fields of a right-hand side are equally spaced arrays of one buffer
    mr.in_fs = a.nin > 1 ? a.in[1] - a.in[0] : 0;
    mr.out_fs = a.nout > 1 ? a.out[1] - a.out[0] : 0;
    for (int f = 1; f < a.nin; ++f)
      if (a.in[f] - a.in[0] != f * mr.in_fs) return false;
    for (int f = 1; f < a.nout; ++f)
      if (a.out[f] - a.out[0] != f * mr.out_fs) return false;
  }
  // 32-bit byte offsets from the first array
  const long top = phys ? (a.nin > a.nout ? a.nin * mr.in_fs : a.nout * mr.out_fs) : nrows * (long)a.kxp;
  if (mr.in_fs < 0 || mr.out_fs < 0 || (size_t)top * sizeof(cpx<T>) >= ((size_t)1 << 32)) return false;
  const size_t per = (size_t)nseq * mr.SS * sizeof(cpx<T>);
  if (per > 65536) return false;
  // Rows per workgroup: about 256 butterflies per pass within 40 KB of LDS
  // (four workgroups per CU), fewer while CUs would stay without one.
  int rows = 1;
  while (rows < 8 && 2 * rows * mr.T3 <= 256 && 2 * rows * per <= 40960 && (units / (2 * rows)) * nf >= 512) rows *= 2;
  mr.rows = rows;
  int thr = rows * (mr.T3 > nseq * mr.J ? mr.T3 : nseq * mr.J);
  thr = (thr + 63) / 64 * 64;
  if (thr > 256) thr = 256;
  const size_t lds = rows * per;
  const unsigned blocks = (unsigned)((units + rows - 1) / rows);
  if (phys) {
    switch (a.physics * 10 + a.ndim) {
      case PH_HYDRO * 10 + 2: mix_row_phys_go<T, PH_HYDRO, 2>(s, a, mr, blocks, thr, lds, nrows); break;
      case PH_HYDRO * 10 + 3: mix_row_phys_go<T, PH_HYDRO, 3>(s, a, mr, blocks, thr, lds, nrows); break;
      case PH_BOUSS * 10 + 2: mix_row_phys_go<T, PH_BOUSS, 2>(s, a, mr, blocks, thr, lds, nrows); break;
      case PH_BOUSS * 10 + 3: mix_row_phys_go<T, PH_BOUSS, 3>(s, a, mr, blocks, thr, lds, nrows); break;
      case PH_MHD * 10 + 2: mix_row_phys_go<T, PH_MHD, 2>(s, a, mr, blocks, thr, lds, nrows); break;
      case PH_MHD * 10 + 3: mix_row_phys_go<T, PH_MHD, 3>(s, a, mr, blocks, thr, lds, nrows); break;
      default: return false;
    }
    return true;
  }
  const dim3 grid(blocks, (unsigned)nf);
  if (group) mix_row_plain_go<T, true>(s, a, mr, grid, thr, lds, nrows, (int)group);
  else mix_row_plain_go<T, false>(s, a, mr, grid, thr, lds, nrows, 0);
  return true;
}

template bool mix_row_launch<double>(hipStream_t, const RowArgs<double>&, const MixRow&, long, long);
template bool mix_row_launch<float>(hipStream_t, const RowArgs<float>&, const MixRow&, long, long);

#endif

}  // namespace ddx
