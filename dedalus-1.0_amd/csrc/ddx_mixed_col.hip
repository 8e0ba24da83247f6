// Mixed-radix column passes; built once per real type (DDX_MIX_T).
#include <hip/hip_runtime.h>

#include "ddx_mixed_dev.h"

namespace ddx {

template <typename T, typename OFF>
static void mix_col_go(hipStream_t s, const ColArgs<T>& a, const MixPlan& mp, dim3 grid, int thr, size_t lds, int dir,
                       bool spectral) {
  // spectral prologues belong to backward passes only
  if (spectral) hipLaunchKernelGGL((mix_col_kernel<T, OFF, 1, true>), grid, dim3(thr), lds, s, a, mp);
  else if (dir > 0) hipLaunchKernelGGL((mix_col_kernel<T, OFF, 1, false>), grid, dim3(thr), lds, s, a, mp);
  else hipLaunchKernelGGL((mix_col_kernel<T, OFF, -1, false>), grid, dim3(thr), lds, s, a, mp);
}

template <typename T>
bool mix_col_launch(hipStream_t s, ColArgs<T>& a, const MixPlan& mp0, int nslabs, int nfields, int dir,
                    bool spectral) {
  MixPlan mp = mp0;
  const int n = mp.n;
  // 32-bit byte offsets from the start of a slab, where they reach
  const size_t lim = ((size_t)1 << 32) / sizeof(cpx<T>);
  const bool big = (size_t)a.in_rows * a.in_rs + a.ncols >= lim || (size_t)a.out_rows * a.out_rs + a.ncols >= lim;
  // Tile width: 16 columns within 48 KB of LDS (three workgroups per CU),
  // then narrower down to 64 bytes while the launch would leave CUs without a
  // workgroup.  Eight FP64 columns: 192^3 hydro step 700 against 686 us, 1000
  // members of 32^2 102 against 92, 75x96x120 transforms back 30.9 against
  // 32.4, most sizes even.  32 FP32 columns: 192^3 step 412 against 403 us,
  // 160x144x180 292 against 275, 1000 members of 32^2 88 against 79 (lanes
  // past the last of their 16 columns), smaller grids even.
  const int wmin = 64 / (int)sizeof(cpx<T>);
  int W = 16;
  while (W > 1 && (size_t)n * W * sizeof(cpx<T>) > 49152) W /= 2;
  while (W > wmin && (long)((a.ncols + W - 1) / W) * nslabs * nfields < 512) W /= 2;
  if ((size_t)n * W * sizeof(cpx<T>) > 65536) return false;
  mp.W = W;
  mp.wshift = 0;
  while ((1 << mp.wshift) < W) ++mp.wshift;
  const int ntiles = (a.ncols + W - 1) / W;
  a.nslabs = nslabs;
  a.nfields = nfields;
  a.ntiles = ntiles;
  dim3 grid(ntiles, nslabs, nfields);
  a.xcd_group = spectral && nfields > 1 && nslabs > 1 ? (a.group_hint ? 2 : 1) : 0;
  if (a.xcd_group == 2) grid = dim3((unsigned)(((nslabs + 7) / 8) * 8 * (long)ntiles * nfields), 1, 1);
  else if (a.xcd_group) grid = dim3((unsigned)((((long)ntiles * nslabs + 7) / 8) * 8 * nfields), 1, 1);
  int thr = (mp.M[0] * W + 63) / 64 * 64;
  thr = thr < 64 ? 64 : (thr > 512 ? 512 : thr);
  const size_t lds = (size_t)n * W * sizeof(cpx<T>);
  if (big) mix_col_go<T, unsigned long>(s, a, mp, grid, thr, lds, dir, spectral);
  else mix_col_go<T, unsigned>(s, a, mp, grid, thr, lds, dir, spectral);
  return true;
}

template bool mix_col_launch<DDX_MIX_T>(hipStream_t, ColArgs<DDX_MIX_T>&, const MixPlan&, int, int, int, bool);

}  // namespace ddx
