// Learned sub-grid closure kernels (gfx950): BF16 MFMA 3x3 periodic
// convolutions with fused epilogues, and the data movement around them.
//
// Layouts
//   activations  [npix][Cp]        bf16 bit patterns, npix = B*H*W (b, y, x
//                                  order), channels padded to multiples of 16
//   weights      [Co][9][Ci]       bf16, tap t = 3*(dy+1) + (dx+1)
//   pre-activations / gradients    fp32, same pixel-major layout
// The domain is periodic in y and x, so taps wrap around.
//
// v_mfma_f32_16x16x16_bf16 per wavefront (D = A B, 16 x 16 x 16):
//   A (rows m, cols k): lane l holds A[l % 16][4*(l/16) + i], i < 4
//   B (rows k, cols n): lane l holds B[4*(l/16) + i][l % 16]
//   D:                  lane l holds D[4*(l/16) + i][l % 16]
// ddx_mfma_probe runs one tile with exactly these placements so the layout
// can be checked against a host product.
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdint>
#include <cstring>
#include <type_traits>
#include <string>

#include "../../include/ddx.h"
#include "../../include/ddx_closure.h"

namespace ddx {
int set_error(int code, const std::string& msg);  // defined in ddx.hip
}

namespace {

// Workgroup barrier that orders LDS only: the release/acquire fences name the
// local address space, so global loads (the next tile's halo, issued before
// the current tile's compute) and stores stay in flight across it; a plain
// __syncthreads() also waits for every outstanding global access.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

#define CL_LAUNCHCHK(name)                                                                  \
  do {                                                                                      \
    hipError_t e_ = hipGetLastError();                                                      \
    if (e_ != hipSuccess)                                                                   \
      return ddx::set_error(DDX_ERR_HIP, std::string(name) + ": " + hipGetErrorString(e_)); \
  } while (0)

// fp32 -> bf16, round to nearest even (gfx950 v_cvt_pk_bf16_f32)
__device__ inline uint16_t f2bf(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }

__device__ inline float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// GELU in its tanh form, written as z sigma(s) with
// s = 2 sqrt(2/pi) (z + 0.044715 z^3): 0.5 z (1 + tanh(s/2)) = z sigma(s), so
// the negative tail has no cancellation.  sigma(s) = 1 / (1 + 2^u) with
// u = -s log2(e) = z (A + B z^2): the constants fold -2 sqrt(2/pi) log2(e),
// so one multiply, one fma and one multiply form the exponent of the
// hardware exp2, and one reciprocal finishes sigma (saturating to 0 and 1).
//   GELU'(z) = sigma(s) + z sigma(s) (1 - sigma(s)) s'(z),
//   s'(z) = 2 sqrt(2/pi) (1 + 3 * 0.044715 z^2)
constexpr float GELU_A = -2.3022082f;            // -2 sqrt(2/pi) log2(e)
constexpr float GELU_B = -2.3022082f * 0.044715f;
__device__ inline float gelu_sigma(float z) {
  const float u = z * __builtin_fmaf(z * z, GELU_B, GELU_A);
  return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(u));
}
__device__ inline float gelu(float z) { return z * gelu_sigma(z); }
__device__ inline float gelu_grad(float z) {
  const float sg = gelu_sigma(z);
  const float ds = 1.5957691216057308f * (1.0f + 0.134145f * z * z);
  return sg + z * sg * (1.0f - sg) * ds;
}

__device__ inline bf16x4 load4(const uint16_t* p) {
  // four consecutive channels; channel offsets are multiples of 4, so 8-byte aligned
  const uint2 v = *reinterpret_cast<const uint2*>(p);
  bf16x4 r;
  r[0] = (short)(v.x & 0xffffu);
  r[1] = (short)(v.x >> 16);
  r[2] = (short)(v.y & 0xffffu);
  r[3] = (short)(v.y >> 16);
  return r;
}

__device__ inline int wrapi(int i, int n) { return i < 0 ? i + n : (i >= n ? i - n : i); }

struct ConvArgs {
  const uint16_t* x;  // [npix][Ci]
  const uint16_t* w;  // [Co][9][Ci]
  const float* bias;  // [Co] or null
  const float* aux;   // [npix][Co] pre-activation for DDX_CONV_GELU_GRAD
  float* out_f32;     // [npix][Co] or null
  uint16_t* out_bf16; // [npix][Co] or null
  int B, H, W, Ci, Co, mode;
  int cout;           // channels per pixel of out_f32 (Co, or fewer: only those are stored)
  double* bpart;      // GELU_GRAD, tile kernel: [gridDim.x][Co] sums of the fp32 result over a block's pixels, or null
};

// One wavefront: 16 consecutive pixels x all Co = 16*NCO output channels.
// Four wavefronts per block; no block-level synchronisation.
template <int NCO>
__global__ void __launch_bounds__(256) conv3x3_kernel(ConvArgs a) {
  const int lane = threadIdx.x & 63;
  const long tile = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  const long npix = (long)a.B * a.H * a.W;
  if (tile * 16 >= npix) return;
  const long p0 = tile * 16;
  const int m = lane & 15, kq = lane >> 4;
  const long pm = p0 + m;
  const long hw = (long)a.H * a.W;
  const int b = (int)(pm / hw);
  const int rem = (int)(pm - (long)b * hw);
  const int py = rem / a.W, px = rem - py * a.W;
  f32x4 acc[NCO];
#pragma unroll
  for (int j = 0; j < NCO; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int t = 0; t < 9; ++t) {
    const int yy = wrapi(py + t / 3 - 1, a.H), xx = wrapi(px + t % 3 - 1, a.W);
    const uint16_t* xrow = a.x + (((long)b * a.H + yy) * a.W + xx) * a.Ci + 4 * kq;
    const uint16_t* wrow = a.w + ((long)m * 9 + t) * a.Ci + 4 * kq;
    const long wstride = 16L * 9 * a.Ci;  // next 16 output channels
    for (int kc = 0; kc < a.Ci; kc += 16) {
      const bf16x4 av = load4(xrow + kc);
#pragma unroll
      for (int j = 0; j < NCO; ++j) {
        const bf16x4 bv = load4(wrow + j * wstride + kc);
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av, bv, acc[j], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < NCO; ++j) {
    const int c = j * 16 + m;
    const float bv = a.bias ? a.bias[c] : 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const long o = (p0 + 4 * kq + i) * a.Co + c;
      float v = acc[j][i];
      float act;
      if (a.mode == DDX_CONV_GELU_GRAD) {
        v *= gelu_grad(a.aux[o]);
        act = v;
      } else {
        v += bv;
        act = a.mode == DDX_CONV_GELU ? gelu(v) : v;
      }
      if (a.out_f32 && c < a.cout) a.out_f32[(p0 + 4 * kq + i) * a.cout + c] = v;
      if (a.out_bf16) a.out_bf16[o] = f2bf(act);
    }
  }
}

__device__ inline bf16x4 lds4(const uint16_t* p) {
  const uint2 v = *reinterpret_cast<const uint2*>(p);
  bf16x4 r;
  r[0] = (short)(v.x & 0xffffu);
  r[1] = (short)(v.x >> 16);
  r[2] = (short)(v.y & 0xffffu);
  r[3] = (short)(v.y >> 16);
  return r;
}

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

// eight consecutive bf16 from LDS (16-byte aligned)
__device__ inline bf16x8 lds16(const uint16_t* p) {
  const uint4 v = *reinterpret_cast<const uint4*>(p);
  const u32x4 u = {v.x, v.y, v.z, v.w};
  return __builtin_bit_cast(bf16x8, u);
}

// eight consecutive bf16 from LDS as two 8-byte reads
__device__ inline bf16x8 lds8(const uint16_t* p) {
  const uint2 lo = *reinterpret_cast<const uint2*>(p);
  const uint2 hi = *reinterpret_cast<const uint2*>(p + 4);
  const u32x4 v = {lo.x, lo.y, hi.x, hi.y};
  return __builtin_bit_cast(bf16x8, v);
}

// LDS-tiled 3x3 convolution for CI, CO in {16, 32}.  Output tile = 256 pixels
// of one image, 4 rows x 64 columns (TC = 64) or 8 x 32 (TC = 32); wavefront w
// owns 64 of them as four 16-pixel fragments.  Blocks loop over tiles (tile c,
// c + gridDim.x, ...): the weights are staged in LDS once per block, and the
// next tile's input halo is loaded into registers while the current tile
// computes.  A training batch of 32 images 64^2 (one tile per block) takes
// 10.8 us per 32-channel layer, the larger part of it the 24 MB of fp32 and
// bf16 stores: stored straight from the accumulators, in 64-byte pieces
// instead of the staging's whole lines, it took a microsecond more.  TC = 32
// multiplies 32 channels in two steps of 16, the sums of conv3x3_kernel.
// Pixel stride and weight-row stride CI + 4 (bf16) place the 16 rows of a
// fragment read in distinct bank pairs.  CI = 32 uses the gfx950 16x16x32
// bf16 MFMA, CI = 16 the 16x16x16 one.
//
// BF (bf16 output only, no fp32 output or GELU gradient: the inference
// pass): bias and activation are applied to the accumulators and the
// results staged as bf16, which halves the staging LDS; the kernel then fits
// three workgroups per CU instead of two.
//
// EX (training): sums of the GELU gradient for the bias, and fp32 outputs of
// fewer than CO channels.  Decided at run time, the two cost every layer call
// 2 to 20 registers and up to 14 % (one image 512^2, 32 -> 32 channels, both
// outputs: 20.0 us, 17.4 without).
//
// Order of the first requests: the halo, then the weights; the GELU
// gradient's pre-activations before the products.  With 32 channels in
// 64-column tiles those registers are short and the reverse is faster (WFIRST:
// the same call 18.6 -> 17.4 us), and with BF the tile's address is formed
// after the products (LATE: the bf16-only call 14.8 -> 13.9 us).
template <int CI, int CO, bool BF, int TC, bool EX, int MINW>
__global__ void __launch_bounds__(256, MINW) conv3x3_tile_kernel(ConvArgs a, long ntiles) {
  constexpr bool WFIRST = CI == 32 && TC == 64 && !BF, LATE = CI == 32 && TC == 64 && BF;
  constexpr int PS = CI + 4, WS = CI + 4;
  constexpr int TR = 256 / TC, HR = TR + 2, HC = TC + 2;
  constexpr int NCO = CO / 16;
  constexpr int CK = CI / 8;                       // 16-byte chunks per pixel
  constexpr int NH = HR * HC * CK, HPT = (NH + 255) / 256;
  constexpr int NW = CO * 9 * CK, WPT = (NW + 255) / 256;
  // the halo buffer also stages each wavefront's 64 x CO results (fp32, or
  // bf16 with BF)
  constexpr int ES = CO + 4;                                  // fp32 staging row stride (floats)
  constexpr int EB = CO + 8;                                  // bf16 staging row stride (bf16)
  constexpr int HALO_B = HR * HC * PS * 2, STAGE_B = BF ? 4 * 64 * EB * 2 : 4 * 64 * ES * 4;
  constexpr int BUF_B = HALO_B > STAGE_B ? HALO_B : STAGE_B;
  __shared__ __align__(16) uint16_t halo[BUF_B / 2];
  __shared__ __align__(16) uint16_t wl[CO * 9 * WS];
  const int tid = threadIdx.x;
  const int tiles_x = a.W / TC, tiles_y = a.H / TR;
  uint4 hv[HPT];
  auto fetch = [&](long tile) {
    long rest = tile;
    const int tx = (int)(rest % tiles_x);
    rest /= tiles_x;
    const int ty = (int)(rest % tiles_y);
    const int b = (int)(rest / tiles_y);
    const int x0 = tx * TC, y0 = ty * TR;
#pragma unroll
    for (int k = 0; k < HPT; ++k) {
      const int i = tid + k * 256;
      if (i < NH) {
        const int pix = i / CK, ch = i - pix * CK;
        const int r = pix / HC, c = pix - r * HC;
        const int yy = wrapi(y0 - 1 + r, a.H), xx = wrapi(x0 - 1 + c, a.W);
        hv[k] = *reinterpret_cast<const uint4*>(&a.x[(((long)b * a.H + yy) * a.W + xx) * CI + ch * 8]);
      }
    }
  };
  const int wave = tid >> 6, lane = tid & 63;
  const int m = lane & 15, kq = lane >> 4;
  const bool grad = a.mode == DDX_CONV_GELU_GRAD, gelu_on = a.mode == DDX_CONV_GELU;
  float bias4[4] = {0.f, 0.f, 0.f, 0.f};   // channels (lane % (CO/4)) * 4 + e (fp32 staging)
  float biasj[NCO];                         // channels j * 16 + m (BF)
#pragma unroll
  for (int j = 0; j < NCO; ++j) biasj[j] = 0.f;
  if (!grad && a.bias) {
    const int cb = (lane % (CO / 4)) * 4;
#pragma unroll
    for (int e = 0; e < 4; ++e) bias4[e] = a.bias[cb + e];
#pragma unroll
    for (int j = 0; j < NCO; ++j) biasj[j] = a.bias[j * 16 + m];
  }
  long tile = blockIdx.x;
  if (!WFIRST && tile < ntiles) fetch(tile);
  uint4 wv[WPT];
#pragma unroll
  for (int k = 0; k < WPT; ++k) {
    const int i = tid + k * 256;
    if (i < NW) wv[k] = *reinterpret_cast<const uint4*>(&a.w[(long)i * 8]);
  }
#pragma unroll
  for (int k = 0; k < WPT; ++k) {
    const int i = tid + k * 256;
    if (i < NW) {
      const int row = i / CK, ch = i - row * CK;
      uint2* d = reinterpret_cast<uint2*>(&wl[row * WS + ch * 8]);
      d[0] = make_uint2(wv[k].x, wv[k].y);
      d[1] = make_uint2(wv[k].z, wv[k].w);
    }
  }
  if (WFIRST && tile < ntiles) fetch(tile);
  double bsum[4] = {0.0, 0.0, 0.0, 0.0};   // EX: this thread's channels (lane % (CO/4)) * 4 + e over its pixels
  // pixel px of the wavefront's 64: tile row and column
  auto prow = [&](int px) { return TC == 64 ? wave : 2 * wave + (px >> 5); };
  auto pcol = [&](int px) { return TC == 64 ? px : px & 31; };
  for (; tile < ntiles; tile += gridDim.x) {
    lds_barrier();  // the previous tile's fragment reads are done
#pragma unroll
    for (int k = 0; k < HPT; ++k) {
      const int i = tid + k * 256;
      if (i < NH) {
        const int pix = i / CK, ch = i - pix * CK;
        uint2* d = reinterpret_cast<uint2*>(&halo[pix * PS + ch * 8]);
        d[0] = make_uint2(hv[k].x, hv[k].y);
        d[1] = make_uint2(hv[k].z, hv[k].w);
      }
    }
    lds_barrier();
    const long next = tile + gridDim.x;
    if (next < ntiles) fetch(next);  // in flight while this tile computes
    long p00 = 0;   // the tile's first pixel
    auto origin = [&]() {
      long rest = tile;
      const int tx = (int)(rest % tiles_x);
      rest /= tiles_x;
      const int ty = (int)(rest % tiles_y);
      const int b = (int)(rest / tiles_y);
      p00 = ((long)b * a.H + ty * TR) * a.W + tx * TC;
    };
    if (!LATE) origin();
    auto gpix = [&](int px) { return p00 + (long)prow(px) * a.W + pcol(px); };
    // pre-activations of this thread's output chunks (see the staging below)
    constexpr int C4 = CO / 4, NR = C4;
    const int c = (lane % C4) * 4;
    float4 zaux[NR];
    auto load_aux = [&]() {
#pragma unroll
      for (int r = 0; r < NR; ++r)
        zaux[r] = *reinterpret_cast<const float4*>(&a.aux[gpix((lane + 64 * r) / C4) * CO + c]);
    };
    if (!BF && !WFIRST && grad) load_aux();
    f32x4 acc[4][NCO];
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int j = 0; j < NCO; ++j) acc[q][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 9; ++t) {
      const int dy = t / 3, dx = t % 3;
      if constexpr (CI % 32 == 0 && TC == 64) {
#pragma unroll
        for (int kc = 0; kc < CI / 32; ++kc) {
          bf16x8 bv[NCO];
#pragma unroll
          for (int j = 0; j < NCO; ++j) bv[j] = lds8(&wl[((j * 16 + m) * 9 + t) * WS + kc * 32 + 8 * kq]);
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const bf16x8 av = lds8(&halo[((prow(q * 16) + dy) * HC + pcol(q * 16) + m + dx) * PS + kc * 32 + 8 * kq]);
#pragma unroll
            for (int j = 0; j < NCO; ++j)
              acc[q][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv[j], acc[q][j], 0, 0, 0);
          }
        }
      } else {
#pragma unroll
        for (int kc = 0; kc < CI / 16; ++kc) {
          bf16x4 bv[NCO];
#pragma unroll
          for (int j = 0; j < NCO; ++j) bv[j] = lds4(&wl[((j * 16 + m) * 9 + t) * WS + kc * 16 + 4 * kq]);
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const bf16x4 av = lds4(&halo[((prow(q * 16) + dy) * HC + pcol(q * 16) + m + dx) * PS + kc * 16 + 4 * kq]);
#pragma unroll
            for (int j = 0; j < NCO; ++j)
              acc[q][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av, bv[j], acc[q][j], 0, 0, 0);
          }
        }
      }
    }
    if (LATE) origin();
    lds_barrier();  // every wavefront is done with the halo
    if constexpr (BF) {
      // activations of the D fragments (pixel q*16 + 4kq + i, channel j*16 + m)
      // as [64][EB] bf16, then 4 channels (8 bytes) per lane and chunk to HBM
      uint16_t* sb = halo + wave * 64 * EB;
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int j = 0; j < NCO; ++j)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float v = acc[q][j][i] + biasj[j];
            sb[(q * 16 + 4 * kq + i) * EB + j * 16 + m] = f2bf(gelu_on ? gelu(v) : v);
          }
      lds_barrier();
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        const int px = (lane + 64 * r) / C4;
        *reinterpret_cast<uint2*>(&a.out_bf16[gpix(px) * CO + c]) =
            *reinterpret_cast<const uint2*>(&sb[px * EB + c]);
      }
      continue;
    }
    // stage D fragments (pixel q*16 + 4kq + i, channel j*16 + m) as [64][ES] fp32
    float* st = reinterpret_cast<float*>(halo) + wave * 64 * ES;
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int j = 0; j < NCO; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) st[(q * 16 + 4 * kq + i) * ES + j * 16 + m] = acc[q][j][i];
    lds_barrier();
    if (WFIRST && grad) load_aux();
    // 4 channels per chunk; a lane's channels c..c+3 are the same in every
    // chunk (C4 divides 64), so its bias was read once before the tile loop
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const int px = (lane + 64 * r) / C4;
      const float4 d = *reinterpret_cast<const float4*>(&st[px * ES + c]);
      float v[4] = {d.x, d.y, d.z, d.w}, act[4];
      const long gp = gpix(px), o = gp * CO + c;
      if (grad) {
        const float zz[4] = {zaux[r].x, zaux[r].y, zaux[r].z, zaux[r].w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[e] *= gelu_grad(zz[e]);
          act[e] = v[e];
          if (EX) bsum[e] += (double)v[e];
        }
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[e] += bias4[e];
          act[e] = gelu_on ? gelu(v[e]) : v[e];
        }
      }
      if (a.out_f32) {
        if (!EX || a.cout == CO) {
          *reinterpret_cast<float4*>(&a.out_f32[o]) = make_float4(v[0], v[1], v[2], v[3]);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (c + e < a.cout) a.out_f32[gp * a.cout + c + e] = v[e];
        }
      }
      if (a.out_bf16)
        *reinterpret_cast<uint2*>(&a.out_bf16[o]) =
            make_uint2((uint32_t)f2bf(act[0]) | ((uint32_t)f2bf(act[1]) << 16),
                       (uint32_t)f2bf(act[2]) | ((uint32_t)f2bf(act[3]) << 16));
    }
  }
  if constexpr (EX) {
    if (a.bpart) {
      // lanes, then wavefronts, in a fixed order
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int d = CO / 4; d < 64; d *= 2) bsum[e] += __shfl_xor(bsum[e], d);
      lds_barrier();
      double* sh = reinterpret_cast<double*>(halo);
      if (lane < CO / 4)
#pragma unroll
        for (int e = 0; e < 4; ++e) sh[wave * CO + lane * 4 + e] = bsum[e];
      lds_barrier();
      if (tid < CO) a.bpart[(long)blockIdx.x * CO + tid] = ((sh[tid] + sh[CO + tid]) + sh[2 * CO + tid]) + sh[3 * CO + tid];
    }
  }
}

// Weight-gradient partials over one chunk of pixels, all nine taps per wavefront:
// partial[chunk][co][t][ci] = sum_{p in chunk} dz[p][co] x[shift_t(p)][ci].
// grid.x = chunks, grid.y = (Co/16) * (Ci/16); one wavefront per block.
__global__ void __launch_bounds__(64) conv3x3_wgrad_kernel(const uint16_t* __restrict__ x,
                                                            const uint16_t* __restrict__ dz,
                                                            float* __restrict__ partial, int B,
                                                            int H, int W, int Ci, int Co,
                                                            int pch) {
  const int lane = threadIdx.x;
  const int m = lane & 15, kq = lane >> 4;
  const int nct = Ci / 16;
  const int co0 = (blockIdx.y / nct) * 16, ci0 = (blockIdx.y % nct) * 16;
  const long hw = (long)H * W;
  const long npix = (long)B * hw;
  const long pstart = (long)blockIdx.x * pch;
  const long pend = pstart + pch < npix ? pstart + pch : npix;
  f32x4 acc[9];
#pragma unroll
  for (int t = 0; t < 9; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (long pk = pstart; pk < pend; pk += 16) {
    bf16x4 av;
    int pb[4], py[4], px[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const long p = pk + 4 * kq + i;
      av[i] = (short)dz[p * Co + co0 + m];  // A[m = co][k = p]
      pb[i] = (int)(p / hw);
      const int rem = (int)(p - (long)pb[i] * hw);
      py[i] = rem / W;
      px[i] = rem - py[i] * W;
    }
#pragma unroll
    for (int t = 0; t < 9; ++t) {
      bf16x4 bv;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int yy = wrapi(py[i] + t / 3 - 1, H), xx = wrapi(px[i] + t % 3 - 1, W);
        bv[i] = (short)x[(((long)pb[i] * H + yy) * W + xx) * Ci + ci0 + m];  // B[k = p][n = ci]
      }
      acc[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av, bv, acc[t], 0, 0, 0);
    }
  }
#pragma unroll
  for (int t = 0; t < 9; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int co = co0 + 4 * kq + i, ci = ci0 + m;
      partial[(((long)blockIdx.x * Co + co) * 9 + t) * Ci + ci] = acc[t][i];
    }
}

// LDS-tiled weight gradient for CI, CO in {16, 32}.  Block c accumulates over
// output tiles c, c + gridDim.x, ... (256 pixels of one image, 4 x 64 for TC =
// 64 and 8 x 32 for TC = 32, as in the forward kernel) and writes
// partial[c][co][t][ci].  Per tile, dz (256 pixels x CO) and the input halo
// are staged channel-major, so the MFMA's K dimension (32 pixels) is
// contiguous: A[m = co][k = p] from dzT[co][p] (16-byte reads), B[k = p][n =
// ci] from haloT[ci][row][col].  The three column shifts of a row come from
// one run of five 4-byte words, shifted in registers by 16 bits for the odd
// one; reading each shifted operand as eight 2-byte words took 36 LDS
// instructions per 16 pixels where this takes 15 per 32 (18.6 -> 11 us for 32
// channels and 32 images 64^2).  The transposed staging writes pixel pairs.
// Wavefront w owns the (co tile, ci tile) pairs w, w + 4, ... with all nine
// tap accumulators.  The next tile's loads are in flight while one computes.
//
// With dzf (the fp32 dz), the block also sums dz over its pixels per output
// channel in double (the bias gradient), thread t taking channel t mod CO and
// every (256 / CO)-th pixel, combined in a fixed order into
// bpartial[block][co]: the column sums ride along with the tiles this
// kernel reads anyway, instead of a separate pass over dz.
template <int CI, int CO, int TC>
__global__ void __launch_bounds__(256) conv3x3_wgrad_tile_kernel(const uint16_t* __restrict__ x,
                                                                 const uint16_t* __restrict__ dz,
                                                                 float* __restrict__ partial,
                                                                 int B, int H, int W,
                                                                 const float* __restrict__ dzf = nullptr,
                                                                 double* __restrict__ bpartial = nullptr) {
  constexpr int TR = 256 / TC, HR = TR + 2, HC = TC + 2;
  constexpr int DS = 264;            // dzT row stride (bf16): 16-byte rows, 16 rows on distinct banks
  constexpr int HRS = TC + 4;        // halo row stride
  constexpr int HS = HR * HRS + 2;   // halo channel stride, odd in 4-byte words
  static_assert((HS / 2) % 2 == 1 && HS % 2 == 0, "halo channel stride");
  constexpr int NCT = CI / 16, NPAIR = (CO / 16) * (CI / 16);
  constexpr int NPW = (NPAIR + 3) / 4;  // pairs per wavefront
  constexpr int ND = 128 * (CO / 4), DPT = (ND + 255) / 256;            // dz pixel pairs x 4 channels
  constexpr int NH = HR * (HC / 2) * (CI / 4), HPT = (NH + 255) / 256;  // halo pixel pairs x 4 channels
  __shared__ __align__(16) uint16_t dzT[CO * DS];
  __shared__ __align__(16) uint16_t haloT[CI * HS];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int m = lane & 15, kq = lane >> 4;
  const int tiles_x = W / TC, tiles_y = H / TR;
  const long ntiles = (long)B * tiles_y * tiles_x;
  f32x4 acc[NPW][9];
#pragma unroll
  for (int u = 0; u < NPW; ++u)
#pragma unroll
    for (int t = 0; t < 9; ++t) acc[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  constexpr int PG = 256 / CO;              // pixel groups of the bias sums
  const int bco = tid % CO, bpg = tid / CO;
  double bsum = 0.0;
  uint2 dv[DPT][2], hv[HPT][2];
  float bv[256 / PG];
  auto fetch = [&](long tile) {
    long rest = tile;
    const int tx = (int)(rest % tiles_x);
    rest /= tiles_x;
    const int ty = (int)(rest % tiles_y);
    const int b = (int)(rest / tiles_y);
    const int x0 = tx * TC, y0 = ty * TR;
#pragma unroll
    for (int k = 0; k < DPT; ++k) {
      const int i = tid + k * 256;
      if (i < ND) {
        const int pp = i / (CO / 4), ch = (i - pp * (CO / 4)) * 4, pix = 2 * pp;
        const uint16_t* q = &dz[(((long)b * H + y0 + pix / TC) * W + x0 + pix % TC) * CO + ch];
        dv[k][0] = *reinterpret_cast<const uint2*>(q);
        dv[k][1] = *reinterpret_cast<const uint2*>(q + CO);
      }
    }
#pragma unroll
    for (int k = 0; k < HPT; ++k) {
      const int i = tid + k * 256;
      if (i < NH) {
        const int pp = i / (CI / 4), ch = (i - pp * (CI / 4)) * 4;
        const int r = pp / (HC / 2), c = 2 * (pp - r * (HC / 2));
        const long row = ((long)b * H + wrapi(y0 - 1 + r, H)) * W;
        hv[k][0] = *reinterpret_cast<const uint2*>(&x[(row + wrapi(x0 - 1 + c, W)) * CI + ch]);
        hv[k][1] = *reinterpret_cast<const uint2*>(&x[(row + wrapi(x0 + c, W)) * CI + ch]);
      }
    }
    if (dzf) {
#pragma unroll
      for (int k = 0; k < 256 / PG; ++k) {
        const int pix = bpg + PG * k;
        bv[k] = dzf[(((long)b * H + y0 + pix / TC) * W + x0 + pix % TC) * CO + bco];
      }
    }
  };
  // four channels of two adjacent pixels -> one 4-byte word per channel
  auto put = [](uint16_t* base, int stride, int o, const uint2 (&v)[2]) {
    *reinterpret_cast<uint32_t*>(&base[o]) = __builtin_amdgcn_perm(v[1].x, v[0].x, 0x05040100u);
    *reinterpret_cast<uint32_t*>(&base[o + stride]) = __builtin_amdgcn_perm(v[1].x, v[0].x, 0x07060302u);
    *reinterpret_cast<uint32_t*>(&base[o + 2 * stride]) = __builtin_amdgcn_perm(v[1].y, v[0].y, 0x05040100u);
    *reinterpret_cast<uint32_t*>(&base[o + 3 * stride]) = __builtin_amdgcn_perm(v[1].y, v[0].y, 0x07060302u);
  };
  long tile = blockIdx.x;
  if (tile < ntiles) fetch(tile);
  for (; tile < ntiles; tile += gridDim.x) {
    lds_barrier();  // the previous tile's reads are done
#pragma unroll
    for (int k = 0; k < DPT; ++k) {
      const int i = tid + k * 256;
      if (i < ND) {
        const int pp = i / (CO / 4), ch = (i - pp * (CO / 4)) * 4;
        put(dzT, DS, ch * DS + 2 * pp, dv[k]);
      }
    }
#pragma unroll
    for (int k = 0; k < HPT; ++k) {
      const int i = tid + k * 256;
      if (i < NH) {
        const int pp = i / (CI / 4), ch = (i - pp * (CI / 4)) * 4;
        const int r = pp / (HC / 2), c = 2 * (pp - r * (HC / 2));
        put(haloT, HS, ch * HS + r * HRS + c, hv[k]);
      }
    }
    if (dzf) {
#pragma unroll
      for (int k = 0; k < 256 / PG; ++k) bsum += (double)bv[k];   // in pixel order
    }
    lds_barrier();
    if (tile + gridDim.x < ntiles) fetch(tile + gridDim.x);
#pragma unroll
    for (int u = 0; u < NPW; ++u) {
      const int pair = wave + 4 * u;
      if (pair >= NPAIR) break;
      const int co0 = (pair / NCT) * 16, ci0 = (pair % NCT) * 16;
      const uint16_t* hb = &haloT[(ci0 + m) * HS + 8 * kq];
#pragma unroll 2
      for (int ks = 0; ks < 8; ++ks) {       // 32 pixels per K step
        const int row = (ks * 32) / TC, col0 = (ks * 32) % TC;
        const bf16x8 av = lds16(&dzT[(co0 + m) * DS + ks * 32 + 8 * kq]);
#pragma unroll
        for (int dy = 0; dy < 3; ++dy) {
          const uint32_t* hp = reinterpret_cast<const uint32_t*>(hb + (row + dy) * HRS + col0);
          const uint32_t d0 = hp[0], d1 = hp[1], d2 = hp[2], d3 = hp[3], d4 = hp[4];
          const u32x4 s0 = {d0, d1, d2, d3}, s2 = {d1, d2, d3, d4};
          const u32x4 s1 = {__builtin_amdgcn_alignbit(d1, d0, 16), __builtin_amdgcn_alignbit(d2, d1, 16),
                            __builtin_amdgcn_alignbit(d3, d2, 16), __builtin_amdgcn_alignbit(d4, d3, 16)};
          acc[u][3 * dy] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, __builtin_bit_cast(bf16x8, s0), acc[u][3 * dy], 0, 0, 0);
          acc[u][3 * dy + 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, __builtin_bit_cast(bf16x8, s1), acc[u][3 * dy + 1], 0, 0, 0);
          acc[u][3 * dy + 2] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, __builtin_bit_cast(bf16x8, s2), acc[u][3 * dy + 2], 0, 0, 0);
        }
      }
    }
  }
  // D[row = co (4 kq + i)][col = ci (m)] of each tap
#pragma unroll
  for (int u = 0; u < NPW; ++u) {
    const int pair = wave + 4 * u;
    if (pair >= NPAIR) break;
    const int co0 = (pair / NCT) * 16, ci0 = (pair % NCT) * 16;
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        partial[(((long)blockIdx.x * CO + co0 + 4 * kq + i) * 9 + t) * CI + ci0 + m] = acc[u][t][i];
  }
  if (dzf) {
    // the PG partial sums of each channel, combined in group order
    lds_barrier();
    double* sh = reinterpret_cast<double*>(haloT);   // 256 doubles fit the halo buffer
    sh[tid] = bsum;
    lds_barrier();
    if (tid < CO) {
      double r = 0.0;
      for (int g = 0; g < PG; ++g) r += sh[g * CO + tid];
      bpartial[(long)blockIdx.x * CO + tid] = r;
    }
  }
}

// out[j] = sum over chunks of partial[c][j] in a fixed order (double):
// block = 64 consecutive j x SUM_GROUPS chunk groups (group q sums chunks q,
// q + SUM_GROUPS, ... with eight loads in flight), the group sums are then
// added in group order.  Sixteen groups keep ~150 k threads loading (a
// 32 x 32 layer's 9216 weights x 512 chunks is 19 MB).
constexpr int SUM_GROUPS = 16;

// chunks q, q + SUM_GROUPS, ... of one element, loads of eight chunks in flight
template <typename T>
__device__ inline double chunk_sum(const T* p, long stride, int nchunk, int q) {
  double s = 0.0;
  int c = q;
  for (; c + 7 * SUM_GROUPS < nchunk; c += 8 * SUM_GROUPS) {
    T v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = p[(long)(c + k * SUM_GROUPS) * stride];
#pragma unroll
    for (int k = 0; k < 8; ++k) s += v[k];
  }
  for (; c < nchunk; c += SUM_GROUPS) s += p[(long)c * stride];
  return s;
}

__global__ void __launch_bounds__(64 * SUM_GROUPS) sum_chunks_kernel(const float* __restrict__ partial,
                                                                     float* __restrict__ out,
                                                                     int nchunk, long n) {
  __shared__ double sh[SUM_GROUPS][64];
  const int e = threadIdx.x & 63, q = threadIdx.x >> 6;
  const long j = (long)blockIdx.x * 64 + e;
  const long jc = j < n ? j : n - 1;   // in-range address for the spare lanes
  sh[q][e] = chunk_sum(partial + jc, n, nchunk, q);
  __syncthreads();
  if (q == 0 && j < n) {
    double t = sh[0][e];
#pragma unroll
    for (int g = 1; g < SUM_GROUPS; ++g) t += sh[g][e];
    out[j] = (float)t;
  }
}

// Column sums of a [npix][C] fp32 array (bias gradient), two stages with a
// fixed summation order.  Stage 1: block b sums pixels [b*chunk, (b+1)*chunk)
// of every column; the 256 threads read rows of C floats contiguously
// (thread t: column t % C, pixel offset t / C, G = 256 / C pixel groups).
__global__ void __launch_bounds__(256) colsum_partial_kernel(const float* __restrict__ a,
                                                             double* __restrict__ partial,
                                                             long npix, int C, long chunk) {
  __shared__ double sh[256];
  const int t = threadIdx.x;
  const int G = 256 / C;
  const int c = t % C, g = t / C;
  const long p0 = (long)blockIdx.x * chunk;
  const long p1 = p0 + chunk < npix ? p0 + chunk : npix;
  double s = 0.0;
  if (g < G)
    for (long p = p0 + g; p < p1; p += G) s += a[p * C + c];
  sh[t] = s;
  __syncthreads();
  if (t < C) {
    double r = 0.0;
    for (int k = 0; k < G; ++k) r += sh[k * C + t];
    partial[(long)blockIdx.x * C + t] = r;
  }
}

// Stage 2: out[c] = sum over blocks of partial[b][c]; one block per column,
// thread t sums blocks t, t+256, ..., then a fixed-order tree
__global__ void __launch_bounds__(256) colsum_final_kernel(const double* __restrict__ partial,
                                                           float* __restrict__ out, int nblk,
                                                           int C) {
  __shared__ double sh[256];
  const int c = blockIdx.x, t = threadIdx.x;
  double s = 0.0;
  for (int b = t; b < nblk; b += 256) s += partial[(long)b * C + c];
  sh[t] = s;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if (t < k) sh[t] += sh[t + k];
    __syncthreads();
  }
  if (t == 0) out[c] = (float)sh[0];
}

// fp32 weights in (co, ci, ky, kx) order -> padded bf16 forward and transposed
// (input-gradient) weights: wf[co][t][ci] = w[co][ci][t], wt[ci][t][co] = w[co][ci][8 - t]
__global__ void wprep_kernel(const float* __restrict__ w, int Co, int Ci, int Cop, int Cip,
                             uint16_t* __restrict__ wf, uint16_t* __restrict__ wt) {
  const long j = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long n = (long)Cop * 9 * Cip;
  if (j >= n) return;
  const int ci = (int)(j % Cip);
  const int t = (int)((j / Cip) % 9);
  const int co = (int)(j / (9L * Cip));
  const float v = (co < Co && ci < Ci) ? w[((long)co * Ci + ci) * 9 + t] : 0.f;
  const uint16_t h = f2bf(v);
  if (wf) wf[j] = h;
  if (wt) wt[((long)ci * 9 + (8 - t)) * Cop + co] = h;
}

// padded weight gradient [Cop][9][Cip] -> (co, ci, ky, kx) order
__global__ void wunpack_kernel(const float* __restrict__ dwp, int Co, int Ci, int Cop, int Cip,
                               float* __restrict__ dw) {
  const long j = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long n = (long)Co * Ci * 9;
  if (j >= n) return;
  const int t = (int)(j % 9);
  const int ci = (int)((j / 9) % Ci);
  const int co = (int)(j / (9L * Ci));
  dw[j] = dwp[((long)co * 9 + t) * Cip + ci];
}

// Gather channels: dst_bf16[p][c] = scale_c * src_c[p * pstride] (0 for c >= C)
struct PackArgs {
  const void* src[DDX_CONV_MAXCH];
  float scale[DDX_CONV_MAXCH];
  long pstride;
  long npix;
  int C, Cp, f64;
  uint16_t* dst_bf16;
  float* dst_f32;
};

__global__ void pack_kernel(PackArgs a) {
  const long j = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= a.npix * a.Cp) return;
  const long p = j / a.Cp;
  const int c = (int)(j - p * a.Cp);
  float v = 0.f;
  if (c < a.C) {
    const long o = p * a.pstride;
    v = a.f64 ? (float)((const double*)a.src[c])[o] : ((const float*)a.src[c])[o];
    v *= a.scale[c];
  }
  if (a.dst_bf16) a.dst_bf16[j] = f2bf(v);
  if (a.dst_f32) a.dst_f32[j] = v;
}

// One pixel per thread (Cp % 8 == 0, 16-byte aligned outputs): the C <= CMAX
// source values are read once, unconditionally (channels past C read channel
// 0 and are zeroed), and the Cp padded channels written as 16-byte chunks.
template <bool F64, int CMAX>
__global__ void pack_pixel_kernel(PackArgs a) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= a.npix) return;
  float v[CMAX], x[CMAX];
  const long o = p * a.pstride;
#pragma unroll
  for (int c = 0; c < CMAX; ++c) {
    const int cc = c < a.C ? c : 0;
    x[c] = F64 ? (float)((const double*)a.src[cc])[o] : ((const float*)a.src[cc])[o];
  }
  // empty asm statements taking the loaded values as operands, after all the
  // loads: no load can be moved under the (uniform) channel test below, which
  // would serialise them
#pragma unroll
  for (int c = 0; c < CMAX; ++c) asm volatile("" : "+v"(x[c]));
#pragma unroll
  for (int c = 0; c < CMAX; ++c) v[c] = c < a.C ? x[c] * a.scale[c < a.C ? c : 0] : 0.f;
  for (int k = 0; k < a.Cp / 8; ++k) {
    float w[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      w[e] = 0.f;
#pragma unroll
      for (int d = 0; d < CMAX; ++d)
        if (d == 8 * k + e) w[e] = v[d];
    }
    if (a.dst_bf16) {
      uint4 q;
      q.x = (uint32_t)f2bf(w[0]) | ((uint32_t)f2bf(w[1]) << 16);
      q.y = (uint32_t)f2bf(w[2]) | ((uint32_t)f2bf(w[3]) << 16);
      q.z = (uint32_t)f2bf(w[4]) | ((uint32_t)f2bf(w[5]) << 16);
      q.w = (uint32_t)f2bf(w[6]) | ((uint32_t)f2bf(w[7]) << 16);
      *reinterpret_cast<uint4*>(&a.dst_bf16[p * a.Cp + 8 * k]) = q;
    }
    if (a.dst_f32) {
      float4* d = reinterpret_cast<float4*>(&a.dst_f32[p * a.Cp + 8 * k]);
      d[0] = make_float4(w[0], w[1], w[2], w[3]);
      d[1] = make_float4(w[4], w[5], w[6], w[7]);
    }
  }
}

// Scatter channels: dst_c[p * pstride] = scale_c * src[p][c] (c < C), fp32 or fp64
struct UnpackArgs {
  void* dst[DDX_CONV_MAXCH];
  const void* add[DDX_CONV_MAXCH];   // all null, or one per channel
  float scale[DDX_CONV_MAXCH];
  long pstride;
  long npix;
  int C, Cp, f64;
  const float* src;
};

__global__ void unpack_kernel(UnpackArgs a) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= a.npix) return;
  const long o = p * a.pstride;
  const float* __restrict__ sp = a.src + p * a.Cp;
  float v[DDX_CONV_MAXCH];
#pragma unroll
  for (int c = 0; c < DDX_CONV_MAXCH; ++c) v[c] = sp[c < a.C ? c : 0];   // loads first
#pragma unroll
  for (int c = 0; c < DDX_CONV_MAXCH; ++c) {
    if (c >= a.C) break;
    const float x = v[c] * a.scale[c];
    if (a.f64)
      ((double*)a.dst[c])[o] = (double)x + (a.add[0] ? ((const double*)a.add[c])[o] : 0.0);
    else
      ((float*)a.dst[c])[o] = x + (a.add[0] ? ((const float*)a.add[c])[o] : 0.f);
  }
}

// Box filter: dst[Y][X] = mean of the f x f block of src starting at (f Y, f X)
template <typename T>
__global__ void box_filter_kernel(const T* __restrict__ src, T* __restrict__ dst, int ny, int nx,
                                  int f) {
  const int mx = nx / f, my = ny / f;
  const long j = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= (long)mx * my) return;
  const int Y = (int)(j / mx), X = (int)(j - (long)Y * mx);
  double s = 0.0;
  for (int a = 0; a < f; ++a) {
    const T* row = src + ((long)(Y * f + a)) * nx + (long)X * f;
    for (int b = 0; b < f; ++b) s += (double)row[b];
  }
  dst[j] = (T)(s / ((double)f * f));
}

// Layout probe, K = 32 (gfx950): lane l holds A[l % 16][8 (l / 16) + i] and
// B[8 (l / 16) + i][l % 16], i < 8; D as for K = 16.

__device__ inline bf16x8 to_bf16x8(const uint16_t (&h)[8]) {
  bf16x8 r;
#pragma unroll
  for (int i = 0; i < 8; ++i) r[i] = __builtin_bit_cast(__bf16, h[i]);
  return r;
}

__global__ void __launch_bounds__(64) mfma_probe32_kernel(const uint16_t* A, const uint16_t* Bm, float* D) {
  const int lane = threadIdx.x;
  const int m = lane & 15, kq = lane >> 4;
  uint16_t ha[8], hb[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    ha[i] = A[m * 32 + 8 * kq + i];
    hb[i] = Bm[(8 * kq + i) * 16 + m];
  }
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(to_bf16x8(ha), to_bf16x8(hb), acc, 0, 0, 0);
#pragma unroll
  for (int i = 0; i < 4; ++i) D[(4 * kq + i) * 16 + m] = acc[i];
}

// Layout probe: D = A B for one 16 x 16 x 16 tile; A, B bf16 row-major, D fp32 row-major.
__global__ void __launch_bounds__(64) mfma_probe_kernel(const uint16_t* A, const uint16_t* Bm, float* D) {
  const int lane = threadIdx.x;
  const int m = lane & 15, kq = lane >> 4;
  bf16x4 a, b;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    a[i] = (short)A[m * 16 + 4 * kq + i];
    b[i] = (short)Bm[(4 * kq + i) * 16 + m];
  }
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc, 0, 0, 0);
#pragma unroll
  for (int i = 0; i < 4; ++i) D[(4 * kq + i) * 16 + m] = acc[i];
}

int check_conv(int B, int H, int W, int Ci, int Co) {
  if (B < 1 || H < 1 || W < 1) return ddx::set_error(DDX_ERR_ARG, "empty convolution");
  if (Ci < 16 || Co < 16 || Ci % 16 || Co % 16)
    return ddx::set_error(DDX_ERR_ARG, "padded channel counts must be positive multiples of 16");
  if (Co > 64) return ddx::set_error(DDX_ERR_UNSUPPORTED, "at most 64 output channels");
  if (((long)B * H * W) % 16) return ddx::set_error(DDX_ERR_ARG, "B*H*W must be a multiple of 16");
  if ((long)B * H * W * (Ci > Co ? Ci : Co) >= (1L << 40)) return ddx::set_error(DDX_ERR_ARG, "problem too large");
  return 0;
}

inline unsigned nblk(long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

// Tile width of the LDS-tiled kernels: 64 or 32 columns, 0 where they do not
// apply
int tile_cols(int H, int W, int Ci, int Co) {
  if ((Ci != 16 && Ci != 32) || (Co != 16 && Co != 32)) return 0;
  if (W % 64 == 0 && H % 4 == 0) return 64;
  if (W % 32 == 0 && H % 8 == 0) return 32;
  return 0;
}

// blocks loop over tiles; about four resident blocks per CU cover the chip
inline long conv_blocks(long ntiles) { return ntiles < 1024 ? ntiles : 1024; }

template <int CI, int CO, bool BF, bool EX>
void conv_tile_go(hipStream_t s, const ConvArgs& a, int tc) {
  const long ntiles = (long)a.B * a.H * a.W / 256;
  const dim3 grid((unsigned)conv_blocks(ntiles));
  constexpr int MINW = BF ? 3 : 2;
  if (tc != 64) {
    hipLaunchKernelGGL((conv3x3_tile_kernel<CI, CO, BF, 32, EX, MINW>), grid, dim3(256), 0, s, a, ntiles);
    return;
  }
  if constexpr (BF && CI == 32 && CO == 16) {
    // Up to two workgroups per CU the time is one tile's latency, and the
    // code for three wavefronts per SIMD reads its operands later: 8 images
    // 64^2 5.1 us without that bound, 5.6 with it; one image 512^2 (four
    // workgroups per CU) 10.3 and 9.4.
    if (ntiles <= 512) {
      hipLaunchKernelGGL((conv3x3_tile_kernel<CI, CO, BF, 64, EX, 1>), grid, dim3(256), 0, s, a, ntiles);
      return;
    }
  }
  hipLaunchKernelGGL((conv3x3_tile_kernel<CI, CO, BF, 64, EX, MINW>), grid, dim3(256), 0, s, a, ntiles);
}

template <bool BF, bool EX>
void conv_tile_ch(hipStream_t s, const ConvArgs& a, int tc) {
  switch (a.Ci * 100 + a.Co) {
    case 1616: conv_tile_go<16, 16, BF, EX>(s, a, tc); break;
    case 1632: conv_tile_go<16, 32, BF, EX>(s, a, tc); break;
    case 3216: conv_tile_go<32, 16, BF, EX>(s, a, tc); break;
    default: conv_tile_go<32, 32, BF, EX>(s, a, tc); break;
  }
}

template <bool BF>
void conv_tile(hipStream_t s, const ConvArgs& a, int tc) {
  if constexpr (BF) conv_tile_ch<true, false>(s, a, tc);
  else if (a.bpart || a.cout != a.Co) conv_tile_ch<false, true>(s, a, tc);
  else conv_tile_ch<false, false>(s, a, tc);
}

// ddx_conv3x3 with out_f32 holding cout <= Co channels per pixel
int conv_run(hipStream_t s, int B, int H, int W, int Ci, int Co, const void* x, const void* w, const float* bias,
             const float* aux, int mode, float* out_f32, void* out_bf16, int cout) {
  int rc = check_conv(B, H, W, Ci, Co);
  if (rc) return rc;
  if (!x || !w || (!out_f32 && !out_bf16)) return ddx::set_error(DDX_ERR_ARG, "null argument");
  if (mode != DDX_CONV_LINEAR && mode != DDX_CONV_GELU && mode != DDX_CONV_GELU_GRAD)
    return ddx::set_error(DDX_ERR_ARG, "unknown convolution mode");
  if (mode == DDX_CONV_GELU_GRAD && !aux)
    return ddx::set_error(DDX_ERR_ARG, "DDX_CONV_GELU_GRAD needs the pre-activation");
  ConvArgs a{(const uint16_t*)x, (const uint16_t*)w, bias, aux, out_f32, (uint16_t*)out_bf16,
             B, H, W, Ci, Co, mode, cout, nullptr};
  auto al = [](const void* q, uintptr_t n) { return ((uintptr_t)q % n) == 0; };
  const bool aligned = al(x, 16) && al(w, 16) && al(out_f32, 16) && al(aux, 16) && al(out_bf16, 8);
  const int tc = aligned ? tile_cols(H, W, Ci, Co) : 0;
  if (tc) {
    // bf16-only output without the GELU gradient stages bf16 (BF)
    if (!out_f32 && mode != DDX_CONV_GELU_GRAD) conv_tile<true>(s, a, tc);
    else conv_tile<false>(s, a, tc);
    CL_LAUNCHCHK("conv3x3 tile");
    return 0;
  }
  const long tiles = (long)B * H * W / 16;
  const dim3 grid(nblk(tiles, 4));
  switch (Co / 16) {
    case 1: hipLaunchKernelGGL(conv3x3_kernel<1>, grid, dim3(256), 0, s, a); break;
    case 2: hipLaunchKernelGGL(conv3x3_kernel<2>, grid, dim3(256), 0, s, a); break;
    case 3: hipLaunchKernelGGL(conv3x3_kernel<3>, grid, dim3(256), 0, s, a); break;
    default: hipLaunchKernelGGL(conv3x3_kernel<4>, grid, dim3(256), 0, s, a); break;
  }
  CL_LAUNCHCHK("conv3x3");
  return 0;
}

template <int CI, int CO>
void wgrad_go(hipStream_t s, int nch, int tc, const uint16_t* x, const uint16_t* dz, const float* dzf, float* partial,
              double* bpartial, int B, int H, int W) {
  if (tc == 64)
    hipLaunchKernelGGL((conv3x3_wgrad_tile_kernel<CI, CO, 64>), dim3(nch), dim3(256), 0, s, x, dz, partial, B, H, W,
                       dzf, bpartial);
  else
    hipLaunchKernelGGL((conv3x3_wgrad_tile_kernel<CI, CO, 32>), dim3(nch), dim3(256), 0, s, x, dz, partial, B, H, W,
                       dzf, bpartial);
}

// The tile kernel's partial sums (tc columns per tile); returns their number
int wgrad_tiles(hipStream_t s, int B, int H, int W, int Ci, int Co, int tc, const void* x, const void* dz,
                const float* dzf, float* partial, double* bpartial, int nchunk) {
  const long ntiles = (long)B * H * W / 256;
  const int nch = (int)(ntiles < nchunk ? ntiles : nchunk);
  const uint16_t* xx = (const uint16_t*)x;
  const uint16_t* dd = (const uint16_t*)dz;
  switch (Ci * 100 + Co) {
    case 1616: wgrad_go<16, 16>(s, nch, tc, xx, dd, dzf, partial, bpartial, B, H, W); break;
    case 1632: wgrad_go<16, 32>(s, nch, tc, xx, dd, dzf, partial, bpartial, B, H, W); break;
    case 3216: wgrad_go<32, 16>(s, nch, tc, xx, dd, dzf, partial, bpartial, B, H, W); break;
    default: wgrad_go<32, 32>(s, nch, tc, xx, dd, dzf, partial, bpartial, B, H, W); break;
  }
  return nch;
}

// ---------------------------------------------------------------------------
// Training: the forward pass that keeps what the backward pass needs, and the
// backward pass, as two native calls.  Issued layer by layer from Python, a
// step of a five-layer network was 45 launches and as many allocations, 780 us
// of host time around 300 us of kernels for 32 images 64^2; 6 launches forward
// and 11 backward take 370 us, of which the loss and autograd's own work are
// about half.
// ---------------------------------------------------------------------------
constexpr int TRAIN_L = 8;   // layers per preparing or summing launch; deeper networks take several

inline int pad16(int c) { return (c + 15) / 16 * 16; }

struct PrepLayer {
  const float* w;   // (co, ci, ky, kx)
  const float* b;
  uint16_t* wf;     // as wprep_kernel
  uint16_t* wt;
  float* bp;        // bias padded with zeros to cop
  int co, ci, cop, cip;
  int end;          // elements of the layers up to this one
};

struct PrepArgs {
  PrepLayer l[TRAIN_L];
  int nl, nw;       // nw = l[nl - 1].end
  const float* x;   // [npix][C]
  uint16_t* xb;     // [npix][16]
  long npix;        // 0: no input in this launch
  int C;
};

// bf16 of 8 of a pixel's 16 padded channels
__device__ inline uint4 pack8(const float (&v)[8]) {
  uint32_t h[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) h[k] = (uint32_t)f2bf(v[2 * k]) | ((uint32_t)f2bf(v[2 * k + 1]) << 16);
  return make_uint4(h[0], h[1], h[2], h[3]);
}

// All layers' weights and biases, and the input rounded to bf16: one thread
// per padded weight, then one per 8 channels (16 bytes) of a pixel
__global__ void __launch_bounds__(256) net_prep_kernel(PrepArgs a) {
  const long j = (long)blockIdx.x * 256 + threadIdx.x;
  if (j < a.nw) {
    int l = 0, first = 0;
    while (j >= a.l[l].end) first = a.l[l++].end;
    const PrepLayer& p = a.l[l];
    const int e = (int)j - first;
    const int ci = e % p.cip, t = (e / p.cip) % 9, co = e / (9 * p.cip);
    const bool in = co < p.co && ci < p.ci;
    const uint16_t h = f2bf(in ? p.w[((long)co * p.ci + ci) * 9 + t] : 0.f);
    p.wf[e] = h;
    p.wt[((long)ci * 9 + (8 - t)) * p.cop + co] = h;
    if (ci == 0 && t == 0) p.bp[co] = co < p.co ? p.b[co] : 0.f;
    return;
  }
  for (long i = j - a.nw; i < 2 * a.npix; i += (long)gridDim.x * 256 - a.nw) {
    const int c0 = (int)(i & 1) * 8;
    float v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = c0 + k < a.C ? a.x[(i >> 1) * a.C + c0 + k] : 0.f;
    *reinterpret_cast<uint4*>(&a.xb[i * 8]) = pack8(v);
  }
}

// The output gradient [npix][C] as bf16 [npix][16], and per block the sums of
// its channels (the last layer's bias gradient) in double
__global__ void __launch_bounds__(256) net_gpack_kernel(const float* __restrict__ g, long npix, int C,
                                                        uint16_t* __restrict__ gb, double* __restrict__ bpart) {
  __shared__ double sh[4][16];
  const int tid = threadIdx.x, c0 = (tid & 1) * 8;
  double s[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  for (long i = (long)blockIdx.x * 256 + tid; i < 2 * npix; i += (long)gridDim.x * 256) {
    float v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      v[k] = c0 + k < C ? g[(i >> 1) * C + c0 + k] : 0.f;
      s[k] += (double)v[k];
    }
    *reinterpret_cast<uint4*>(&gb[i * 8]) = pack8(v);
  }
#pragma unroll
  for (int k = 0; k < 8; ++k) {
#pragma unroll
    for (int d = 2; d < 64; d *= 2) s[k] += __shfl_xor(s[k], d);
    if ((tid & 63) < 2) sh[tid >> 6][c0 + k] = s[k];
  }
  __syncthreads();
  if (tid < 16) bpart[(long)blockIdx.x * 16 + tid] = ((sh[0][tid] + sh[1][tid]) + sh[2][tid]) + sh[3][tid];
}

struct SumLayer {
  const float* part;    // [nch][cop][9][cip]
  const double* bpart;  // [nb][cop]
  float* dw;            // (co, ci, ky, kx)
  float* db;
  int nch, nb, co, ci, cop, cip;
  int end;              // blocks of the layers up to this one; the last of a layer sums its biases
};

struct SumArgs {
  SumLayer l[TRAIN_L];
};

// Partial weight and bias gradients of several layers, added in
// sum_chunks_kernel's order; only the layer's own channels are read, and the
// weights are written in (co, ci, ky, kx) order
__global__ void __launch_bounds__(64 * SUM_GROUPS) net_sum_kernel(SumArgs a) {
  __shared__ double sh[SUM_GROUPS][64];
  const int e = threadIdx.x & 63, q = threadIdx.x >> 6;
  int l = 0, first = 0;
  while ((int)blockIdx.x >= a.l[l].end) first = a.l[l++].end;
  const SumLayer& p = a.l[l];
  const bool bias = (int)blockIdx.x == p.end - 1;
  const int n = bias ? p.co : 9 * p.ci * p.co;
  const int i = ((int)blockIdx.x - first) * 64 + e, j = bias ? e : i;
  const int jc = j < n ? j : n - 1;    // in-range address for the spare lanes
  const int ci = jc % p.ci, t = (jc / p.ci) % 9, co = jc / (9 * p.ci);
  sh[q][e] = bias ? chunk_sum(p.bpart + jc, p.cop, p.nb, q)
                  : chunk_sum(p.part + ((long)co * 9 + t) * p.cip + ci, 9L * p.cop * p.cip, p.nch, q);
  __syncthreads();
  if (q == 0 && j < n) {
    double s = sh[0][e];
#pragma unroll
    for (int g = 1; g < SUM_GROUPS; ++g) s += sh[g][e];
    if (bias) p.db[j] = (float)s;
    else p.dw[((long)co * p.ci + ci) * 9 + t] = (float)s;
  }
}

// What a forward pass leaves for the backward pass, in one buffer: the packed
// input and the activations (bf16), the pre-activations (fp32), the transposed
// weights, and behind them the forward weights and biases
struct NetSaved {
  long npix;
  int nl;
  const int* ch;
  static long up(long b) { return (b + 255) / 256 * 256; }
  long wbytes(int l) const { return up(2L * 9 * pad16(ch[l]) * pad16(ch[l + 1])); }
  long act(int l) const {
    long o = 0;
    for (int k = 0; k < l; ++k) o += up(2 * npix * pad16(ch[k]));
    return o;
  }
  long z(int l) const {
    long o = act(nl);
    for (int k = 0; k < l; ++k) o += up(4 * npix * pad16(ch[k + 1]));
    return o;
  }
  long wt(int l) const {
    long o = z(nl - 1);
    for (int k = 0; k < l; ++k) o += wbytes(k);
    return o;
  }
  long wf(int l) const { return wt(nl) + wt(l) - wt(0); }
  long bp(int l) const {
    long o = wf(nl);
    for (int k = 0; k < l; ++k) o += up(4L * pad16(ch[k + 1]));
    return o;
  }
  long bytes() const { return bp(nl); }
};

constexpr int WGRAD_CHUNKS = 512;         // as many partial weight gradients
constexpr long PART_BYTES = 128L << 20;   // partials of several layers up to this wait for one summing launch
constexpr int GPACK_BLOCKS = 512;

// Backward scratch: two bf16 gradients, an fp32 one where a layer's shape
// needs the separate column sums, partial bias and weight gradients
struct NetScratch {
  long npix;
  int B, H, W, nl;
  const int* ch;
  static long up(long b) { return NetSaved::up(b); }
  int cmax() const {
    int c = 0;
    for (int l = 1; l <= nl; ++l) c = pad16(ch[l]) > c ? pad16(ch[l]) : c;
    return c;
  }
  // tile width of the convolution that gives the gradient at layer l's output
  int dgrad_tc(int l) const { return tile_cols(H, W, pad16(ch[l + 2]), pad16(ch[l + 1])); }
  long dz(int k) const { return k * up(2 * npix * cmax()); }
  long dzf() const { return dz(2); }
  long bpart(int k) const {
    long c = 0;
    for (int l = 0; l < nl - 1; ++l) {
      if (!dgrad_tc(l) && pad16(ch[l + 1]) > c) c = pad16(ch[l + 1]);
    }
    return dzf() + up(4 * npix * c) + k * (1024L * 8 * 64);
  }
  long part() const { return bpart(TRAIN_L); }
  int nchunk() const {
    const long n = npix / 256;
    return (int)(n < 1 ? 1 : n < WGRAD_CHUNKS ? n : WGRAD_CHUNKS);
  }
  long pbytes(int l) const { return up(4L * nchunk() * 9 * pad16(ch[l]) * pad16(ch[l + 1])); }
  long part_bytes() const {
    long sum = 0, one = 0;
    for (int l = 0; l < nl; ++l) {
      sum += pbytes(l);
      one = pbytes(l) > one ? pbytes(l) : one;
    }
    return sum < PART_BYTES ? sum : one > PART_BYTES ? one : PART_BYTES;
  }
  long bytes() const { return part() + part_bytes(); }
};

int check_net(int B, int H, int W, int nl, const int* ch) {
  if (!ch || nl < 1) return ddx::set_error(DDX_ERR_ARG, "bad network");
  for (int l = 0; l <= nl; ++l)
    if (ch[l] < 1) return ddx::set_error(DDX_ERR_ARG, "bad network channels");
  if (ch[0] > DDX_CONV_MAXCH) return ddx::set_error(DDX_ERR_ARG, "at most 16 input channels");
  for (int l = 0; l < nl; ++l) {
    const int rc = check_conv(B, H, W, pad16(ch[l]), pad16(ch[l + 1]));
    if (rc) return rc;
  }
  return 0;
}

// ---------------------------------------------------------------------------
// The whole network in one launch (inference)
// ---------------------------------------------------------------------------
//
// NL layers of 3x3 periodic convolution: 16 (padded) input channels, HID
// hidden channels with GELU, 16 (padded) linear output channels.  A
// workgroup computes one TX x TY output tile of one image: it stages the
// tile's input with a halo of NL pixels in LDS, then each layer reads its
// input region from one LDS buffer and writes its output region, NL - 1 - l
// pixels of halo narrower, to the other.  Only the network's input and
// output touch HBM; the halo is recomputed by neighbouring tiles.
//
// Every layer is the same arithmetic as conv3x3_tile_kernel's (tap loop
// t = 0..8, K in the same chunks, bias then GELU, bf16 activations), with
// the MFMA operands swapped: A = weights (16 output channels x K), B = 16
// pixels' input channels, so a lane's D values are four consecutive output
// channels of one pixel (one 8-byte LDS write).
constexpr int NET_MAXL = 6;

struct NetArgs {
  const uint16_t* w[NET_MAXL];    // layer l: [Cop][9][Cip] bf16
  const float* bias[NET_MAXL];    // layer l: [Cop] fp32
  const uint16_t* x;              // [npix][16] bf16, or null: the fields below
  const double* src[DDX_CONV_MAXCH];
  float in_scale[DDX_CONV_MAXCH];
  int cin;
  float* out;                     // [npix][16] fp32, or null: the fields below
  double* dst[DDX_CONV_MAXCH];
  const double* add[DDX_CONV_MAXCH];  // all null, or one per output channel
  float out_scale[DDX_CONV_MAXCH];
  int cout;
  int B, H, W;
};

// LDS plan of one tile: buffer 0 holds the input and the outputs of layers
// 1, 3, ...; buffer 1 the outputs of layers 0, 2, ...  Pixel strides of 16 + 4
// and HID + 4 bf16 (8-byte aligned rows, consecutive pixels on distinct banks).
template <int NL, int HID, int TX, int TY>
struct NetPlan {
  static constexpr int PSI = 16 + 4, PSH = HID + 4;
  static constexpr int in_bytes() { return (TX + 2 * NL) * (TY + 2 * NL) * PSI * 2; }
  static constexpr int out_bytes(int l) {
    return (TX + 2 * (NL - 1 - l)) * (TY + 2 * (NL - 1 - l)) * PSH * 2;
  }
  static constexpr int buf_bytes(int b) {
    int m = b == 0 ? in_bytes() : 0;
    for (int l = 0; l < NL - 1; ++l)
      if ((l + 1) % 2 == b && out_bytes(l) > m) m = out_bytes(l);
    return (m + 15) / 16 * 16;
  }
  // the current layer's weights, staged as MFMA A operands (NetStage)
  static constexpr int wbuf_bytes() {
    int m = 0;
    for (int l = 0; l < NL; ++l) {
      const int ci = l == 0 ? 16 : HID, co = l == NL - 1 ? 16 : HID;
      const int b = 9 * (co / 16) * 64 * (ci == 32 ? 16 : 8);
      if (b > m) m = b;
    }
    return m;
  }
  static constexpr int lds_bytes() { return buf_bytes(0) + buf_bytes(1) + wbuf_bytes(); }
};

__device__ inline bf16x8 gld8(const uint16_t* p) {
  const uint4 v = *reinterpret_cast<const uint4*>(p);
  const u32x4 u = {v.x, v.y, v.z, v.w};
  return __builtin_bit_cast(bf16x8, u);
}

__device__ inline bf16x4 gld4(const uint16_t* p) { return load4(p); }

__device__ inline int wrapm(int i, int n) {
  const int r = i % n;
  return r < 0 ? r + n : r;
}

// A layer's weights staged through registers into LDS, and its bias.  The
// LDS copy holds the MFMA A operands in lane order: block (t, j) (tap t,
// output channels 16 j ..) is 64 consecutive chunks, chunk l = output channel
// 16 j + l % 16, input channels (l / 16) KQ .. (KQ = 8 of 32 input channels,
// 4 of 16), so a wavefront's operand read of one block is one contiguous run
// of LDS.  The workgroup's threads share the chunks: the layer is read from
// global memory once per tile, not once per wavefront.  load() runs a layer
// ahead, under the previous layer's arithmetic; the bias stays in registers
// (a lane's four output channels of each 16).
template <int CI, int CO, int NT>
struct NetStage {
  static constexpr int NCO = CO / 16, KQ = CI == 32 ? 8 : 4;
  static constexpr int NCH = 9 * NCO * 64, R = (NCH + NT - 1) / NT;
  typedef typename std::conditional<CI == 32, u32x4, u32x2>::type chunk;
  chunk c[R];
  float b[NCO][4];
  __device__ __forceinline__ void load(const uint16_t* w_l, const float* b_l) {
    // unconditional loads (threads past the last chunk repeat it; store()
    // skips them), which keeps the chunks in registers
#pragma unroll
    for (int r = 0; r < R; ++r) {
      int q = (int)threadIdx.x + r * NT;
      q = q < NCH ? q : NCH - 1;
      const int blk = q >> 6, l = q & 63;
      const int t = blk / NCO, j = blk - t * NCO;
      c[r] = *reinterpret_cast<const chunk*>(w_l + ((j * 16 + (l & 15)) * 9 + t) * CI + (l >> 4) * KQ);
    }
    const int kq = (threadIdx.x & 63) >> 4;
#pragma unroll
    for (int j = 0; j < NCO; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) b[j][i] = b_l[j * 16 + 4 * kq + i];
  }
  __device__ __forceinline__ void store(uint16_t* wl) const {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int q = (int)threadIdx.x + r * NT;
      if (q < NCH) *reinterpret_cast<chunk*>(wl + q * KQ) = c[r];
    }
  }
};

// One layer over an output region of w x h pixels (row-major, flattened into
// 16-pixel fragments; the last fragment's spare lanes repeat the last pixel
// and store nothing).  in: (w + 2) x (h + 2) pixels with stride psi;
// LAST layers write the tile's pixels to global memory.
template <int CI, int CO, bool LAST, int NT>
__device__ __forceinline__ void net_layer(const NetArgs& a, const uint16_t* wl, const float (&bv)[CO / 16][4],
                                          const uint16_t* in, int psi, uint16_t* outb, int pso,
                                          int w, int h, int b, int y0, int x0) {
  constexpr int NCO = CO / 16;
  constexpr int NW = NT / 64;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m = lane & 15, kq = lane >> 4;
  const int npx = w * h, nfrag = (npx + 15) / 16;
  const int wi = w + 2;
  const int npairs = (nfrag + 1) / 2;
  // A pair of 16-pixel fragments per step: four independent accumulation
  // chains per wave.  The steps are software-pipelined over two accumulator
  // sets: the MFMAs of one pair are issued, then the epilogue (bias, GELU,
  // bf16 stores: VALU work) of the previous pair runs while the matrix cores
  // work through them.
  auto compute = [&](int pr, f32x4 (&acc)[2][NCO], int (&pp)[2], bool (&valid)[2]) {
    int base[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      int p = (2 * pr + u) * 16 + m;
      valid[u] = p < npx;
      if (!valid[u]) p = npx - 1;
      const int r = p / w, c = p - r * w;
      pp[u] = p;
      base[u] = r * wi + c;
    }
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int j = 0; j < NCO; ++j) acc[u][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 9; ++t) {
      const int off = (t / 3) * wi + (t % 3);
      if constexpr (CI == 32) {
        bf16x8 wv[NCO];
#pragma unroll
        for (int j = 0; j < NCO; ++j) wv[j] = lds16(wl + ((t * NCO + j) * 64 + lane) * 8);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const bf16x8 xv = lds8(in + (base[u] + off) * psi + 8 * kq);
#pragma unroll
          for (int j = 0; j < NCO; ++j)
            acc[u][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[j], xv, acc[u][j], 0, 0, 0);
        }
      } else {
        bf16x4 wv[NCO];
#pragma unroll
        for (int j = 0; j < NCO; ++j) wv[j] = lds4(wl + ((t * NCO + j) * 64 + lane) * 4);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const bf16x4 xv = lds4(in + (base[u] + off) * psi + 4 * kq);
#pragma unroll
          for (int j = 0; j < NCO; ++j)
            acc[u][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(wv[j], xv, acc[u][j], 0, 0, 0);
        }
      }
    }
  };
  auto finish = [&](const f32x4 (&acc)[2][NCO], const int (&pp)[2], const bool (&valid)[2]) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (!LAST) {
        // no branch on valid[u]: a spare lane computed the clamped last pixel
        // with the same operands as the lane that owns it, so its store
        // writes the same bits to the same LDS address
#pragma unroll
        for (int j = 0; j < NCO; ++j) {
          uint32_t h2[2];
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const float v0 = gelu(acc[u][j][2 * e] + bv[j][2 * e]);
            const float v1 = gelu(acc[u][j][2 * e + 1] + bv[j][2 * e + 1]);
            h2[e] = (uint32_t)f2bf(v0) | ((uint32_t)f2bf(v1) << 16);
          }
          *reinterpret_cast<uint2*>(&outb[pp[u] * pso + j * 16 + 4 * kq]) = make_uint2(h2[0], h2[1]);
        }
      } else {
        if (!valid[u]) continue;
        const int r = pp[u] / w, c = pp[u] - r * w;
        const long gp = ((long)b * a.H + y0 + r) * a.W + x0 + c;
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = acc[u][0][i] + bv[0][i];
        if (a.out) {
          *reinterpret_cast<float4*>(&a.out[gp * 16 + 4 * kq]) = make_float4(v[0], v[1], v[2], v[3]);
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int co = 4 * kq + i;
            if (co < a.cout) {
              const float x = v[i] * a.out_scale[co];
              a.dst[co][gp] = (double)x + (a.add[0] ? a.add[co][gp] : 0.0);
            }
          }
        }
      }
    }
  };
  f32x4 accA[2][NCO], accB[2][NCO];
  int ppA[2], ppB[2];
  bool vA[2], vB[2];
  bool pendA = false, pendB = false;
  for (int pr = wave; pr < npairs;) {
    compute(pr, accA, ppA, vA);
    if (pendB) finish(accB, ppB, vB);
    pendA = true;
    pendB = false;
    pr += NW;
    if (pr >= npairs) break;
    compute(pr, accB, ppB, vB);
    finish(accA, ppA, vA);
    pendA = false;
    pendB = true;
    pr += NW;
  }
  if (pendA) finish(accA, ppA, vA);
  if (pendB) finish(accB, ppB, vB);
}

template <int L, int NL, int HID, int NT>
struct NetLayerShape {
  static constexpr int CI = L == 0 ? 16 : HID;
  static constexpr int CO = L == NL - 1 ? 16 : HID;
  typedef NetStage<CI, CO, NT> W;
};

// Layer L with its weights in LDS (wl) and its bias in cur: the next
// layer's weights are loaded into registers first, then layer L runs; after
// a barrier (every wavefront done with layer L's input and weights) the next
// weights go to LDS, and after a second one the next layer runs.
template <int L, int NL, int HID, int TX, int TY, int NT>
__device__ __forceinline__ void net_layers(const NetArgs& a, uint16_t* buf0, uint16_t* buf1, uint16_t* wl,
                                           int b, int y0, int x0,
                                           const typename NetLayerShape<L, NL, HID, NT>::W& cur) {
  using P = NetPlan<NL, HID, TX, TY>;
  using S = NetLayerShape<L, NL, HID, NT>;
  constexpr int g = NL - 1 - L;  // output halo
  const uint16_t* in = (L % 2 == 0) ? buf0 : buf1;
  uint16_t* outb = (L % 2 == 0) ? buf1 : buf0;
  if constexpr (L < NL - 1) {
    typename NetLayerShape<L + 1, NL, HID, NT>::W nxt;
    nxt.load(a.w[L + 1], a.bias[L + 1]);
    net_layer<S::CI, S::CO, false, NT>(a, wl, cur.b, in, L == 0 ? P::PSI : P::PSH, outb, P::PSH,
                                       TX + 2 * g, TY + 2 * g, b, y0, x0);
    lds_barrier();
    nxt.store(wl);
    lds_barrier();
    net_layers<L + 1, NL, HID, TX, TY, NT>(a, buf0, buf1, wl, b, y0, x0, nxt);
  } else {
    net_layer<S::CI, S::CO, true, NT>(a, wl, cur.b, in, P::PSH, outb, P::PSH, TX + 2 * g, TY + 2 * g,
                                      b, y0, x0);
  }
}

template <int NL, int HID, int TX, int TY, int NT>
__global__ void __launch_bounds__(NT) conv_net_kernel(NetArgs a) {
  using P = NetPlan<NL, HID, TX, TY>;
  extern __shared__ __align__(16) uint16_t netlds[];
  uint16_t* buf0 = netlds;
  uint16_t* buf1 = netlds + P::buf_bytes(0) / 2;
  uint16_t* wl = netlds + (P::buf_bytes(0) + P::buf_bytes(1)) / 2;
  const int tiles_x = a.W / TX, tiles_y = a.H / TY;
  int rest = blockIdx.x;
  const int tx = rest % tiles_x;
  rest /= tiles_x;
  const int ty = rest % tiles_y;
  const int b = rest / tiles_y;
  const int x0 = tx * TX, y0 = ty * TY;
  // the first layer's weights load while the input is staged
  typename NetLayerShape<0, NL, HID, NT>::W w0;
  w0.load(a.w[0], a.bias[0]);
  // stage the input region with a halo of NL pixels (periodic wrap)
  constexpr int RW = TX + 2 * NL, RH = TY + 2 * NL;
  for (int i = threadIdx.x; i < RW * RH; i += NT) {
    const int r = i / RW, c = i - r * RW;
    const int yy = wrapm(y0 - NL + r, a.H), xx = wrapm(x0 - NL + c, a.W);
    const long gp = ((long)b * a.H + yy) * a.W + xx;
    uint4 q0, q1;
    if (a.x) {
      q0 = *reinterpret_cast<const uint4*>(&a.x[gp * 16]);
      q1 = *reinterpret_cast<const uint4*>(&a.x[gp * 16 + 8]);
    } else {
      float v[16];
#pragma unroll
      for (int ch = 0; ch < 16; ++ch) {
        const int cc = ch < a.cin ? ch : 0;
        v[ch] = ch < a.cin ? (float)a.src[cc][gp] * a.in_scale[cc] : 0.f;
      }
      q0 = make_uint4((uint32_t)f2bf(v[0]) | ((uint32_t)f2bf(v[1]) << 16),
                      (uint32_t)f2bf(v[2]) | ((uint32_t)f2bf(v[3]) << 16),
                      (uint32_t)f2bf(v[4]) | ((uint32_t)f2bf(v[5]) << 16),
                      (uint32_t)f2bf(v[6]) | ((uint32_t)f2bf(v[7]) << 16));
      q1 = make_uint4((uint32_t)f2bf(v[8]) | ((uint32_t)f2bf(v[9]) << 16),
                      (uint32_t)f2bf(v[10]) | ((uint32_t)f2bf(v[11]) << 16),
                      (uint32_t)f2bf(v[12]) | ((uint32_t)f2bf(v[13]) << 16),
                      (uint32_t)f2bf(v[14]) | ((uint32_t)f2bf(v[15]) << 16));
    }
    uint2* d = reinterpret_cast<uint2*>(&buf0[i * P::PSI]);
    d[0] = make_uint2(q0.x, q0.y);
    d[1] = make_uint2(q0.z, q0.w);
    d[2] = make_uint2(q1.x, q1.y);
    d[3] = make_uint2(q1.z, q1.w);
  }
  w0.store(wl);
  lds_barrier();
  net_layers<0, NL, HID, TX, TY, NT>(a, buf0, buf1, wl, b, y0, x0, w0);
}

// Lets a kernel take this much dynamic LDS; once per device (done: a bit
// each), from any thread.
int allow_lds(const void* kernel, int bytes, std::atomic<uint64_t>& done, const char* name) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  const uint64_t bit = dev < 64 ? 1ull << dev : 0;   // beyond: set on each call
  if (e == hipSuccess && !(done.load(std::memory_order_acquire) & bit)) {
    e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e == hipSuccess) done.fetch_or(bit, std::memory_order_release);
  }
  if (e != hipSuccess) return ddx::set_error(DDX_ERR_HIP, std::string(name) + " LDS attribute: " + hipGetErrorString(e));
  return 0;
}

template <int NL, int HID, int TX, int TY, int NT>
int launch_net(const NetArgs& a, hipStream_t s) {
  using P = NetPlan<NL, HID, TX, TY>;
  constexpr int lds = P::lds_bytes();
  static_assert(lds <= 160 * 1024, "tile does not fit the LDS");
  static std::atomic<uint64_t> done{0};
  const int rc = allow_lds((const void*)conv_net_kernel<NL, HID, TX, TY, NT>, lds, done, "conv_net");
  if (rc) return rc;
  const long ntiles = (long)a.B * (a.H / TY) * (a.W / TX);
  hipLaunchKernelGGL((conv_net_kernel<NL, HID, TX, TY, NT>), dim3((unsigned)ntiles), dim3(NT), lds, s, a);
  CL_LAUNCHCHK("conv_net");
  return 0;
}

// ---------------------------------------------------------------------------
// The whole network, row by row
// ---------------------------------------------------------------------------
//
// A workgroup runs all five layers over a strip of rows of one image, full
// width W (32 or 64): at step t layer l computes row y0 - 4 + t - 3 l from
// the three rows that layer l - 1 left in a ring of four rows in LDS.
// Columns wrap inside the row, so only the strip's ends are recomputed (S + 8
// rows of layer 0 for S outputs, ..., S of layer 4), where the tile kernel's
// halo is 1.83 times the network's work.  A wavefront keeps one layer and one
// 16-pixel fragment of the row for the whole strip, and its weights in
// registers (72 for 32 x 32 channels), so LDS carries little but activations:
// group 0 takes the first and the last layer (half a layer each; the last
// one's weights are read from LDS in MFMA operand order, for which its
// registers do not suffice), group g layer g; with W = 64 each SIMD holds one
// wavefront of every group.
//
// A step issues the row's MFMAs interleaved with bias, GELU and rounding of
// the row of the step before: the matrix pipe takes 16 cycles an MFMA and
// the activations 1.5 times that in VALU cycles, and wavefronts that leave a
// barrier together do not overlap the two by themselves.  That row is
// written a step late, hence the lag of three rows per layer.  The loop is
// unrolled over the four ring positions, which makes every LDS row an
// immediate offset.
//
// What bounds it: VALU issue first, about 1700 cycles of a step's 2750 (8
// activations of 14.5 issue slots per lane and wavefront, and the addresses),
// beside 1300 of MFMAs; the barrier of each step keeps either from filling it
// (wavefronts wait 48 % of their cycles).  256 images 64^2: 213 us with the
// tile kernel, 1.83 times the network's MFMAs; row by row 150 us with two
// fragments per wavefront and 8 wavefronts per CU, 128 with one and 16, 112
// with the last layer's weights in LDS (128 registers without spills).
//
// One 16-byte chunk q (8 channels) of pixel p lies at chunk q ^ ((p >> 2) & 3)
// of the pixel's 64 bytes: the 16 pixels of a fragment lie in 16 distinct
// 16-byte bank groups, for any shift of the fragment.  The counters still
// show 3.5 conflict cycles per LDS instruction; which accesses take them is
// not measured.
//
// The arithmetic is conv_net_kernel's: the same products in the same order.
// Rows before a layer's first and after its last are computed from whatever
// the rings hold and never reach a row that is stored.
template <int W>
struct RowNet {
  static constexpr int WPG = W / 16;                   // wavefronts per group
  static constexpr int NT = 4 * WPG * 64;
  static constexpr int HROW = W * 64, IROW = W * 32;   // bytes of a row: hidden, input
  static constexpr int HB = 4 * HROW, IB = 4 * IROW;   // rings of four rows
  static constexpr int WG_PER_CU = 1024 / NT;          // 128 registers: 16 wavefronts per CU
  static constexpr int WB = 9 * 64 * 16;               // the last layer's weights
  static constexpr int lds_bytes() { return IB + 4 * HB + WB; }
};

__device__ __forceinline__ int rn_off(int p, int q) { return p * 64 + ((q ^ (p >> 2)) & 3) * 16; }
__device__ __forceinline__ int rn_ioff(int p, int h) { return p * 32 + ((h ^ (p >> 3)) & 1) * 8 + (h & 2) * 8; }

// two fp32 -> packed bf16, round to nearest even (one v_cvt_pk_bf16_f32)
__device__ __forceinline__ uint32_t f2bf2(float a, float b) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  const f32x2 v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

template <int CI, int CO>
struct RowWeights {
  static constexpr int NCO = CO / 16, KQ = CI == 32 ? 8 : 4;
  typedef typename std::conditional<CI == 32, bf16x8, bf16x4>::type frag;
  frag w[9][NCO];
  float b[NCO][4];
  __device__ __forceinline__ void load(const uint16_t* wp, const float* bp, int lane) {
    const int m = lane & 15, kq = lane >> 4;
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
      for (int j = 0; j < NCO; ++j) {
        const uint16_t* q = wp + ((j * 16 + m) * 9 + t) * CI + kq * KQ;
        if constexpr (CI == 32) w[t][j] = gld8(q);
        else w[t][j] = __builtin_bit_cast(bf16x4, *reinterpret_cast<const u32x2*>(q));
      }
#pragma unroll
    for (int j = 0; j < NCO; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) b[j][i] = bp[j * 16 + 4 * kq + i];
  }
};

// One row of a layer at this wavefront's fragment: off[dx] the LDS offset of
// the lane's operand, shifted by dx - 1, in ring slot 0; the three rows lie
// in slots S0, S0 + 1, S0 + 2 (mod 4).
template <int CI, int CO, int ROW, int S0>
__device__ __forceinline__ void rn_conv(const unsigned char* lds, const int (&off)[3], const RowWeights<CI, CO>& wt,
                                        f32x4 (&acc)[CO / 16]) {
  constexpr int NCO = CO / 16;
  constexpr int base[3] = {(S0 & 3) * ROW, ((S0 + 1) & 3) * ROW, ((S0 + 2) & 3) * ROW};
#pragma unroll
  for (int j = 0; j < NCO; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < 9; ++t) {
    const uint16_t* p = reinterpret_cast<const uint16_t*>(lds + off[t % 3] + base[t / 3]);
    if constexpr (CI == 32) {
      const bf16x8 xv = lds16(p);
#pragma unroll
      for (int j = 0; j < NCO; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wt.w[t][j], xv, acc[j], 0, 0, 0);
    } else {
      const bf16x4 xv = __builtin_bit_cast(bf16x4, *reinterpret_cast<const u32x2*>(p));
#pragma unroll
      for (int j = 0; j < NCO; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(wt.w[t][j], xv, acc[j], 0, 0, 0);
    }
  }
}

// The last layer's row, its weights from LDS (chunk t 64 + lane)
template <int ROW, int S0>
__device__ __forceinline__ void rn_conv_last(const unsigned char* lds, const int (&off)[3], const unsigned char* wl,
                                             f32x4& acc) {
  constexpr int base[3] = {(S0 & 3) * ROW, ((S0 + 1) & 3) * ROW, ((S0 + 2) & 3) * ROW};
  acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < 9; ++t) {
    const bf16x8 xv = lds16(reinterpret_cast<const uint16_t*>(lds + off[t % 3] + base[t / 3]));
    const bf16x8 wv = lds16(reinterpret_cast<const uint16_t*>(wl + t * 1024));
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv, xv, acc, 0, 0, 0);
  }
}

// Activations of a row, written to ring slot SLOT: out[j] the LDS offset of
// the lane's four channels, output channels 16 j ..
template <int CI, int ROW, int SLOT>
__device__ __forceinline__ void rn_hidden(unsigned char* lds, const int (&out)[2], const RowWeights<CI, 32>& wt,
                                          const f32x4 (&acc)[2]) {
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    float v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = gelu(acc[j][i] + wt.b[j][i]);
    *reinterpret_cast<uint2*>(lds + out[j] + (SLOT & 3) * ROW) = make_uint2(f2bf2(v[0], v[1]), f2bf2(v[2], v[3]));
  }
}

// An input row y (wrapped), 32 bytes of 16 bf16 channels per pixel: thread
// tid < 2 W of group 0 brings half tid & 1 of pixel tid >> 1
template <int W>
struct RowInput {
  uint4 q;
  __device__ __forceinline__ void load(const NetArgs& a, int b, int y, int tid) {
    if (tid >= 2 * W) return;
    const int p = tid >> 1, h = tid & 1;
    const long gp = ((long)b * a.H + wrapm(y, a.H)) * W + p;
    q = *reinterpret_cast<const uint4*>(&a.x[gp * 16 + 8 * h]);
  }
  __device__ __forceinline__ void store(unsigned char* row, int tid) const {
    if (tid >= 2 * W) return;
    const int p = tid >> 1, h = tid & 1;
    *reinterpret_cast<uint2*>(row + rn_ioff(p, 2 * h)) = make_uint2(q.x, q.y);
    *reinterpret_cast<uint2*>(row + rn_ioff(p, 2 * h + 1)) = make_uint2(q.z, q.w);
  }
};

// Instruction order of a step: operand reads four ahead of their MFMAs (an
// LDS read takes about as long as three pairs of MFMAs), and after each
// operand's MFMAs a share of the activation arithmetic
__device__ __forceinline__ void rn_interleave() {
  __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);     // LDS reads
#pragma unroll
  for (int i = 0; i < 9; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);   // MFMAs
    __builtin_amdgcn_sched_group_barrier(0x002, 7, 0);   // VALU
    if (i < 5) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
  }
}

template <int W>
__global__ void __launch_bounds__(RowNet<W>::NT, 4) conv_rows_kernel(NetArgs a, int S, int strips) {
  using P = RowNet<W>;
  constexpr int HROW = P::HROW, IROW = P::IROW;
  extern __shared__ __align__(16) unsigned char rnlds[];   // the input ring, then layers 0..3's
  const int b = blockIdx.x / strips, y0 = (blockIdx.x - b * strips) * S;
  const int rows = a.H - y0 < S ? a.H - y0 : S;
  const int tid = threadIdx.x, lane = tid & 63, m = lane & 15, kq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), group = wave / P::WPG, part = wave % P::WPG;
  int px[3];   // the lane's pixel of the fragment, shifted by -1, 0, 1
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const int c = part * 16 + m + d - 1;
    px[d] = c < 0 ? c + W : (c >= W ? c - W : c);
  }
  int out[2];  // this group's ring (group 0: layer 0's)
#pragma unroll
  for (int j = 0; j < 2; ++j) out[j] = P::IB + group * P::HB + rn_off(px[1], 2 * j + (kq >> 1)) + (kq & 1) * 8;
  const int steps = rows + 17;   // the last output row leaves a step after its MFMAs
  if (group == 0) {
    int off0[3], off4[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      off0[d] = rn_ioff(px[d], kq);
      off4[d] = P::IB + 3 * P::HB + rn_off(px[d], kq);
    }
    // group 0 also brings the input: rows y0 - 5 .. y0 - 3 before the first
    // step, then one a step, loaded a step ahead
    RowInput<W> in;
#pragma unroll 1
    for (int r = 0; r < 3; ++r) {
      in.load(a, b, y0 - 5 + r, tid);
      in.store(rnlds + r * IROW, tid);
    }
    in.load(a, b, y0 - 2, tid);
    RowWeights<16, 32> w0;
    w0.load(a.w[0], a.bias[0], lane);
    unsigned char* const wlast = rnlds + P::IB + 4 * P::HB;
    for (int i = tid; i < 9 * 64; i += P::WPG * 64) {
      const int t = i >> 6, l = i & 63;
      *reinterpret_cast<uint4*>(wlast + i * 16) =
          *reinterpret_cast<const uint4*>(a.w[4] + ((l & 15) * 9 + t) * 32 + (l >> 4) * 8);
    }
    const unsigned char* const wl = wlast + lane * 16;
    float b4[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) b4[i] = a.bias[4][4 * kq + i];
    f32x4 accA[2], accB[2], oc;
    accB[0] = accB[1] = oc = f32x4{0.f, 0.f, 0.f, 0.f};
    lds_barrier();
    auto step = [&](auto ph, int t, f32x4(&ac)[2], const f32x4(&ap)[2]) {
      constexpr int PH = decltype(ph)::value;
      in.store(rnlds + ((PH + 3) & 3) * IROW, tid);
      in.load(a, b, y0 - 1 + t, tid);
      const int r4 = y0 + t - 17;   // the output row of the step before
      if (t >= 17 && t < rows + 17) {
        const long gp = ((long)b * a.H + r4) * W + px[1];
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = oc[i] + b4[i];
        *reinterpret_cast<float4*>(&a.out[gp * 16 + 4 * kq]) = make_float4(v[0], v[1], v[2], v[3]);
      }
      __builtin_amdgcn_sched_barrier(0);
      rn_conv<16, 32, IROW, PH>(rnlds, off0, w0, ac);
      rn_hidden<16, HROW, PH + 3>(rnlds, out, w0, ap);
      rn_interleave();
      __builtin_amdgcn_sched_barrier(0);
      rn_conv_last<HROW, PH>(rnlds, off4, wl, oc);
      lds_barrier();
    };
    for (int t = 0;; t += 4) {
      step(std::integral_constant<int, 0>{}, t, accA, accB);
      if (t + 1 >= steps) break;
      step(std::integral_constant<int, 1>{}, t + 1, accB, accA);
      if (t + 2 >= steps) break;
      step(std::integral_constant<int, 2>{}, t + 2, accA, accB);
      if (t + 3 >= steps) break;
      step(std::integral_constant<int, 3>{}, t + 3, accB, accA);
      if (t + 4 >= steps) break;
    }
  } else {
    int off[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) off[d] = P::IB + (group - 1) * P::HB + rn_off(px[d], kq);
    RowWeights<32, 32> wt;
    wt.load(a.w[group], a.bias[group], lane);
    f32x4 accA[2], accB[2];
    accB[0] = accB[1] = f32x4{0.f, 0.f, 0.f, 0.f};
    lds_barrier();
    auto step = [&](auto ph, f32x4(&ac)[2], const f32x4(&ap)[2]) {
      constexpr int PH = decltype(ph)::value;
      rn_conv<32, 32, HROW, PH>(rnlds, off, wt, ac);
      rn_hidden<32, HROW, PH + 3>(rnlds, out, wt, ap);
      rn_interleave();
      lds_barrier();
    };
    for (int t = 0;; t += 4) {
      step(std::integral_constant<int, 0>{}, accA, accB);
      if (t + 1 >= steps) break;
      step(std::integral_constant<int, 1>{}, accB, accA);
      if (t + 2 >= steps) break;
      step(std::integral_constant<int, 2>{}, accA, accB);
      if (t + 3 >= steps) break;
      step(std::integral_constant<int, 3>{}, accB, accA);
      if (t + 4 >= steps) break;
    }
  }
}

template <int W>
int launch_rows(const NetArgs& a, int S, hipStream_t s) {
  using P = RowNet<W>;
  constexpr int lds = P::lds_bytes();
  static_assert(lds * P::WG_PER_CU <= 160 * 1024, "rings do not fit the LDS");
  static std::atomic<uint64_t> done{0};
  const int rc = allow_lds((const void*)conv_rows_kernel<W>, lds, done, "conv_rows");
  if (rc) return rc;
  const int strips = (a.H + S - 1) / S;
  hipLaunchKernelGGL((conv_rows_kernel<W>), dim3((unsigned)(a.B * strips)), dim3(P::NT), lds, s, a, S, strips);
  CL_LAUNCHCHK("conv_rows");
  return 0;
}

// Strip height of the row kernel for B images of H rows: the strips run in
// rounds of 256 CUs' workgroups, a strip of S rows takes S + 17 steps.
int rows_plan(int B, int H, int per_cu) {
  long best = -1;
  int S = H;
  for (int n = 1; n <= 8 && n <= H; ++n) {
    const int s = (H + n - 1) / n;
    const long wgs = (long)B * ((H + s - 1) / s);
    const long cost = ((wgs + 256L * per_cu - 1) / (256L * per_cu)) * (s + 17);
    if (best < 0 || cost < best) { best = cost; S = s; }
  }
  return S;
}

// Strip height where the network of depth 5 and width 32 runs row by row
// between packed arrays, 0 where it runs on tiles.  Both kernels' times are
// sums of rounds, fitted (in ns) to 292 shapes of 256 to 4096 tiles, 16 to 512
// rows (nine in ten within 5 %; a few strips 32 wide run faster than the
// sum): the tiles take 22.2 us for every 256, a 64-wide strip 6.6
// us to start and 1.15 a step.  Of the 32-wide ones two share a CU: a step
// takes 0.83 us alone, 1.26 where every CU holds two.  256 images 64^2 105 us
// against 184, 128 images 66 against 94; 64 images are even (47.4 and 47.0).
// Short strips in several rounds lose to the tiles: 1150 images 16 x 64 220 us
// against 203, 128 images 64 x 32 48.5 against 46.3.
// From float64 fields a step also waits for its row of inputs and addends,
// and holding them a step ahead spills: 128 images 114 us against 113 on
// tiles, 96 images 109 against 86, so fields stay on tiles.
int rows_strip(int B, int H, int W, int nl, int hid) {
  const long big = (H % 16 == 0 && W % 32 == 0) ? (long)B * (H / 16) * (W / 32) : 0;
  if (nl != 5 || hid != 32 || big < 256 || (W != 32 && W != 64)) return 0;
  const int S = rows_plan(B, H, W == 64 ? RowNet<64>::WG_PER_CU : RowNet<32>::WG_PER_CU);
  const long wgs = (long)B * ((H + S - 1) / S), steps = S + 17;
  long ns;
  if (W == 64) {
    ns = 1000 + ((wgs + 255) / 256) * (6600 + 1150 * steps);
  } else {
    const long full = wgs / 512, rest = wgs % 512;
    ns = 6000 + steps * (1260 * full + (rest == 0 ? 0 : rest <= 256 ? 830 : 830 + 460 * rest / 512));
  }
  return ns < 3000 + 22200 * ((big + 255) / 256) ? S : 0;
}

}  // namespace

extern "C" {

int ddx_conv3x3(void* stream, int B, int H, int W, int Ci, int Co, const void* x, const void* w,
                const float* bias, const float* aux, int mode, float* out_f32, void* out_bf16) {
  return conv_run((hipStream_t)stream, B, H, W, Ci, Co, x, w, bias, aux, mode, out_f32, out_bf16, Co);
}

int ddx_conv3x3_wgrad(void* stream, int B, int H, int W, int Ci, int Co, const void* x,
                      const void* dz, float* partial, int nchunk, float* dw) {
  int rc = check_conv(B, H, W, Ci, Co);
  if (rc) return rc;
  if (!x || !dz || !partial || !dw || nchunk < 1) return ddx::set_error(DDX_ERR_ARG, "null argument");
  const long npix = (long)B * H * W;
  hipStream_t s = (hipStream_t)stream;
  const long n = (long)Co * 9 * Ci;
  // the tile kernel reads both arrays 8 bytes at a time
  const int tc = ((uintptr_t)x | (uintptr_t)dz) % 8 == 0 ? tile_cols(H, W, Ci, Co) : 0;
  if (tc) {
    const int nch = wgrad_tiles(s, B, H, W, Ci, Co, tc, x, dz, nullptr, partial, nullptr, nchunk);
    CL_LAUNCHCHK("conv3x3_wgrad tile");
    hipLaunchKernelGGL(sum_chunks_kernel, dim3(nblk(n, 64)), dim3(64 * SUM_GROUPS), 0, s, partial, dw, nch, n);
    CL_LAUNCHCHK("conv3x3_wgrad sum");
    return 0;
  }
  long pch = (npix + nchunk - 1) / nchunk;
  pch = (pch + 15) / 16 * 16;
  const int nch = (int)((npix + pch - 1) / pch);  // <= nchunk
  hipLaunchKernelGGL(conv3x3_wgrad_kernel, dim3(nch, (Co / 16) * (Ci / 16)), dim3(64), 0, s,
                     (const uint16_t*)x, (const uint16_t*)dz, partial, B, H, W, Ci, Co, (int)pch);
  CL_LAUNCHCHK("conv3x3_wgrad");
  hipLaunchKernelGGL(sum_chunks_kernel, dim3(nblk(n, 64)), dim3(64 * SUM_GROUPS), 0, s, partial, dw, nch, n);
  CL_LAUNCHCHK("conv3x3_wgrad sum");
  return 0;
}

int ddx_conv3x3_grads(void* stream, int B, int H, int W, int Ci, int Co, const void* x,
                      const void* dz, const float* dzf, float* partial, double* bpartial, int nchunk,
                      float* dw, float* db) {
  int rc = check_conv(B, H, W, Ci, Co);
  if (rc) return rc;
  if (!x || !dz || !dzf || !partial || !bpartial || !dw || !db || nchunk < 1)
    return ddx::set_error(DDX_ERR_ARG, "null argument");
  if (!(W % 64 == 0 && H % 4 == 0 && (Ci == 16 || Ci == 32) && (Co == 16 || Co == 32)))
    return ddx::set_error(DDX_ERR_UNSUPPORTED,
                          "fused gradients need W % 64 == 0, H % 4 == 0 and 16 or 32 channels");
  hipStream_t s = (hipStream_t)stream;
  const int nch = wgrad_tiles(s, B, H, W, Ci, Co, 64, x, dz, dzf, partial, bpartial, nchunk);
  CL_LAUNCHCHK("conv3x3 grads");
  const long n = (long)Co * 9 * Ci;
  hipLaunchKernelGGL(sum_chunks_kernel, dim3(nblk(n, 64)), dim3(64 * SUM_GROUPS), 0, s, partial, dw, nch, n);
  CL_LAUNCHCHK("conv3x3 grads: weight sum");
  hipLaunchKernelGGL(colsum_final_kernel, dim3(Co), dim3(256), 0, s, bpartial, db, nch, Co);
  CL_LAUNCHCHK("conv3x3 grads: bias sum");
  return 0;
}

int ddx_conv_colsum(void* stream, const float* a, int64_t npix, int C, double* partial, int nchunk,
                    float* out) {
  if (!a || !out || !partial || npix < 1 || C < 1 || C > 256 || nchunk < 1)
    return ddx::set_error(DDX_ERR_ARG, "bad column-sum arguments");
  const long chunk = (npix + nchunk - 1) / nchunk;
  const int nblk = (int)((npix + chunk - 1) / chunk);  // <= nchunk
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(colsum_partial_kernel, dim3(nblk), dim3(256), 0, s, a, partial, (long)npix, C,
                     chunk);
  CL_LAUNCHCHK("conv_colsum");
  hipLaunchKernelGGL(colsum_final_kernel, dim3(C), dim3(256), 0, s, partial, out, nblk, C);
  CL_LAUNCHCHK("conv_colsum final");
  return 0;
}

int ddx_conv_wprep(void* stream, const float* w, int Co, int Ci, int Cop, int Cip, void* wf, void* wt) {
  if (!w || (!wf && !wt) || Co < 1 || Ci < 1 || Cop < Co || Cip < Ci)
    return ddx::set_error(DDX_ERR_ARG, "bad weight-prep arguments");
  const long n = (long)Cop * 9 * Cip;
  hipLaunchKernelGGL(wprep_kernel, dim3(nblk(n, 256)), dim3(256), 0, (hipStream_t)stream, w, Co, Ci,
                     Cop, Cip, (uint16_t*)wf, (uint16_t*)wt);
  CL_LAUNCHCHK("conv_wprep");
  return 0;
}

int ddx_conv_wunpack(void* stream, const float* dwp, int Co, int Ci, int Cop, int Cip, float* dw) {
  if (!dwp || !dw || Co < 1 || Ci < 1 || Cop < Co || Cip < Ci)
    return ddx::set_error(DDX_ERR_ARG, "bad weight-unpack arguments");
  const long n = (long)Co * Ci * 9;
  hipLaunchKernelGGL(wunpack_kernel, dim3(nblk(n, 256)), dim3(256), 0, (hipStream_t)stream, dwp, Co,
                     Ci, Cop, Cip, dw);
  CL_LAUNCHCHK("conv_wunpack");
  return 0;
}

int ddx_conv_pack(void* stream, int64_t npix, int C, int Cp, const void* const* src, int64_t pstride,
                  int src_f64, const float* scale, void* dst_bf16, float* dst_f32) {
  if (!src || npix < 1 || C < 1 || C > DDX_CONV_MAXCH || Cp < C || pstride < 1 || (!dst_bf16 && !dst_f32))
    return ddx::set_error(DDX_ERR_ARG, "bad pack arguments");
  PackArgs a{};
  for (int c = 0; c < C; ++c) {
    if (!src[c]) return ddx::set_error(DDX_ERR_ARG, "null channel source");
    a.src[c] = src[c];
    a.scale[c] = scale ? scale[c] : 1.0f;
  }
  a.pstride = pstride;
  a.npix = npix;
  a.C = C;
  a.Cp = Cp;
  a.f64 = src_f64 ? 1 : 0;
  a.dst_bf16 = (uint16_t*)dst_bf16;
  a.dst_f32 = dst_f32;
  const bool al = ((uintptr_t)dst_bf16 % 16) == 0 && ((uintptr_t)dst_f32 % 16) == 0;
  const dim3 pg(nblk(npix, 256));
  hipStream_t ps = (hipStream_t)stream;
  if (Cp % 8 == 0 && al) {
    if (a.f64 && C <= 4) hipLaunchKernelGGL((pack_pixel_kernel<true, 4>), pg, dim3(256), 0, ps, a);
    else if (a.f64) hipLaunchKernelGGL((pack_pixel_kernel<true, DDX_CONV_MAXCH>), pg, dim3(256), 0, ps, a);
    else if (C <= 4) hipLaunchKernelGGL((pack_pixel_kernel<false, 4>), pg, dim3(256), 0, ps, a);
    else hipLaunchKernelGGL((pack_pixel_kernel<false, DDX_CONV_MAXCH>), pg, dim3(256), 0, ps, a);
  } else
    hipLaunchKernelGGL(pack_kernel, dim3(nblk(npix * Cp, 256)), dim3(256), 0, (hipStream_t)stream, a);
  CL_LAUNCHCHK("conv_pack");
  return 0;
}

int ddx_conv_unpack(void* stream, int64_t npix, int C, int Cp, const float* src, void* const* dst,
                    int64_t pstride, int dst_f64, const float* scale, const void* const* add) {
  if (!src || !dst || npix < 1 || C < 1 || C > DDX_CONV_MAXCH || Cp < C || pstride < 1)
    return ddx::set_error(DDX_ERR_ARG, "bad unpack arguments");
  UnpackArgs a{};
  for (int c = 0; c < C; ++c) {
    if (!dst[c]) return ddx::set_error(DDX_ERR_ARG, "null channel destination");
    if (add && !add[c]) return ddx::set_error(DDX_ERR_ARG, "null channel addend");
    a.dst[c] = dst[c];
    a.add[c] = add ? add[c] : nullptr;
    a.scale[c] = scale ? scale[c] : 1.0f;
  }
  a.pstride = pstride;
  a.npix = npix;
  a.C = C;
  a.Cp = Cp;
  a.f64 = dst_f64 ? 1 : 0;
  a.src = src;
  hipLaunchKernelGGL(unpack_kernel, dim3(nblk(npix, 256)), dim3(256), 0, (hipStream_t)stream, a);
  CL_LAUNCHCHK("conv_unpack");
  return 0;
}

int ddx_box_filter(void* stream, int ny, int nx, int factor, int f64, const void* src, void* dst) {
  if (!src || !dst || ny < 1 || nx < 1 || factor < 1 || ny % factor || nx % factor)
    return ddx::set_error(DDX_ERR_ARG, "box filter: extents must be positive multiples of the factor");
  const long n = (long)(ny / factor) * (nx / factor);
  hipStream_t s = (hipStream_t)stream;
  if (f64)
    hipLaunchKernelGGL(box_filter_kernel<double>, dim3(nblk(n, 256)), dim3(256), 0, s,
                       (const double*)src, (double*)dst, ny, nx, factor);
  else
    hipLaunchKernelGGL(box_filter_kernel<float>, dim3(nblk(n, 256)), dim3(256), 0, s,
                       (const float*)src, (float*)dst, ny, nx, factor);
  CL_LAUNCHCHK("box_filter");
  return 0;
}

int ddx_conv_net(void* stream, int B, int H, int W, int nl, const int* chans,
                 const void* const* w, const float* const* bias, const void* x, float* out,
                 const void* const* src, const float* in_scale, void* const* dst,
                 const void* const* add, const float* out_scale) {
  if (B < 1 || H < 1 || W < 1) return ddx::set_error(DDX_ERR_ARG, "bad image shape");
  if (!chans || !w || !bias) return ddx::set_error(DDX_ERR_ARG, "null argument");
  if ((!x && !src) || (!out && !dst)) return ddx::set_error(DDX_ERR_ARG, "no input or no output");
  if (nl < 2 || nl > NET_MAXL) return ddx::set_error(DDX_ERR_UNSUPPORTED, "network depth");
  const int cin = chans[0], cout = chans[nl], hid = chans[1];
  if (cin < 1 || cin > 16 || cout < 1 || cout > 16)
    return ddx::set_error(DDX_ERR_UNSUPPORTED, "network input and output need <= 16 channels");
  for (int l = 1; l < nl; ++l)
    if (chans[l] != hid) return ddx::set_error(DDX_ERR_UNSUPPORTED, "hidden layers of one width");
  NetArgs a;
  memset(&a, 0, sizeof(a));
  for (int l = 0; l < nl; ++l) {
    if (!w[l] || !bias[l]) return ddx::set_error(DDX_ERR_ARG, "null weights or bias");
    if ((uintptr_t)w[l] % 16) return ddx::set_error(DDX_ERR_ARG, "weights must be 16-byte aligned");
    a.w[l] = (const uint16_t*)w[l];
    a.bias[l] = bias[l];
  }
  if (x && (uintptr_t)x % 16) return ddx::set_error(DDX_ERR_ARG, "x must be 16-byte aligned");
  if (out && (uintptr_t)out % 16) return ddx::set_error(DDX_ERR_ARG, "out must be 16-byte aligned");
  a.x = (const uint16_t*)x;
  a.out = out;
  a.cin = cin;
  a.cout = cout;
  if (!x) {
    for (int c = 0; c < cin; ++c) {
      if (!src[c]) return ddx::set_error(DDX_ERR_ARG, "null input field");
      a.src[c] = (const double*)src[c];
      a.in_scale[c] = in_scale ? in_scale[c] : 1.f;
    }
  }
  if (!out) {
    for (int c = 0; c < cout; ++c) {
      if (!dst[c] || (add && !add[c])) return ddx::set_error(DDX_ERR_ARG, "null output field");
      a.dst[c] = (double*)dst[c];
      a.add[c] = add ? (const double*)add[c] : nullptr;
      a.out_scale[c] = out_scale ? out_scale[c] : 1.f;
    }
  }
  a.B = B;
  a.H = H;
  a.W = W;
  hipStream_t s = (hipStream_t)stream;
  // large tiles (less recomputed halo) when they alone fill the chip, small
  // tiles (more workgroups) for a few images
  const long big = (H % 16 == 0 && W % 32 == 0) ? (long)B * (H / 16) * (W / 32) : 0;
  const bool small_ok = H % 8 == 0 && W % 16 == 0;
  if (nl == 5 && hid == 32) {
    if (x && out) {
      const int S = rows_strip(B, H, W, nl, hid);
      if (S) return W == 64 ? launch_rows<64>(a, S, s) : launch_rows<32>(a, S, s);
    }
    if (big >= 256 || (big > 0 && !small_ok)) return launch_net<5, 32, 32, 16, 768>(a, s);
    // a few images: small tiles, whose layers are a few short dependent
    // phases each (one 64^2 image, a single coarse run: 4 x 4 tiles, one
    // per CU, 9.4 us per pass against 10.0 us with 8 x 8 tiles, though the
    // executed MFMA work grows from 3.0x to 5.5x the network's: the pass
    // is a chain of latencies, not of arithmetic)
    if ((long)B * (H / 4) * (W / 4) <= 256 && H % 4 == 0 && W % 4 == 0)
      return launch_net<5, 32, 4, 4, 256>(a, s);
    // then 8 x 8 tiles: each layer's region at most one fragment pair per
    // wavefront, so the five layers are five short phases rather than rounds
    // of pairs
    const long small = small_ok ? (long)B * (H / 8) * (W / 16) : 0;
    if (small < 128 && H % 8 == 0 && W % 8 == 0) return launch_net<5, 32, 8, 8, 512>(a, s);
    if (small_ok) return launch_net<5, 32, 16, 8, 256>(a, s);
  } else if (nl == 3 && hid == 16) {
    if (big >= 256 || (big > 0 && !small_ok)) return launch_net<3, 16, 32, 16, 256>(a, s);
    if (small_ok) return launch_net<3, 16, 16, 8, 256>(a, s);
  }
  return ddx::set_error(DDX_ERR_UNSUPPORTED,
                        "fused network: depth 5 width 32 on images of multiples of 8 x 8 "
                        "pixels, or depth 3 width 16 on multiples of 8 x 16");
}

int ddx_conv_net_rows(int B, int H, int W, int nl, const int* chans) {
  if (B < 1 || H < 1 || W < 1 || nl < 2 || nl > NET_MAXL || !chans) return 0;
  for (int l = 2; l < nl; ++l)
    if (chans[l] != chans[1]) return 0;
  return rows_strip(B, H, W, nl, chans[1]);
}

int ddx_net_bytes(int B, int H, int W, int nl, const int* chans, int64_t* saved, int64_t* scratch) {
  int rc = check_net(B, H, W, nl, chans);
  if (rc) return rc;
  if (!saved || !scratch) return ddx::set_error(DDX_ERR_ARG, "null argument");
  const long npix = (long)B * H * W;
  *saved = NetSaved{npix, nl, chans}.bytes();
  *scratch = NetScratch{npix, B, H, W, nl, chans}.bytes();
  return 0;
}

int ddx_net_forward(void* stream, int B, int H, int W, int nl, const int* chans, const float* x,
                    const float* const* w, const float* const* bias, void* saved, float* out) {
  int rc = check_net(B, H, W, nl, chans);
  if (rc) return rc;
  if (!x || !w || !bias || !saved || !out) return ddx::set_error(DDX_ERR_ARG, "null argument");
  if ((uintptr_t)saved % 16) return ddx::set_error(DDX_ERR_ARG, "the saved buffer must be 16-byte aligned");
  for (int l = 0; l < nl; ++l)
    if (!w[l] || !bias[l]) return ddx::set_error(DDX_ERR_ARG, "null argument");
  hipStream_t s = (hipStream_t)stream;
  const long npix = (long)B * H * W;
  const NetSaved m{npix, nl, chans};
  char* base = (char*)saved;
  auto act = [&](int l) { return (uint16_t*)(base + m.act(l)); };
  for (int l0 = 0; l0 < nl; l0 += TRAIN_L) {
    PrepArgs a{};
    a.nl = nl - l0 < TRAIN_L ? nl - l0 : TRAIN_L;
    for (int k = 0; k < a.nl; ++k) {
      const int l = l0 + k, co = chans[l + 1], ci = chans[l];
      a.nw += 9 * pad16(ci) * pad16(co);
      a.l[k] = PrepLayer{w[l], bias[l], (uint16_t*)(base + m.wf(l)), (uint16_t*)(base + m.wt(l)),
                         (float*)(base + m.bp(l)), co, ci, pad16(co), pad16(ci), a.nw};
    }
    if (l0 == 0) {
      a.x = x;
      a.xb = act(0);
      a.npix = npix;
      a.C = chans[0];
    }
    const long items = 2 * a.npix < (1L << 28) ? 2 * a.npix : 1L << 28;   // a loop covers more
    hipLaunchKernelGGL(net_prep_kernel, dim3(nblk(a.nw + items, 256)), dim3(256), 0, s, a);
    CL_LAUNCHCHK("net_forward: prepare");
  }
  for (int l = 0; l < nl; ++l) {
    const bool last = l == nl - 1;
    rc = conv_run(s, B, H, W, pad16(chans[l]), pad16(chans[l + 1]), act(l), base + m.wf(l),
                  (const float*)(base + m.bp(l)), nullptr, last ? DDX_CONV_LINEAR : DDX_CONV_GELU,
                  last ? out : (float*)(base + m.z(l)), last ? nullptr : act(l + 1),
                  last ? chans[nl] : pad16(chans[l + 1]));
    if (rc) return rc;
  }
  return 0;
}

int ddx_net_backward(void* stream, int B, int H, int W, int nl, const int* chans, const float* g,
                     const void* saved, void* scratch, float* const* dw, float* const* db) {
  int rc = check_net(B, H, W, nl, chans);
  if (rc) return rc;
  if (!g || !saved || !scratch || !dw || !db) return ddx::set_error(DDX_ERR_ARG, "null argument");
  if (chans[nl] > DDX_CONV_MAXCH) return ddx::set_error(DDX_ERR_ARG, "at most 16 output channels");
  if ((uintptr_t)saved % 16 || (uintptr_t)scratch % 16)
    return ddx::set_error(DDX_ERR_ARG, "the saved and scratch buffers must be 16-byte aligned");
  for (int l = 0; l < nl; ++l)
    if (!dw[l] || !db[l]) return ddx::set_error(DDX_ERR_ARG, "null argument");
  hipStream_t s = (hipStream_t)stream;
  const long npix = (long)B * H * W;
  const NetSaved m{npix, nl, chans};
  const NetScratch t{npix, B, H, W, nl, chans};
  const char* base = (const char*)saved;
  char* sc = (char*)scratch;
  SumArgs sums{};
  int ns = 0;
  long used = 0;
  uint16_t* dz = (uint16_t*)(sc + t.dz(0));
  // nb partial column sums of layer l's output gradient, in bpart slot ns
  const long gb = (2 * npix + 255) / 256;
  int nb = (int)(gb < GPACK_BLOCKS ? gb : GPACK_BLOCKS);
  hipLaunchKernelGGL(net_gpack_kernel, dim3(nb), dim3(256), 0, s, g, npix, chans[nl], dz, (double*)(sc + t.bpart(0)));
  CL_LAUNCHCHK("net_backward: pack");
  for (int l = nl - 1; l >= 0; --l) {
    const int cip = pad16(chans[l]), cop = pad16(chans[l + 1]);
    const uint16_t* x = (const uint16_t*)(base + m.act(l));
    float* part = (float*)(sc + t.part() + used);
    int nch = t.nchunk();
    const int tc = tile_cols(H, W, cip, cop);
    if (tc) {
      nch = wgrad_tiles(s, B, H, W, cip, cop, tc, x, dz, nullptr, part, nullptr, nch);
    } else {
      long pch = (npix + nch - 1) / nch;
      pch = (pch + 15) / 16 * 16;
      nch = (int)((npix + pch - 1) / pch);
      hipLaunchKernelGGL(conv3x3_wgrad_kernel, dim3(nch, (cop / 16) * (cip / 16)), dim3(64), 0, s, x, dz, part, B, H, W,
                         cip, cop, (int)pch);
    }
    CL_LAUNCHCHK("net_backward: weight gradient");
    const int blocks = (int)nblk(9L * chans[l] * chans[l + 1], 64) + 1;
    sums.l[ns] = SumLayer{part, (const double*)(sc + t.bpart(ns)), dw[l], db[l], nch, nb, chans[l + 1], chans[l],
                          cop, cip, (ns ? sums.l[ns - 1].end : 0) + blocks};
    ++ns;
    used += t.pbytes(l);
    if (l == 0 || ns == TRAIN_L || used + t.pbytes(l - 1) > t.part_bytes()) {
      hipLaunchKernelGGL(net_sum_kernel, dim3(sums.l[ns - 1].end), dim3(64 * SUM_GROUPS), 0, s, sums);
      CL_LAUNCHCHK("net_backward: sums");
      ns = 0;
      used = 0;
    }
    if (l == 0) break;
    // the gradient at layer l - 1's output
    uint16_t* dn = (uint16_t*)(sc + t.dz((nl - l) & 1));
    const float* z = (const float*)(base + m.z(l - 1));
    const int dtc = t.dgrad_tc(l - 1);
    if (dtc) {
      const ConvArgs a{dz, (const uint16_t*)(base + m.wt(l)), nullptr, z, nullptr, dn, B, H, W, cop, cip,
                       DDX_CONV_GELU_GRAD, cip, (double*)(sc + t.bpart(ns))};
      conv_tile<false>(s, a, dtc);
      CL_LAUNCHCHK("net_backward: input gradient");
      nb = (int)conv_blocks(npix / 256);
    } else {
      float* dzf = (float*)(sc + t.dzf());
      double* bp = (double*)(sc + t.bpart(ns));
      rc = conv_run(s, B, H, W, cop, cip, dz, base + m.wt(l), nullptr, z, DDX_CONV_GELU_GRAD, dzf, dn, cip);
      if (rc) return rc;
      const long nc = npix / 1024 < 1 ? 1 : npix / 1024 < 1024 ? npix / 1024 : 1024;
      const long chunk = (npix + nc - 1) / nc;
      const int nblocks = (int)((npix + chunk - 1) / chunk);
      hipLaunchKernelGGL(colsum_partial_kernel, dim3(nblocks), dim3(256), 0, s, dzf, bp, npix, cip, chunk);
      CL_LAUNCHCHK("net_backward: column sums");
      nb = nblocks;
    }
    dz = dn;
  }
  return 0;
}

int ddx_mfma_probe(void* stream, int k, const void* A, const void* Bm, float* D) {
  if (!A || !Bm || !D) return ddx::set_error(DDX_ERR_ARG, "null argument");
  if (k != 16 && k != 32) return ddx::set_error(DDX_ERR_ARG, "probe K must be 16 or 32");
  if (k == 16)
    hipLaunchKernelGGL(mfma_probe_kernel, dim3(1), dim3(64), 0, (hipStream_t)stream,
                       (const uint16_t*)A, (const uint16_t*)Bm, D);
  else
    hipLaunchKernelGGL(mfma_probe32_kernel, dim3(1), dim3(64), 0, (hipStream_t)stream,
                       (const uint16_t*)A, (const uint16_t*)Bm, D);
  CL_LAUNCHCHK("mfma_probe");
  return 0;
}

}  // extern "C"
