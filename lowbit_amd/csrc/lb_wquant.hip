// Weight quantizers on the device: fp32 [N, K] row-major in HBM -> the public packed
// int4 (groups of 128, or 32) and MXFP4 formats, byte for byte what the host packers produce
// (src/lowbit/formats.py:90-142 and :182-212). A model's weights are uploaded once as
// fp32 and packed where they will be read, instead of on the host.
//
// Packed layouts (src/lowbit/csrc/lowbit.h:9-19): inside each block (128 int4 codes,
// 32 E2M1 codes) byte j holds element j in its low nibble and element j + block/2 in
// its high nibble; K is padded to a whole block and padded elements get the code that
// decodes to 0.
//
// Bit-exactness: every division is IEEE float32 (the build keeps fp32 division
// correctly rounded and denormals), rint is round-half-to-even, and reductions are
// max / min / first-index selections, which do not depend on the order of combining.
#include <math.h>

#include <type_traits>

#include "lb_device.h"
#include "lb_internal.h"

namespace lbk {

// Both kernels stream: a lane holds four consecutive elements of each half of its group (or
// MX block), two 16-byte loads and one 4-byte store of packed bytes, and the reductions cross
// the group's lanes by DPP within a row of 16. (With two elements per lane, 4-byte loads,
// 1-byte stores and a permute per reduction step, int4 asym 4096 x 11008 took 88.6 us and
// MXFP4 121.8; now 45.3 and 40.1, against 41 us for the bytes at a large copy's rate.)
// Rows that are not 16-byte aligned (VEC false: K % 4, or the pointers) take the same loads
// at any float's address, element by element only where the row ends inside one, and store
// bytes only where qw itself is not aligned (each element loaded and each byte stored by
// itself, int4 groups of 32 at 4096 x 1001 took 9.3 us, and 7.6 before the lanes held four
// elements; now 5.1).
constexpr int kQT = 256;  // 4 waves per workgroup
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));

template <bool VEC>
__device__ __forceinline__ void load4(const float *wr, int k, int K, bool live, float (&x)[4]) {
  if constexpr (VEC) {
    const float4 t = live && k < K ? *reinterpret_cast<const float4 *>(wr + k) : make_float4(0.f, 0.f, 0.f, 0.f);
    x[0] = t.x, x[1] = t.y, x[2] = t.z, x[3] = t.w;
  } else if (live && k + 4 <= K) {
    const f4u t = *reinterpret_cast<const f4u *>(wr + k);
#pragma unroll
    for (int i = 0; i < 4; i++) x[i] = t[i];
  } else {
#pragma unroll
    for (int i = 0; i < 4; i++) x[i] = live && k + i < K ? wr[k + i] : 0.0f;
  }
}
template <bool VEC>
__device__ __forceinline__ void store4(uint8_t *qw, size_t off, uint32_t v) {  // off % 4 == 0
  uint8_t *dst = qw + off;
  if (VEC || reinterpret_cast<uintptr_t>(qw) % 4 == 0) {
    *reinterpret_cast<uint32_t *>(dst) = v;
  } else {
#pragma unroll
    for (int i = 0; i < 4; i++) dst[i] = (uint8_t)(v >> (8 * i));
  }
}
// f(ctrl) for each DPP step of a reduction over the L = 4 or 16 lanes of a group
template <int L, typename F>
__device__ __forceinline__ void over_lanes(F f) {
  f(std::integral_constant<int, kDppQuad1032>{});
  f(std::integral_constant<int, kDppQuad2301>{});
  if constexpr (L == 16) {
    f(std::integral_constant<int, kDppRowHalfMirror>{});
    f(std::integral_constant<int, kDppRowMirror>{});
  }
}

// int4, groups of GS = 128 or 32 elements: L = GS / 8 lanes per group, 64 / L groups
// per wave; lane j of a group holds elements 4 j .. 4 j + 3 and the same + GS / 2, exactly
// the nibbles of packed bytes 4 j .. 4 j + 3 of the group (the "j / j+half" layout).
//   absmax:     s = max|w| / 7,          q = clip(rint(w / s), -8, 7) + 8
//   signed-max: s = m / -8 (m = the first element of largest magnitude, sign kept)
//   asym:       s = (max(w, 0) - min(w, 0)) / 15, z = clip(rint(-min / s), 0, 15),
//               q = clip(rint(w / s) + z, 0, 15)
// A scale that is not > 0 (absmax, asym) or is 0 (signed-max) becomes 1.
template <int MODE, int GS, bool VEC>  // MODE 0 absmax, 1 signed-max, 2 asym
__global__ __launch_bounds__(kQT) void quantize_int4_kernel(const float *__restrict__ w, int N, int K, int G,
                                                             uint8_t *__restrict__ qw, float *__restrict__ scales,
                                                             uint8_t *__restrict__ zeros) {
  constexpr int L = GS / 8, GPW = kWave / L;
  const int lane = threadIdx.x & (kWave - 1);
  const int GQ = (G + GPW - 1) / GPW;  // wave items per row
  const long long item = (long long)blockIdx.x * (kQT / kWave) + threadIdx.x / kWave;
  if (item >= (long long)N * GQ) return;  // whole waves only: no barrier below
  const int row = (int)(item / GQ), g = (int)(item % GQ) * GPW + lane / L, j = lane % L;
  const bool live = g < G;  // the last item of a row may hold groups past the row
  const int k0 = g * GS + 4 * j;
  const float *wr = w + (size_t)row * K;
  float x[2][4];
  load4<VEC>(wr, k0, K, live, x[0]);
  load4<VEC>(wr, k0 + GS / 2, K, live, x[1]);
  float s, zf = 8.0f, lo_q = -8.0f, hi_q = 7.0f;
  if (MODE == 2) {
    float hi = 0.0f, lo = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; i++) hi = fmaxf(hi, x[i >> 2][i & 3]), lo = fminf(lo, x[i >> 2][i & 3]);
    over_lanes<L>([&](auto c) { hi = fmaxf(hi, dpp_f<c()>(hi, 0.0f)), lo = fminf(lo, dpp_f<c()>(lo, 0.0f)); });
    s = (hi - lo) / 15.0f;
    s = s > 0.0f ? s : 1.0f;
    zf = fminf(fmaxf(__builtin_rintf(-lo / s), 0.0f), 15.0f);
    lo_q = 0.0f;
    hi_q = 15.0f;
  } else if (MODE == 1) {
    // first element of largest magnitude: larger |x|, then the smaller index
    float m = x[0][0], a = fabsf(m);
    int ix = k0;
#pragma unroll
    for (int i = 1; i < 8; i++) {
      const float v = x[i >> 2][i & 3];
      if (fabsf(v) > a) a = fabsf(v), m = v, ix = k0 + (i >> 2) * (GS / 2) + (i & 3);
    }
    over_lanes<L>([&](auto c) {
      const float om = dpp_f<c()>(m, 0.0f);
      const int oi = dpp_i<c()>(ix, 0);
      if (fabsf(om) > a || (fabsf(om) == a && oi < ix)) a = fabsf(om), m = om, ix = oi;
    });
    s = m / -8.0f;
    s = s != 0.0f ? s : 1.0f;
  } else {
    float a = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; i++) a = fmaxf(a, fabsf(x[i >> 2][i & 3]));
    over_lanes<L>([&](auto c) { a = fmaxf(a, dpp_f<c()>(a, 0.0f)); });
    s = a / 7.0f;
    s = s > 0.0f ? s : 1.0f;
  }
  // symmetric: code = clip(rint(w / s), -8, 7) + 8; asym: clip(rint(w / s) + z, 0, 15)
  const float add = MODE == 2 ? zf : 0.0f, off = MODE == 2 ? 0.0f : 8.0f;
  const uint32_t pad = (uint32_t)zf;  // padded elements, read as 0, decode to 0
  uint32_t bytes = 0;
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const float c = fminf(fmaxf(__builtin_rintf(x[i >> 2][i & 3] / s) + add, lo_q), hi_q) + off;
    bytes |= (uint32_t)c << (8 * (i & 3) + 4 * (i >> 2));
  }
  if (!live) return;
  store4<VEC>(qw, (size_t)row * ((size_t)G * (GS / 2)) + (size_t)g * (GS / 2) + 4 * j, bytes);
  if (j == 0) {
    scales[(size_t)row * G + g] = s;
    if (MODE == 2) zeros[(size_t)row * G + g] = (uint8_t)pad;
  }
}

// E2M1 code of v (already divided by the block scale): round to nearest, ties to the
// even mantissa code, saturating at +-6; the magnitude code counts the decision
// points below |v| (ties at .25, 1.25, 2.5, 5 round down, at .75, 1.75, 3.5 up).
// -0 and values that round to 0 give code 0.
__device__ __forceinline__ uint32_t e2m1_code(float v) {
  const float a = fabsf(v);
  const uint32_t mag = (uint32_t)(a > 0.25f) + (uint32_t)(a >= 0.75f) + (uint32_t)(a > 1.25f) +
                       (uint32_t)(a >= 1.75f) + (uint32_t)(a > 2.5f) + (uint32_t)(a >= 3.5f) + (uint32_t)(a > 5.0f);
  return mag | ((signbit(v) && mag) ? 8u : 0u);
}

// MXFP4: one wave per 512 elements of a row = 16 blocks of 32; lanes 4b .. 4b + 3 own block
// b, lane j holding elements 4 j .. 4 j + 3 and the same + 16, the nibbles of packed bytes
// 4 j .. 4 j + 3. Shared exponent (OCP MX v1.0): e = floor(log2(amax))
// - 2 + 127 clipped to [0, 254] (127 for an all-zero block), scale 2^(e - 127).
// log2 is the float32 log2 correctly rounded (double log2, rounded once to float32):
// just below a power of two it rounds up to the integer, and the host packer's
// float32 log2 does the same there (the only place where the floor can differ). That takes
// an amax within 2^-17 ln 2 (half an ulp of the largest log2) of the power of two,
// relatively; elsewhere the floor is the exponent field, and the double log2 is not taken.
template <bool VEC>
__global__ __launch_bounds__(kQT) void quantize_mxfp4_kernel(const float *__restrict__ w, int N, int K, int Kp,
                                                              int C, uint8_t *__restrict__ qw,
                                                              uint8_t *__restrict__ e8m0) {
  const int lane = threadIdx.x & (kWave - 1);
  const long long item = (long long)blockIdx.x * (kQT / kWave) + threadIdx.x / kWave;
  if (item >= (long long)N * C) return;
  const int row = (int)(item / C), chunk = (int)(item % C);
  const int blk = chunk * 16 + (lane >> 2), j = lane & 3;  // block index in the row
  const bool live = blk * 32 < Kp;
  const int k0 = blk * 32 + 4 * j;
  const float *wr = w + (size_t)row * K;
  float x[2][4];
  load4<VEC>(wr, k0, K, live, x[0]);
  load4<VEC>(wr, k0 + 16, K, live, x[1]);
  float a = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; i++) a = fmaxf(a, fabsf(x[i >> 2][i & 3]));
  over_lanes<4>([&](auto c) { a = fmaxf(a, dpp_f<c()>(a, 0.0f)); });
  int e = 127;
  const uint32_t ab = __float_as_uint(a);
  if (a > 0.0f) {
    int sh = (int)(ab >> 23) - 2;
    // the top 2^-15 of a binade (four times what can round up), subnormals, infinity
    if ((ab & 0x7FFFFFu) >= 0x7FFF00u || ab < 0x800000u || ab >= 0x7F800000u)
      sh = (int)floorf((float)log2((double)a)) - 2 + 127;
    e = sh < 0 ? 0 : (sh > 254 ? 254 : sh);
  }
  if (!live) return;
  // x / 2^(e - 127) as the product with the exact inverse: the same real value, rounded once
  const float inv = e == 254 ? 0x1p-127f : __uint_as_float((uint32_t)(254 - e) << 23);
  uint32_t bytes = 0;
#pragma unroll
  for (int i = 0; i < 8; i++) bytes |= e2m1_code(x[i >> 2][i & 3] * inv) << (8 * (i & 3) + 4 * (i >> 2));
  const int nb = Kp / 32;
  store4<VEC>(qw, (size_t)row * (Kp / 2) + blk * 16 + 4 * j, bytes);
  if (j == 0) e8m0[(size_t)row * nb + blk] = (uint8_t)e;
}

// 16-byte loads and 4-byte stores stay inside rows and aligned
static bool vector_rows(const float *w, int K, const uint8_t *qw) {
  return K % 4 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0 && reinterpret_cast<uintptr_t>(qw) % 4 == 0;
}

static unsigned waves_grid(long long items) { return (unsigned)((items + kQT / kWave - 1) / (kQT / kWave)); }

template <int GS, bool VEC>
static void launch_quantize_int4_g(const float *w, int N, int K, int mode, uint8_t *qw, float *scales, uint8_t *zeros,
                                   hipStream_t s) {
  const int G = (K + GS - 1) / GS, GPW = kWave / (GS / 8);
  const dim3 grid(waves_grid((long long)N * ((G + GPW - 1) / GPW))), block(kQT);
  if (mode == 2)
    hipLaunchKernelGGL((quantize_int4_kernel<2, GS, VEC>), grid, block, 0, s, w, N, K, G, qw, scales, zeros);
  else if (mode == 1)
    hipLaunchKernelGGL((quantize_int4_kernel<1, GS, VEC>), grid, block, 0, s, w, N, K, G, qw, scales, zeros);
  else
    hipLaunchKernelGGL((quantize_int4_kernel<0, GS, VEC>), grid, block, 0, s, w, N, K, G, qw, scales, zeros);
}

hipError_t launch_quantize_int4(const float *w, int N, int K, int mode, int group, uint8_t *qw, float *scales,
                                uint8_t *zeros, hipStream_t s) {
  if (group != 128 && group != 32) return hipErrorInvalidValue;
  const bool vec = vector_rows(w, K, qw);
  const auto go = group == 128 ? (vec ? launch_quantize_int4_g<128, true> : launch_quantize_int4_g<128, false>)
                               : (vec ? launch_quantize_int4_g<32, true> : launch_quantize_int4_g<32, false>);
  go(w, N, K, mode, qw, scales, zeros, s);
  return hipGetLastError();
}

hipError_t launch_quantize_mxfp4(const float *w, int N, int K, uint8_t *qw, uint8_t *e8m0, hipStream_t s) {
  const int Kp = (K + 31) / 32 * 32, C = (Kp + 511) / 512;
  const dim3 grid(waves_grid((long long)N * C)), block(kQT);
  if (vector_rows(w, K, qw))
    hipLaunchKernelGGL(quantize_mxfp4_kernel<true>, grid, block, 0, s, w, N, K, Kp, C, qw, e8m0);
  else
    hipLaunchKernelGGL(quantize_mxfp4_kernel<false>, grid, block, 0, s, w, N, K, Kp, C, qw, e8m0);
  return hipGetLastError();
}

}  // namespace lbk
