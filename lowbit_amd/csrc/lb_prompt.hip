// Prompt GEMMs (many activation rows) on the matrix cores: Y[M,N] = X[M,Kp] . W[N,Kp]^T
// with the weights in the t16 tile layout and the activations in the operand tiles that
// the quantizer and the split kernels write (lb_kernels.hip).
//
// The batch kernels of lb_kernels.hip hold a few row blocks in registers and stream the
// weights past them, every weight tile ending in a reduction over the workgroup's waves;
// with hundreds of rows that reads and decodes the weights once per 16-64 rows and
// reduces far too often. Here a workgroup owns a tile of 16 TM rows x 16 WN NW columns
// of Y and walks K group by group:
//   * activations: the stage of the next group goes straight to LDS (buffer loads with
//     the LDS flag, no registers) while the current one is consumed from the other
//     buffer; the tiles are in operand order, so every LDS access is a conflict-free
//     16-byte read of 64 consecutive lanes. One barrier a group.
//   * weights: each wave owns WN 16-row subtiles and loads their tiles, scales and
//     zero-points for the next group into registers; they are decoded once per TM row
//     blocks and never pass through LDS.
//   * sums stay in the wave's registers for all of K: no reduction, no second pass.
#include <algorithm>
#include <cmath>

#include "lb_device.h"
#include "lb_internal.h"

namespace lbk {

constexpr int kPWaves = 4, kPThreads = kPWaves * kWave;

// A stage's two buffers are separate objects (not one array indexed by parity), so that
// the compiler sees that reads of one do not depend on the loads still filling the other.
__device__ __forceinline__ void lds_load16(Rsrc r, char *dst, uint32_t voff, uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void *)dst, 16, (int)voff, (int)soff,
                                           0, 0);
}
__device__ __forceinline__ void lds_load4(Rsrc r, char *dst, uint32_t voff, uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void *)dst, 4, (int)voff, (int)soff, 0,
                                           0);
}

// This wave's loads but the last LATER have arrived, those to LDS too (which a barrier
// alone does not wait for), and every wave is done with the stage before. Loads retire in
// order, and every wave issues the same number a group, so LATER = the loads of the groups
// after the one about to run.
template <int LATER>
__device__ __forceinline__ void stage_ready() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LATER) : "memory");
  __syncthreads();
}

template <typename Kern>
static hipError_t launch_prompt(Kern kern, const GemmArgs &a, PromptTile t, hipStream_t s) {
  const int mt = (a.M + 16 * t.tm - 1) / (16 * t.tm), nt = (a.N + 64 * t.wn - 1) / (64 * t.wn);
  hipLaunchKernelGGL(kern, dim3(prompt_grid(mt, nt)), dim3(kPThreads), 0, s, a, mt, nt);
  return hipGetLastError();
}

// ============================================================ W4A8
//
// The exact int32 group accumulators come out of the int8 MFMAs as float bits: the
// first product's C operand is the bit pattern of 1.5 * 2^23 (whose unit is 1), so the
// accumulator 1.5 * 2^23 + sum, |sum| <= 128 x 127 x 64 < 2^20, is that float's bit pattern
// plus an integer, i.e. the float 12582912 + sum exactly. One subtraction (a full-rate
// instruction, unlike an int conversion) and one FMA with the group scale per output.
// Codes enter as q - z + 64 (a positive byte for z <= 64: no borrow between bytes); the
// activations' group sums, times -64, are part of the C operand (kPromptMagic - 64 asum,
// which the quantizer writes in place of the sums). Zero-points above 64, which no
// packer writes, are taken off afterwards, in float, as in the batch kernel.
template <int TM, int WN>
__global__ __launch_bounds__(kPThreads, 2) void w4a8_prompt_kernel(GemmArgs a, int mt, int nt) {
  constexpr int SA = TM * 2048;  // bytes of a stage's operand tiles
  __shared__ __align__(16) char xs0[SA], xs1[SA];
  constexpr int CW = (TM + 3) / 4;  // loads of 4 row blocks' C values
  __shared__ __align__(16) char cs0[CW * 256], cs1[CW * 256];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int q = lane >> 4, c = lane & 15;
  const int M = a.M, N = a.N, Kp = a.Kp, G = Kp / kGroup, G4 = t16_groups(Kp), S = (N + 15) / 16;
  int tm, tn;
  if (!prompt_tile(blockIdx.x, mt, nt, tm, tn)) return;
  const int mb0 = tm * TM, s0 = (tn * kPWaves + wave) * WN;
  const uint32_t mblocks = (uint32_t)((M + 15) / 16);
  const Rsrc rx = make_rsrc(a.xq, mblocks * 16u * (uint32_t)Kp);
  const Rsrc rc = make_rsrc(a.asum, mblocks * (uint32_t)G * 64u);
  const Rsrc rw = make_rsrc(a.qw, (uint32_t)min(t16_qw_bytes(N, Kp), (size_t)0xFFFFFFF0u));
  const size_t gents = t16_group_entries(N, Kp);
  const Rsrc rs = make_rsrc(a.scales, (uint32_t)(gents * 4));
  const Rsrc rz = make_rsrc(a.zeros ? a.zeros : a.qw, a.zeros ? (uint32_t)gents : 0u);
  const uint32_t zadd = a.zeros ? 0u : 8u;

  // stage of group g: row block i's two operand tiles (2 KiB, consecutive) and its 16 C values;
  // row blocks past the last read 0
  const auto stage = [&](char *xd, char *cd, int g) {
#pragma unroll
    for (int k = 0; k < TM * 2 / kPWaves; k++) {
      const int t = wave * (TM * 2 / kPWaves) + k, i = t >> 1, h = t & 1;
      lds_load16(rx, xd + t * 1024, ((((uint32_t)(mb0 + i) * G + g) * 2 + h) * kWave + lane) * 16u, 0);
    }
    // every wave loads (the same values where there are fewer loads than waves): a load that
    // only some paths issue would make the waits below count on it never having been issued
    const int cw = wave % CW;
    lds_load4(rc, cd + cw * 256, (((uint32_t)(mb0 + 4 * cw + q) * G + g) * 16 + c) * 4u, 0);
  };
  struct Weights {
    uint4 w[WN];
    float s[WN];
    uint32_t z[WN];
  } w0, w1;
  // subtiles past the last one read it again (their columns are not stored)
  const auto weights = [&](Weights &n, int g) {
#pragma unroll
    for (int j = 0; j < WN; j++) {
      const uint32_t sj = (uint32_t)min(s0 + j, S - 1);
      n.w[j] = ld_b128(rw, (uint32_t)lane * 16u, (sj * G4 + g) * 1024u);
      const uint32_t gu = (sj * (G4 / 4) + g / 4) * 64u;
      n.s[j] = ld_f32(rs, (uint32_t)c * 16u, (gu + (g & 3)) * 4u);
      n.z[j] = ld_u32(rz, (uint32_t)c * 4u, gu);  // no zero-points: a zero-length range reads 0
    }
  };
  v4f facc[TM][WN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < WN; j++) facc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

  const auto group = [&](const char *xd, const char *cd, const Weights &n, int g) {
    v4i blo[WN], bhi[WN];
    float s[WN];
    int rz4[WN], over = 0;
#pragma unroll
    for (int j = 0; j < WN; j++) {
      s[j] = n.s[j];
      const uint32_t z = ((n.z[j] >> (8 * (g & 3))) & 0xFFu) + zadd, z64 = min(z, 64u);
      rz4[j] = (int)(z - z64);
      over |= rz4[j];
      const uint32_t add = 0x40404040u - __builtin_amdgcn_perm(z64, z64, 0u);
      const uint32_t w[4] = {n.w[j].x, n.w[j].y, n.w[j].z, n.w[j].w};
#pragma unroll
      for (int d = 0; d < 4; d++) {
        blo[j][d] = (int)(lo_nibbles(w[d]) + add);
        bhi[j][d] = (int)(hi_nibbles(w[d]) + add);
      }
    }
    // row block i's operands are read while block i - 1 multiplies, and its products are
    // scaled while block i + 1 does
    v4i xlo[2], xhi[2], ci[2], acc[2][WN];
    const auto read = [&](int i) {
      xlo[i & 1] = *reinterpret_cast<const v4i *>(xd + (2 * i) * 1024 + lane * 16);
      xhi[i & 1] = *reinterpret_cast<const v4i *>(xd + (2 * i + 1) * 1024 + lane * 16);
      ci[i & 1] = *reinterpret_cast<const v4i *>(cd + i * 64 + q * 16);
    };
    // (subtractions and FMAs in phases of their own: a dependent pair back to back stalls)
    const auto unbias = [&](int i) {
#pragma unroll
      for (int j = 0; j < WN; j++)
#pragma unroll
        for (int r = 0; r < 4; r++)
          acc[i & 1][j][r] = __float_as_int(__int_as_float(acc[i & 1][j][r]) - 12582912.0f);
    };
    const auto scale = [&](int i) {
#pragma unroll
      for (int j = 0; j < WN; j++)
#pragma unroll
        for (int r = 0; r < 4; r++)
          facc[i][j][r] = __builtin_fmaf(__int_as_float(acc[i & 1][j][r]), s[j], facc[i][j][r]);
    };
    read(0);
#pragma unroll
    for (int i = 0; i < TM; i++) {
      const int b = i & 1;
      if (i + 1 < TM) read(i + 1);
#pragma unroll
      for (int j = 0; j < WN; j++) acc[b][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(xlo[b], blo[j], ci[b], 0, 0, 0);
      if (i > 0) unbias(i - 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < WN; j++)
        acc[b][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(xhi[b], bhi[j], acc[b][j], 0, 0, 0);
      if (i > 0) scale(i - 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    unbias(TM - 1);
    __builtin_amdgcn_sched_barrier(0);
    scale(TM - 1);
    if (__any(over)) {
#pragma unroll
      for (int i = 0; i < TM; i++) {
        const v4i ci = *reinterpret_cast<const v4i *>(cd + i * 64 + q * 16);
#pragma unroll
        for (int j = 0; j < WN; j++)
#pragma unroll
          for (int r = 0; r < 4; r++)
            facc[i][j][r] = __builtin_fmaf((float)(rz4[j] * ((ci[r] - kPromptMagic) >> 6)), s[j], facc[i][j][r]);
      }
    }
  };
  stage(xs0, cs0, 0);
  weights(w0, 0);
  // the next group's loads are issued first (the scheduler would sink them to the end)
  const auto step = [&](char *xd, char *cd, Weights &n, char *nxd, char *ncd, Weights &nn, int g) {
    stage_ready<0>();
    stage(nxd, ncd, min(g + 1, G - 1));
    weights(nn, min(g + 1, G - 1));
    __builtin_amdgcn_sched_barrier(0);
    group(xd, cd, n, g);
  };
  for (int g = 0; g < G; g += 2) {
    step(xs0, cs0, w0, xs1, cs1, w1, g);
    if (g + 1 < G) step(xs1, cs1, w1, xs0, cs0, w0, g + 1);
  }
  stage_ready<0>();  // no load to LDS outlives the workgroup
#pragma unroll
  for (int i = 0; i < TM; i++) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int m = (mb0 + i) * 16 + 4 * q + r;
      if (m >= M) continue;
      const float xs = a.xs[m];
#pragma unroll
      for (int j = 0; j < WN; j++) {
        const int n = 16 * (s0 + j) + c;
        if (n < N) a.y[(size_t)m * N + n] = facc[i][j][r] * xs;
      }
    }
  }
}

hipError_t launch_w4a8_prompt(const GemmArgs &a, PromptTile t, hipStream_t s) {
  if (!a.wt16 || !a.tiled) return hipErrorInvalidValue;
  if (t.tm == 8) return launch_prompt(w4a8_prompt_kernel<8, 2>, a, t, s);
  if (t.tm == 4) return launch_prompt(w4a8_prompt_kernel<4, 2>, a, t, s);
  return launch_prompt(w4a8_prompt_kernel<2, 2>, a, t, s);
}

// ============================================================ MXFP4
//
// The MX matrix instruction (v_mfma_scale_f32_16x16x128_f8f6f4) takes E2M1 weights and
// their E8M0 block scales as they are, a 128-element group per instruction, at four
// times the bf16 rate when the other operand is 6 bits wide. So the weights need no
// decode at all, and each activation becomes kDigits signed digits of E2M3, which holds
// every integer of [-16, 16] and every even one of [-32, 32] (times 1/8): with 2^ex above
// the largest |x| of its block of 32, x 2^(5 - ex) = d1 + d2 2^-5 + d3 2^-10 ..., d1 the
// nearest such integer, and so on with the exact remainders (at most 1/2 where |d| <= 16
// and 1 elsewhere, so that the next digit is within 32 again), the powers of two in the
// activations' own E8M0 scales. Eight digits reach 2^(ex - 40), which is the last bit of
// any float32 from 2^(ex - 17) on: a block with no nonzero element below that is held
// exactly. (A remainder above 1/2 goes back to a first
// digit above 16, whose element ends 24 bits below its leading one, within five digits.)
//
// Other blocks (an element further below its block's largest: 9e-4 of the blocks of normal
// activations with a few channels 8 times the rest; 1e-2 where those are 512 times the
// rest; blocks whose digits' scales would run out; infinities and NaN) are marked, their
// digits are zeros, and the GEMM takes them from the activations as the batch kernel does,
// in three bf16 terms. What a block becomes depends on its own elements only. Products and
// their sums over a group are exact up to the float32 accumulator. The leading digits add
// to one accumulator and the other seven, 2^-5 of its size, to a second, so that Y sees one
// float32 rounding per group.
//
// (Seven digits with marks only where four elements lost bits dropped small elements beside
// a large one. Marks on every loss take 80 % of the 16-row groups of normal activations with
// seven digits, 5 % with eight.)
//
// Measured at 777 x 4096 x 11008, the bf16 batch kernel taking 336 us: 146 us with no marked
// block, 169 for normal activations, 173 with a few channels 8 times the rest, 175 and 182
// with four channels 128 and 512 times the rest (2048 x 11008 x 4096: 306, 367, 368, 398, 428
// against 837). The digits' products bound it, the split takes 17 of it.
//
// Digit tile of (row block, group, digit): lane 16 q + c holds row c, block 4 g + q, slots
// 2 j / 2 j + 1 = elements j / j + 16 (the nibbles of byte j of the packed weights),
// 24 bytes as 16 (1 KiB for the wave) then 8 (512 B), row blocks within a group. After all
// digit tiles, a dword per lane of each (row block, group): the first digit's E8M0 scale;
// after these, 8 bytes of each, groups within a row block: bit l the mark of lane l.
constexpr int kDigitTile = kWave * 24, kDigitBlock = kDigits * kDigitTile, kDigitScale = kWave * 4;
static_assert(kDigitBlock == 12 * 1024, "the GEMM stages whole KiB");
__host__ __device__ inline size_t digit_blocks(int M, int Kp) {
  return (size_t)((M + 15) / 16) * ((Kp + 127) / 128);
}
size_t digit_bytes(int M, int Kp) { return digit_blocks(M, Kp) * (kDigitBlock + kDigitScale + 8); }

typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v32f __attribute__((ext_vector_type(32)));
typedef unsigned int v6u __attribute__((ext_vector_type(6)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef unsigned int v2u __attribute__((ext_vector_type(2)));

// One wave per (row block, group), one lane per (row, block).
__global__ __launch_bounds__(kPThreads) void split_digits_kernel(const float *__restrict__ x, int M, int Kp,
                                                                 char *__restrict__ out) {
  const int lane = threadIdx.x & (kWave - 1), G = (Kp + 127) / 128, mblocks = (M + 15) / 16;
  const size_t items = (size_t)mblocks * G, item = (size_t)blockIdx.x * kPWaves + threadIdx.x / kWave;
  if (item >= items) return;  // whole waves only
  const int mb = (int)(item % mblocks), g = (int)(item / mblocks);
  const int row = 16 * mb + (lane & 15), b = 4 * g + (lane >> 4);
  const Rsrc rx = make_rsrc(x, (uint32_t)((size_t)M * Kp * 4));
  const uint32_t off = row < M && 32 * b < Kp ? (uint32_t)(((size_t)row * Kp + 32 * b) * 4) : 0xFFFFFF00u;
  v16f lo, hi;  // the block's halves, then their remainders in units of the next digit
  uint32_t top = 0, low = 0x7F800000u;  // largest magnitude, smallest nonzero one
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const float4 t = ld_f4(rx, off + 16 * i);
    const float e[4] = {t.x, t.y, t.z, t.w};
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const uint32_t u = __float_as_uint(e[k]) & 0x7FFFFFFFu;
      top = max(top, u);
      low = min(low, u ? u : 0x7F800000u);
      if (i < 4) lo[4 * i + k] = e[k];
      else hi[4 * (i - 4) + k] = e[k];
    }
  }
  int ex = 0;
  (void)frexpf(__uint_as_float(top), &ex);  // top < 2^ex
  // the eighth digit's scale, 2^(ex - 37) in E8M0, must be one
  const bool mark = top >= 0x7F800000u || (top && (ex < -90 || low < __float_as_uint(ldexpf(1.0f, ex - 17))));
  if (mark || !top) ex = 0;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    lo[i] = mark ? 0.0f : ldexpf(lo[i], 5 - ex);
    hi[i] = mark ? 0.0f : ldexpf(hi[i], 5 - ex);
  }
  char *dst = out + item * kDigitBlock;
  // (a loop: unrolled, fetching its code takes most of a small call's time)
#pragma unroll 1
  for (int t = 0; t < kDigits; t++) {
    const v6u p = __builtin_amdgcn_cvt_scalef32_2xpk16_fp6_f32(lo, hi, 8.0f);
    const v32f d = __builtin_amdgcn_cvt_scalef32_pk32_f32_fp6(p, 8.0f);
#pragma unroll
    for (int i = 0; i < 16; i++) {
      lo[i] = (lo[i] - d[2 * i]) * 32.0f;
      hi[i] = (hi[i] - d[2 * i + 1]) * 32.0f;
    }
    *reinterpret_cast<uint4 *>(dst + t * kDigitTile + lane * 16) = make_uint4(p[0], p[1], p[2], p[3]);
    *reinterpret_cast<uint2 *>(dst + t * kDigitTile + 1024 + lane * 8) = make_uint2(p[4], p[5]);
  }
  // digit t + 1 counts units of 2^(ex - 5 - 5 t), the tiles hold eighths: scale 2^(ex - 2 - 5 t)
  char *scales = out + items * kDigitBlock;
  *reinterpret_cast<uint32_t *>(scales + item * kDigitScale + lane * 4) = (uint32_t)(127 + ex - 2);
  const unsigned long long marks = __ballot(mark);
  if (lane == 0)
    reinterpret_cast<unsigned long long *>(scales + items * kDigitScale)[(size_t)mb * G + g] = marks;
}

hipError_t launch_split_digits(const float *x, int M, int Kp, void *out, hipStream_t s) {
  const size_t items = digit_blocks(M, Kp);
  hipLaunchKernelGGL(split_digits_kernel, dim3((unsigned)((items + kPWaves - 1) / kPWaves)), dim3(kPThreads), 0, s, x,
                     M, Kp, static_cast<char *>(out));
  return hipGetLastError();
}

// c + x . w: six-bit digits with scale byte `sel` of sx, E2M1 weights with scale sw.
__device__ __forceinline__ v4f mx_product(int sel, v8i x, int sx, uint4 w4, int sw, v4f c) {
  const v8i w = {(int)w4.x, (int)w4.y, (int)w4.z, (int)w4.w, 0, 0, 0, 0};
  switch (sel) {  // a constant once the callers are unrolled
    case 0: return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(x, w, c, 2, 4, 0, sx, 0, sw);
    case 1: return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(x, w, c, 2, 4, 1, sx, 0, sw);
    case 2: return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(x, w, c, 2, 4, 2, sx, 0, sw);
    default: return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(x, w, c, 2, 4, 3, sx, 0, sw);
  }
}

template <int TM, int WN>
__global__ __launch_bounds__(kPThreads, 2) void mxfp4_prompt_kernel(GemmArgs a, int mt, int nt) {
  constexpr int SK = TM * kDigitBlock / 1024, PW = SK / kPWaves;  // KiB of a stage, and of a wave's share
  __shared__ __align__(16) char xs0[SK * 1024], xs1[SK * 1024], xs2[SK * 1024];
  __shared__ __align__(16) char es0[TM * kDigitScale], es1[TM * kDigitScale], es2[TM * kDigitScale];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int q = lane >> 4, c = lane & 15;
  const int M = a.M, N = a.N, Kp = a.Kp, G = (Kp + 127) / 128, G4 = t16_groups(Kp), S = (N + 15) / 16;
  int tm, tn;
  if (!prompt_tile(blockIdx.x, mt, nt, tm, tn)) return;
  const int mb0 = tm * TM, s0 = (tn * kPWaves + wave) * WN;
  const uint32_t mblocks = (uint32_t)((M + 15) / 16);
  const uint32_t xbytes = mblocks * (uint32_t)G * (uint32_t)kDigitBlock;
  const Rsrc rd = make_rsrc(a.x3, xbytes);
  const Rsrc rse = make_rsrc(reinterpret_cast<const char *>(a.x3) + xbytes, mblocks * (uint32_t)G * (uint32_t)kDigitScale);
  const Rsrc rx = make_rsrc(a.x, (uint32_t)((size_t)M * Kp * 4));
  const Rsrc rw = make_rsrc(a.qw, (uint32_t)min(t16_qw_bytes(N, Kp), (size_t)0xFFFFFFF0u));
  const Rsrc re = make_rsrc(a.e8m0, (uint32_t)t16_e8m0_bytes(N, Kp));

  struct Weights {
    uint4 w[WN];
    uint32_t e[WN];
  } w0, w1, w2;
  // load `op` of this wave for group g: the first PW copy its share of the stage (row blocks
  // are consecutive within a group, so a stage is one run of KiB; past the last row block
  // it reads the next group's, rows that are not stored, or zeros at the end), the next a
  // row block's scales (every wave one, so that all wait for as many loads), the others
  // its subtiles' weights and scales (past the last subtile: its columns are not stored)
  constexpr int OPS = PW + 1 + 2 * WN;
  const auto load = [&](int op, char *xd, char *ed, Weights &n, int g) {
    const uint32_t block = (uint32_t)g * mblocks + (uint32_t)mb0;
    if (op < PW) {
      const int t = wave * PW + op;
      lds_load16(rd, xd + t * 1024, block * (uint32_t)kDigitBlock + (uint32_t)t * 1024u + (uint32_t)lane * 16u, 0);
    } else if (op == PW) {
      const int t = wave % TM;
      lds_load4(rse, ed + t * kDigitScale, (block + t) * (uint32_t)kDigitScale + (uint32_t)lane * 4u, 0);
    } else if (op < OPS) {
      const int j = (op - PW - 1) >> 1;
      const uint32_t sj = (uint32_t)min(s0 + j, S - 1);
      if ((op - PW - 1) & 1) n.e[j] = ld_u32(re, (uint32_t)(lane & ~3), (sj * G4 + g) * 64u);
      else n.w[j] = ld_b128(rw, (uint32_t)lane * 16u, (sj * G4 + g) * 1024u);
    }
  };
  v4f hi[TM][WN], lo[TM][WN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < WN; j++) hi[i][j] = v4f{0.f, 0.f, 0.f, 0.f}, lo[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

  // One group, with the loads of the one after the next between its products. A product
  // occupies the matrix core for 16 cycles and the wave's issue for 8, so
  // what is issued one by one between products costs nothing, and in clumps its whole time;
  // every slot is pinned, as the scheduler would make clumps (and sink the loads to the end).
  const auto group = [&](const char *xd, const char *ed, const Weights &n, char *nxd, char *ned, Weights &nn, int g) {
    constexpr int K = TM * kDigits;  // step k: row block k / kDigits, digit k % kDigits
    v4i xa[3];
    v2u xb[3];
    uint32_t sc[2][2];
    const auto read_a = [&](int k) {
      xa[k % 3] = *reinterpret_cast<const v4i *>(xd + (k / kDigits) * kDigitBlock + (k % kDigits) * kDigitTile + lane * 16);
    };
    const auto read_b = [&](int k) {
      const char *blk = xd + (k / kDigits) * kDigitBlock;
      xb[k % 3] = *reinterpret_cast<const v2u *>(blk + (k % kDigits) * kDigitTile + 1024 + lane * 8);
      if (k % kDigits == 0) {  // scales five apart, no borrow between bytes: the first is at least 35
        uint32_t *p = sc[(k / kDigits) & 1];
        const uint32_t e = *reinterpret_cast<const uint32_t *>(ed + (k / kDigits) * kDigitScale + lane * 4);
        p[0] = __builtin_amdgcn_perm(e, e, 0u) - 0x0F0A0500u;
        p[1] = p[0] - 0x14141414u;
      }
    };
    read_a(0);
    read_b(0);
    read_a(1);
    read_b(1);
    int sw[WN];  // the lane's byte of its dword of scales (the instruction reads the lowest)
#pragma unroll
    for (int j = 0; j < WN; j++) sw[j] = (int)(n.e[j] >> (8 * (lane & 3)));
    int op = 0;
#pragma unroll
    for (int k = 0; k < K; k++) {
      const int i = k / kDigits, t = k % kDigits;
      const v8i x = {xa[k % 3][0], xa[k % 3][1], xa[k % 3][2], xa[k % 3][3], (int)xb[k % 3][0], (int)xb[k % 3][1], 0, 0};
#pragma unroll
      for (int j = 0; j < WN; j++) {
        v4f &o = t == 0 ? hi[i][j] : lo[i][j];
        o = mx_product(t & 3, x, (int)sc[i & 1][t >> 2], n.w[j], sw[j], o);
        __builtin_amdgcn_sched_barrier(0);
        if (j == 0 && k + 2 < K) read_a(k + 2);
        if (j == 1 && k + 2 < K) read_b(k + 2);
        if (j >= 2) load(op++, nxd, ned, nn, min(g + 2, G - 1));
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    static_assert(K * (WN - 2) >= OPS, "every load has a slot");
  };
  // the marks of groups g0 + lane (those of the first 64 groups are loaded ahead)
  unsigned long long mine[TM];
  const auto load_marks = [&](int g0) {
    const auto *marks = reinterpret_cast<const unsigned long long *>(reinterpret_cast<const char *>(a.x3) + xbytes +
                                                                     (size_t)mblocks * G * kDigitScale);
#pragma unroll
    for (int i = 0; i < TM; i++)
      mine[i] = mb0 + i < (int)mblocks && g0 + lane < G ? marks[(size_t)(mb0 + i) * G + g0 + lane] : 0;
  };
  load_marks(0);
  __builtin_amdgcn_sched_barrier(0);
  // two groups are in flight ahead of the one that runs
#pragma unroll
  for (int op = 0; op < OPS; op++) load(op, xs0, es0, w0, 0);
  __builtin_amdgcn_sched_barrier(0);  // stage_ready counts on all of group 0's loads coming first
#pragma unroll
  for (int op = 0; op < OPS; op++) load(op, xs1, es1, w1, min(1, G - 1));
  __builtin_amdgcn_sched_barrier(0);
  const auto step = [&](const char *xd, const char *ed, const Weights &n, char *nxd, char *ned, Weights &nn, int g) {
    stage_ready<OPS>();
    group(xd, ed, n, nxd, ned, nn, g);
  };
  // (no way into a step but from the one before it: where two meet, the compiler waits for
  // the loads that either has in flight)
  int g = 0;
  for (; g + 3 <= G; g += 3) {
    step(xs0, es0, w0, xs2, es2, w2, g);
    step(xs1, es1, w1, xs0, es0, w0, g + 1);
    step(xs2, es2, w2, xs1, es1, w1, g + 2);
  }
  if (g < G) step(xs0, es0, w0, xs2, es2, w2, g);
  if (g + 1 < G) step(xs1, es1, w1, xs0, es0, w0, g + 1);
  stage_ready<0>();  // no load to LDS outlives the workgroup
  // Marked blocks: weights, terms and order of the batch kernel (bf3_gemm_kernel), the terms
  // of the other blocks zero, so that no row changes with the others of its row block. Apart
  // from the loop above, whose registers they would spill. Up to 3 TM (row block, group)s at
  // once: wave u makes their operands u in the stages' LDS, then every wave takes them all.
  // (Little code: for a call of one round, fetching it is most of the cost.)
  constexpr int R = 3 * TM;
  const auto room = [&](int t) { return (t < TM ? xs0 : t < 2 * TM ? xs1 : xs2) + t % TM * kDigitBlock; };
  for (int g0 = 0; g0 < G; g0 += kWave) {
    if (g0 > 0) load_marks(g0);
    unsigned long long todo[TM];
#pragma unroll
    for (int i = 0; i < TM; i++) todo[i] = __ballot(mine[i] != 0);
    // the next of a list: row block i, group g0 + gl; false (and gl = 0) past its end
    const auto next = [](unsigned long long (&t)[TM], int &i, int &gl) {
      i = TM > 1 && !t[0];
      const unsigned long long v = t[0] ? t[0] : t[TM - 1];
      gl = v ? __builtin_ctzll(v) : 0;
      if (TM > 1 && i) t[TM - 1] = v & (v - 1);
      else t[0] = v & (v - 1);
      return v != 0;
    };
    while (todo[0] | todo[TM - 1]) {
      float4 l4[R], h4[R];
      unsigned long long list[TM];
      int count = 0, i, gl;
#pragma unroll
      for (int k = 0; k < TM; k++) list[k] = todo[k];
#pragma unroll
      for (int t = 0; t < R; t++) {
        const bool some = next(list, i, gl);
        count += some;
        const unsigned long long m = i ? mine[TM - 1] : mine[0];
        const uint32_t half = lane < 32 ? __builtin_amdgcn_readlane((uint32_t)m, gl)
                                        : __builtin_amdgcn_readlane((uint32_t)(m >> 32), gl);
        const bool mark = some && (half >> (lane & 31) & 1u);
        // (a marked block is inside the activations)
        const uint32_t off = (uint32_t)(((size_t)(16 * (mb0 + i) + c) * Kp + 128 * (g0 + gl) + 32 * q + 4 * wave) * 4);
        l4[t] = ld_f4(rx, mark ? off : 0xFFFFFF00u);
        h4[t] = ld_f4(rx, mark ? off + 64 : 0xFFFFFF00u);
      }
      const auto weights = [&](Weights &n, int g) {
#pragma unroll
        for (int op = PW + 1; op < OPS; op++) load(op, nullptr, nullptr, n, g);
      };
      Weights n;
      next(todo, i, gl);
      weights(n, g0 + gl);
      __builtin_amdgcn_sched_barrier(0);
      __syncthreads();
#pragma unroll
      for (int t = 0; t < R; t++) {
        if (t >= count) break;
        const float v[8] = {l4[t].x, h4[t].x, l4[t].y, h4[t].y, l4[t].z, h4[t].z, l4[t].w, h4[t].w};
        uint32_t x3[3][4];
#pragma unroll
        for (int k = 0; k < 4; k++) split3_pair(v[2 * k], v[2 * k + 1], x3[0][k], x3[1][k], x3[2][k]);
#pragma unroll
        for (int p = 0; p < 3; p++)
          *reinterpret_cast<uint4 *>(room(t) + (wave * 3 + p) * 1024 + lane * 16) =
              make_uint4(x3[p][0], x3[p][1], x3[p][2], x3[p][3]);
      }
      __syncthreads();
#pragma unroll 1
      for (int t = 0; t < count; t++) {
        const Weights w = n;
        const int it = i;
        if (t + 1 < count) {
          next(todo, i, gl);
          weights(n, g0 + gl);
        }
        const char *xb = room(t) + lane * 16;
        v4f d[WN];
        float bs[WN], fs[WN];
#pragma unroll
        for (int j = 0; j < WN; j++) {
          const int e = (int)((w.e[j] >> (8 * (lane & 3))) & 0xFFu);
          int emax = max(e, __shfl_xor(e, 16));
          emax = max(emax, __shfl_xor(emax, 32));
          bs[j] = e - emax >= -126 ? __uint_as_float((uint32_t)(e - emax + 127) << 23) : 0.0f;
          fs[j] = e8m0_to_f32((uint32_t)emax);
          d[j] = v4f{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
          v4u wb[WN];
#pragma unroll
          for (int j = 0; j < WN; j++) {
            const uint32_t wu = u == 0 ? w.w[j].x : u == 1 ? w.w[j].y : u == 2 ? w.w[j].z : w.w[j].w;
            wb[j] = v4u{__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(wu, bs[j], 0)),
                        __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(wu, bs[j], 1)),
                        __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(wu, bs[j], 2)),
                        __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(wu, bs[j], 3))};
          }
#pragma unroll
          for (int p = 0; p < 3; p++) {
            const v8bf x = *reinterpret_cast<const v8bf *>(xb + (u * 3 + p) * 1024);
#pragma unroll
            for (int j = 0; j < WN; j++)
              d[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, __builtin_bit_cast(v8bf, wb[j]), d[j], 0, 0, 0);
          }
        }
#pragma unroll
        for (int k = 0; k < TM; k++) {
          if (it != k) continue;
#pragma unroll
          for (int j = 0; j < WN; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) hi[k][j][r] = __builtin_fmaf(fs[j], d[j][r], hi[k][j][r]);
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < TM; i++) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int m = (mb0 + i) * 16 + 4 * q + r;
      if (m >= M) continue;
#pragma unroll
      for (int j = 0; j < WN; j++) {
        const int n = 16 * (s0 + j) + c;
        if (n < N) a.y[(size_t)m * N + n] = hi[i][j][r] + lo[i][j][r];
      }
    }
  }
}

hipError_t launch_mxfp4_prompt(const GemmArgs &a, PromptTile t, hipStream_t s) {
  if (!a.wt16 || !a.x3) return hipErrorInvalidValue;
  if (t.tm == 1) return launch_prompt(mxfp4_prompt_kernel<1, 4>, a, t, s);
  return launch_prompt(mxfp4_prompt_kernel<2, 4>, a, t, s);
}

// ============================================================ W4A16
//
// The arithmetic of the batch kernel (bf3_gemm_kernel with H2): two float16 terms per
// activation, hi + lo 2^-11, each row times 2^xexp, against the exact float16 q - z; the
// two sums of a group meet and take the group scale in float32, and eight groups' sums
// meet before they join the total, so that the float32 roundings of a long K do not all
// happen at the total's size.
//
//   t16 decode: the bytes 00 64 with the low one a nibble are the float16 1024 + q, less
//   1024 + z exact. t16f8 weights, two conversions a dword, become the same operands in the
//   same order, so both layouts give the same bits.
template <int TM, int WN, bool F8>
__global__ __launch_bounds__(kPThreads, 2) void w4a16_prompt_kernel(GemmArgs a, int mt, int nt) {
  constexpr int SK = TM * 8, PW = SK / kPWaves;  // KiB of a stage, and of a wave's share
  __shared__ __align__(16) char xs0[SK * 1024], xs1[SK * 1024];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int q = lane >> 4, c = lane & 15;
  const int M = a.M, N = a.N, Kp = a.Kp, G = Kp / kGroup, G4 = t16_groups(Kp), S = (N + 15) / 16;
  int tm, tn;
  if (!prompt_tile(blockIdx.x, mt, nt, tm, tn)) return;
  const int mb0 = tm * TM, s0 = (tn * kPWaves + wave) * WN;
  const Rsrc rx = make_rsrc(a.x3, (uint32_t)min(x2h_bytes(M, Kp), (size_t)0xFFFFFFF0u));
  const Rsrc rw = make_rsrc(a.qw, (uint32_t)min(F8 ? t16f8_qw_bytes(N, Kp) : t16_qw_bytes(N, Kp), (size_t)0xFFFFFFF0u));
  const size_t gents = t16_group_entries(N, Kp);
  const Rsrc rs = make_rsrc(a.scales, (uint32_t)(gents * 4));
  const Rsrc rz = make_rsrc(a.zeros ? a.zeros : a.qw, !F8 && a.zeros ? (uint32_t)gents : 0u);
  const uint32_t zadd = a.zeros ? 0u : 8u;

  struct Weights {
    uint4 w[WN], w2[F8 ? WN : 1];
    float s[WN];
    uint32_t z[WN];
  } wt;
  constexpr int OPS = PW + 3 * WN;
  const auto load = [&](int op, char *xd, int g) {
    if (op < PW) {
      const int t = wave * PW + op;  // KiB t % 8 of row block t / 8; past the last row block zeros
      lds_load16(rx, xd + t * 1024, (((uint32_t)(mb0 + (t >> 3)) * G + g) * 8u + (t & 7)) * 1024u + (uint32_t)lane * 16u, 0);
    } else if (op < OPS) {
      const int j = (op - PW) / 3;
      const uint32_t sj = (uint32_t)min(s0 + j, S - 1), gu = (sj * (G4 / 4) + g / 4) * 64u;
      const uint32_t wb = (sj * G4 + g) * (F8 ? 2048u : 1024u);
      if ((op - PW) % 3 == 0) wt.w[j] = ld_b128(rw, (uint32_t)lane * 16u, wb);
      else if ((op - PW) % 3 == 1) wt.s[j] = ld_f32(rs, (uint32_t)c * 16u, (gu + (g & 3)) * 4u);
      else if constexpr (F8) wt.w2[j] = ld_b128(rw, (uint32_t)lane * 16u, wb + 1024u);
      else wt.z[j] = ld_u32(rz, (uint32_t)c * 4u, gu);
    }
  };
  v4f facc[TM][WN], total[TM][WN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < WN; j++) facc[i][j] = v4f{0.f, 0.f, 0.f, 0.f}, total[i][j] = facc[i][j];

  const auto group = [&](const char *xd, char *nxd, int g) {
    const int gn = min(g + 1, G - 1);
    v4u b[WN][4];
    float s[WN];
#pragma unroll
    for (int j = 0; j < WN; j++) {
      s[j] = wt.s[j];
      if constexpr (F8) {  // operand u, element e = lane byte 8 u + e, already less its zero-point
        const uint32_t w[8] = {wt.w[j].x, wt.w[j].y, wt.w[j].z, wt.w[j].w, wt.w2[j].x, wt.w2[j].y, wt.w2[j].z, wt.w2[j].w};
#pragma unroll
        for (int d = 0; d < 8; d++) {
          b[j][d >> 1][2 * (d & 1)] =
              __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w[d], 512.0f, false));
          b[j][d >> 1][2 * (d & 1) + 1] =
              __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w[d], 512.0f, true));
        }
      } else {
        const float z = (float)(((wt.z[j] >> (8 * (g & 3))) & 0xFFu) + zadd);
        const h2v z2 = {(_Float16)(1024.0f + z), (_Float16)(1024.0f + z)};
        const uint32_t w[4] = {wt.w[j].x, wt.w[j].y, wt.w[j].z, wt.w[j].w};
#pragma unroll
        for (int d = 0; d < 8; d++) {  // operands u = d / 2: low nibbles of dwords 0 .. 3, then high
          const uint32_t nib = d < 4 ? lo_nibbles(w[d & 3]) : hi_nibbles(w[d & 3]);
          const h2v lo = __builtin_bit_cast(h2v, __builtin_amdgcn_perm(0x64646464u, nib, 0x07010700u));
          const h2v hi = __builtin_bit_cast(h2v, __builtin_amdgcn_perm(0x64646464u, nib, 0x07030702u));
          b[j][d >> 1][2 * (d & 1)] = __builtin_bit_cast(uint32_t, lo - z2);
          b[j][d >> 1][2 * (d & 1) + 1] = __builtin_bit_cast(uint32_t, hi - z2);
        }
      }
    }
    v8h xa[2][2];  // [parity][hi, lo] of step k = (row block k / 4, u = k % 4)
    v4f dh[2][WN], dl[2][WN];
    const auto read = [&](int k, int p) {
      xa[k & 1][p] = *reinterpret_cast<const v8h *>(xd + (k * 2 + p) * 1024 + lane * 16);
    };
    // products of row block i go through the scale while row block i + 1 multiplies: merges
    // first, then the scale (a dependent pair back to back stalls)
    const auto scale = [&](int i, int slot) {
      const int e0 = (slot % (2 * WN)) * 2;
#pragma unroll
      for (int e = e0; e < e0 + 2; e++) {
        const int j = e >> 2, r = e & 3;
        if (slot < 2 * WN) dh[i & 1][j][r] = __builtin_fmaf(dl[i & 1][j][r], 0x1p-11f, dh[i & 1][j][r]);
        else facc[i][j][r] = __builtin_fmaf(s[j], dh[i & 1][j][r], facc[i][j][r]);
      }
    };
    read(0, 0);
    read(0, 1);
    __builtin_amdgcn_sched_barrier(0);
    int op = 0;
#pragma unroll
    for (int k = 0; k < 4 * TM; k++) {
      const int i = k >> 2, u = k & 3;
#pragma unroll
      for (int j = 0; j < WN; j++) {
        const v4f zero = {0.f, 0.f, 0.f, 0.f};
        const v8h bj = __builtin_bit_cast(v8h, b[j][u]);
        dh[i & 1][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[k & 1][0], bj, u ? dh[i & 1][j] : zero, 0, 0, 0);
        if (j < 2 && k + 1 < 4 * TM) read(k + 1, j);
        else load(op++, nxd, gn);
        dl[i & 1][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[k & 1][1], bj, u ? dl[i & 1][j] : zero, 0, 0, 0);
        if (i > 0) scale(i - 1, u * WN + j);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    static_assert((4 * TM - 1) * (WN - 2) + WN >= OPS, "every load has a slot");
#pragma unroll
    for (int n = 0; n < 4 * WN; n++) scale(TM - 1, n);
  };
  const auto meet = [&]() {
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < WN; j++) total[i][j] += facc[i][j], facc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
  };
#pragma unroll
  for (int op = 0; op < OPS; op++) load(op, xs0, 0);
  const auto step = [&](const char *xd, char *nxd, int g) {
    stage_ready<0>();
    group(xd, nxd, g);
  };
  for (int g = 0; g < G; g += 2) {
    step(xs0, xs1, g);
    if (g + 1 < G) step(xs1, xs0, g + 1);
    if ((g & 7) == 6) meet();
  }
  meet();
  stage_ready<0>();  // no load to LDS outlives the workgroup
#pragma unroll
  for (int i = 0; i < TM; i++) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int m = (mb0 + i) * 16 + 4 * q + r;
      if (m >= M) continue;
      const int e = -a.xexp[m];
#pragma unroll
      for (int j = 0; j < WN; j++) {
        const int n = 16 * (s0 + j) + c;
        if (n < N) a.y[(size_t)m * N + n] = ldexpf(total[i][j][r], e);
      }
    }
  }
}

hipError_t launch_w4a16_prompt(const GemmArgs &a, PromptTile t, bool f8, hipStream_t s) {
  if (!a.wt16 || !a.x3 || !a.xexp) return hipErrorInvalidValue;
  return f8 ? launch_prompt(w4a16_prompt_kernel<2, 4, true>, a, t, s)
            : launch_prompt(w4a16_prompt_kernel<2, 4, false>, a, t, s);
}

// ============================================================ dispatch
//
// Where these kernels beat the batch kernels, from both sides' times (us) at 56 shapes of
// 80-1024 rows, N 300-11008, K 896-11008 with the weights warm. A tile walks K serially:
// a launch that leaves each CU one workgroup or less takes (a little more than) G times
// its time per group however few rows there are, while the batch kernels' time falls with
// the work; so the line is drawn in 16 x 16 tiles of Y per CU, T.
//   MXFP4  11 us + 0.68 a group with 16-row tiles, taken while they fill one round of the CUs;
//          12.5 + 0.97 a group with 32-row ones in one round, 1 + r / 2 in r <= 2, r + 0.6 in
//          more; against 8 us + (0.5 + 0.0002 M) a group and chunk of the batch kernel, a chunk
//          being 6 of the 16-column subtiles that a workgroup of its grid walks (normal
//          activations with a few large channels; 170 shapes of 33-1552 rows): 192 x 4096 x
//          4096 40.7 -> 32.2, 448 x 4096 x 4096 64.5 -> 46.1, 1024 x 4096 x 4096 179 -> 80,
//          33 x 28672 x 8192 93.3 -> 72.5, 1024 x 4096 x 11008 448 -> 187. Not taken: 192 x
//          4096 x 1024 15.4 against 16.3, 112 x 11008 x 4096 40.3 against 44.3, 240 x 9085 x
//          7008 98.1 against 101, 272 x 8013 x 2048 35.9 against 41.0.
//   W4A16  1.13 us a group and round of 256 workgroups against 0.055 T of the batch kernel
//          (512 x 4096 x 4096 60.5 -> 49.0, 2048 x 11008 x 4096 642 -> 364; 256 x 4096 x
//          4096 39.9 against 44.4, not taken).
//   W4A8   32-, 64- and 128-row tiles: 0.57, 0.72, 1.13 us a group, 0.0205, 0.0163, 0.0140 T
//          when the chip is full, against 0.0235 T a group of the batch kernel, which
//          works on phases of 32 groups (1024 x 4096 x 11008 231 -> 90, 384 x 4096 x 1024
//          22.9 -> 12.4, 2048 x 11008 x 4096 252 -> 150; 256 x 4096 x 4096 17.8 against 25).
//          One whole phase is the batch kernel at its best (256 x 9728 x 4096 32.6 against
//          34.2, not taken; 384 x 9728 x 4096 44.1 -> 35.1).
// Few rows (32 and less) stay with the batch kernels, which are built for them.
bool prompt_tile_for(int fmt, int M, int N, int Kp, int num_cus, PromptTile *out) {
  if (M <= 32) return false;
  // 32-bit offsets, up to a tile past the last row (the other formats' callers have checked)
  if (fmt == F_W4A8 && ((size_t)M + 160) * Kp > 0xFFFFFF00u) return false;
  const double cus = num_cus > 0 ? num_cus : 256, G = (Kp + 127) / 128;
  const double T = (double)((M + 15) / 16) * ((N + 15) / 16) / cus;
  const auto rounds = [&](int tm, int wn) {
    return (double)((M + 16 * tm - 1) / (16 * tm)) * ((N + 64 * wn - 1) / (64 * wn)) / cus;
  };
  PromptTile t;
  if (fmt == F_MXFP4) {
    t = PromptTile{rounds(1, 4) <= 1 ? 1 : 2, 4};
    const double r = rounds(2, 4), per = t.tm == 1 ? 0.68 : r <= 1 ? 0.97 : r <= 2 ? 1 + 0.5 * r : r + 0.6;
    const int gy = (M + 31) / 32, S = (N + 15) / 16, gx = std::max(1, std::min(S, (int)cus / gy));
    const double chunks = ((S + gx - 1) / gx + 5) / 6;
    if ((t.tm == 1 ? 11 : 12.5) + G * per > 0.97 * (8 + G * chunks * (0.5 + 0.0002 * M))) return false;
  } else if (fmt == F_W4A16) {
    t = PromptTile{2, 4};
    if (1.13 * std::ceil(rounds(2, 4)) > 0.055 * T) return false;
  } else if (fmt == F_W4A8) {
    const double per[3] = {std::max(0.57, 0.0205 * T), std::max(0.72, 0.0163 * T), std::max(1.13, 0.0140 * T)};
    const int best = (int)(std::min_element(per, per + 3) - per);
    t = PromptTile{2 << best, 2};
    const double batch = 0.0235 * T * 32 * std::ceil(G / 32);
    if (1.0 + G * per[best] > (G == 32 ? 0.8 : 0.9) * batch) return false;
  } else {
    return false;
  }
  *out = t;
  return true;
}

}  // namespace lbk
