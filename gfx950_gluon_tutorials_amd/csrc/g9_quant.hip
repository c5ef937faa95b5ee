// Operand quantizers (declared in include/gfx950_gemm.h): MXFP4 in one pass,
// BF8 (e5m2, one scale per tensor) in two.
//
// Bound by HBM: 16-bit values are read once (MXFP4) or twice (BF8) and written
// as 4.25 or 8 bits.  A thread converts 8 consecutive values (16 bytes of a
// 16-bit input), so a wave reads and writes contiguous runs; the four threads
// of a 32-value MXFP4 group exchange their largest magnitude.  4096 x 7168
// BF16 to MXFP4, one MI355X: 13.2 us (5.6 TB/s); the same in torch,
// as ~40 passes over the tensor with 64-bit intermediates, 1669 us.  To BF8:
// 32 us (147 MB in two passes; the division is fp32), 192 us in torch.
#include "../../include/gfx950_gemm.h"
#include "g9_common.hpp"

using namespace g9;

namespace {

enum { IN_F16 = 0, IN_BF16 = 1, IN_F32 = 2 };
constexpr int kThreads = 256;
constexpr u32 kInf = 0x7f800000u;

// Values 8 i .. 8 i + 7 as fp32.
template <int IN>
G9_DEV void load8(const void* x, size_t i, float (&v)[8]) {
  if constexpr (IN == IN_F32) {
    const f32x4* p = static_cast<const f32x4*>(x) + 2 * i;
    const f32x4 a = p[0], b = p[1];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = a[k], v[4 + k] = b[k];
  } else {
    const u32x4 w = static_cast<const u32x4*>(x)[i];
    if constexpr (IN == IN_BF16) {
#pragma unroll
      for (int k = 0; k < 4; ++k) v[2 * k] = __uint_as_float(w[k] << 16), v[2 * k + 1] = __uint_as_float(w[k] & 0xffff0000u);
    } else {
      const f16x8 h = __builtin_bit_cast(f16x8, w);
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = (float)h[k];
    }
  }
}
// Magnitudes compare as integers, NaN above infinity.
G9_DEV u32 mag(float x) { return __float_as_uint(x) & 0x7fffffffu; }

// E = floor(log2(amax)) - 2 clamped to +-127 (-127 for a zero or NaN group, -3
// for an infinite one, whose frexp exponent is 0).  Codes are |x| / 2^E rounded
// to e2m1 and saturated: by the conversion instruction, or in its special
// cases (below) by comparing |x| with the midpoints times 2^E, which are exact
// in fp32, denormals included (for all values that would be bound by the VALU:
// 30.3 us where the instruction takes 13.2).  Ties go to the even code, except
// where pow(2, -E) comes out below 2^-E: the product x * pow(2, -E), which
// defines the bytes, then falls below the midpoint.  Which exponents those
// are is worked out once per block (an fp64 pow per 8-value piece would cost
// as much as the memory traffic).
template <int IN>
__global__ __launch_bounds__(kThreads) void quant_mxfp4(const void* x, u32* packed, unsigned char* scales, size_t n8) {
  __shared__ unsigned char low[256];
  {
    const int e = 127 - (int)threadIdx.x;  // -E for E = threadIdx.x - 127
    low[threadIdx.x] = pow(2.0, (double)e) < ldexp(1.0, e);
  }
  __syncthreads();
  // n8 is a multiple of 4 and so is the stride: the four lanes of a group
  // leave the loop together.
  for (size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x; i < n8; i += (size_t)gridDim.x * kThreads) {
    float v[8];
    load8<IN>(x, i, v);
    u32 m = mag(v[0]);
#pragma unroll
    for (int k = 1; k < 8; ++k) m = max(m, mag(v[k]));
    m = max(m, (u32)__shfl_xor((int)m, 1, 64));
    m = max(m, (u32)__shfl_xor((int)m, 2, 64));
    int E = max((int)(m >> 23) - 127 - 2, -127);  // zero and denormals (biased exponent 0) clamp as well
    if (m >= kInf) E = m == kInf ? -3 : -127;
    if (threadIdx.x % 4 == 0) scales[i / 4] = (unsigned char)(E + 127);
    const bool down = low[E + 127];
    // 2^E, also where it is denormal.
    const float s = E >= -126 ? __uint_as_float((u32)(E + 127) << 23) : __uint_as_float(0x00400000u);
    u32 w = 0;
    if (__builtin_expect(!(down | (m >= kInf) | (E < -126)), 1)) {
      // The conversion instructions (round to nearest even, saturating); the
      // sum turns -0, whose code is 0, into 0.
      w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, v[0] + 0.f, v[1] + 0.f, s, 0);
      w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, v[2] + 0.f, v[3] + 0.f, s, 1);
      w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, v[4] + 0.f, v[5] + 0.f, s, 2);
      w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, v[6] + 0.f, v[7] + 0.f, s, 3);
    } else {
      const float t1 = 0.25f * s, t2 = 0.75f * s, t3 = 1.25f * s, t4 = 1.75f * s, t5 = 2.5f * s, t6 = 3.5f * s,
                  t7 = 5.f * s;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const float a = __builtin_fabsf(v[k]);
        u32 c = (u32)(a > t1) + (u32)(a > t2) + (u32)(a > t3) + (u32)(a > t4) + (u32)(a > t5) + (u32)(a > t6) +
                (u32)(a > t7);
        // The ties whose even neighbour is above.
        if (!down) c += (u32)(a == t2) + (u32)(a == t4) + (u32)(a == t6);
        if (v[k] < 0.f) c |= 8;
        w |= c << (4 * k);
      }
    }
    packed[i] = w;
  }
}

// Largest magnitude (as bits) of each block's share, grid-stride.
template <int IN>
__global__ __launch_bounds__(kThreads) void quant_amax(const void* x, size_t n, u32* part) {
  __shared__ u32 red[kThreads / 64];
  const size_t n8 = n / 8;
  u32 m = 0;
  for (size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x; i < n8; i += (size_t)gridDim.x * kThreads) {
    float v[8];
    load8<IN>(x, i, v);
#pragma unroll
    for (int k = 0; k < 8; ++k) m = max(m, mag(v[k]));
  }
  if (blockIdx.x == 0 && threadIdx.x < n % 8) {
    const size_t i = n8 * 8 + threadIdx.x;
    const float v = IN == IN_F32    ? static_cast<const float*>(x)[i]
                    : IN == IN_BF16 ? __uint_as_float((u32) static_cast<const uint16_t*>(x)[i] << 16)
                                    : (float)static_cast<const _Float16*>(x)[i];
    m = max(m, mag(v));
  }
#pragma unroll
  for (int d = 32; d; d >>= 1) m = max(m, (u32)__shfl_xor((int)m, d, 64));
  if (threadIdx.x % 64 == 0) red[threadIdx.x / 64] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kThreads / 64; ++w) m = max(m, red[w]);
    part[blockIdx.x] = m;
  }
}

// fp32 -> e5m2, round to nearest even; |x| <= 57344 or NaN.
G9_DEV u32 e5m2(float x) {
  const u32 b = __float_as_uint(x), u = b & 0x7fffffffu, sign = (b >> 24) & 0x80u;
  if (u > kInf) return 0x7fu | sign;
  if (u < (113u << 23)) return (u32)(int)__builtin_rintf(__uint_as_float(u) * 65536.f) | sign;  // units of 2^-16
  return ((u + 0xfffffu + ((u >> 21) & 1u)) >> 21) - (112u << 2) | sign;
}
G9_DEV u32 code8(float v, float scale) {
  const float q = v / scale;
  // A NaN stays one.
  return e5m2(q > 57344.f ? 57344.f : q < -57344.f ? -57344.f : q);
}

template <int IN>
__global__ __launch_bounds__(kThreads) void quant_e5m2(const void* x, size_t n, const u32* part, int parts,
                                                       unsigned char* codes, float* scale_out) {
  __shared__ u32 red[kThreads / 64];
  u32 m = 0;
  for (int k = threadIdx.x; k < parts; k += kThreads) m = max(m, part[k]);
#pragma unroll
  for (int d = 32; d; d >>= 1) m = max(m, (u32)__shfl_xor((int)m, d, 64));
  if (threadIdx.x % 64 == 0) red[threadIdx.x / 64] = m;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kThreads / 64; ++w) m = max(m, red[w]);
  // amax / 57344, as a product with the constant's reciprocal; 1 for an
  // all-zero or NaN tensor.
  const float scale = m == 0 || m > kInf ? 1.f : __uint_as_float(m) * (1.f / 57344.f);
  if (blockIdx.x == 0 && threadIdx.x == 0) *scale_out = scale;
  // The conversion instruction where no quotient is a NaN: a finite tensor
  // whose scale has not underflowed.
  const bool plain = m < kInf && scale >= 1e-30f;
  const size_t n8 = n / 8;
  for (size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x; i < n8; i += (size_t)gridDim.x * kThreads) {
    float v[8];
    load8<IN>(x, i, v);
    u32 w[2] = {0, 0};
    if (plain) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float q[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) q[k] = __builtin_fmaxf(__builtin_fminf(v[4 * h + k] / scale, 57344.f), -57344.f);
        w[h] = __builtin_amdgcn_cvt_pk_bf8_f32(q[0], q[1], 0, false);
        w[h] = __builtin_amdgcn_cvt_pk_bf8_f32(q[2], q[3], w[h], true);
      }
    } else {
#pragma unroll
      for (int k = 0; k < 8; ++k) w[k / 4] |= code8(v[k], scale) << (8 * (k % 4));
    }
    reinterpret_cast<u32x2*>(codes)[i] = u32x2{w[0], w[1]};
  }
  if (blockIdx.x == 0 && threadIdx.x < n % 8) {
    const size_t i = n8 * 8 + threadIdx.x;
    const float v = IN == IN_F32    ? static_cast<const float*>(x)[i]
                    : IN == IN_BF16 ? __uint_as_float((u32) static_cast<const uint16_t*>(x)[i] << 16)
                                    : (float)static_cast<const _Float16*>(x)[i];
    codes[i] = (unsigned char)code8(v, scale);
  }
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

int launched(hipError_t e) { return e == hipSuccess ? G9_OK : G9_ERR_HIP; }

}  // namespace

extern "C" {

int g9_quantize_mxfp4(const void* x, int in_bits, int bf16, int64_t groups, void* packed, void* scales, void* stream) {
  if (in_bits != 16 && in_bits != 32) return G9_ERR_DTYPE;
  if (groups < 0 || groups > (int64_t(1) << 36)) return G9_ERR_SHAPE;
  if (groups == 0) return G9_OK;
  if (!x || !packed || !scales || !aligned16(x) || !aligned16(packed)) return G9_ERR_LAYOUT;
  size_t n8 = (size_t)groups * 4;
  // At most four blocks per CU, then a grid-stride loop.
  const size_t want = (n8 + kThreads - 1) / kThreads;
  const size_t blocks = want < 1024 ? want : 1024;
  u32* pk = static_cast<u32*>(packed);
  unsigned char* sc = static_cast<unsigned char*>(scales);
  void* args[] = {&x, &pk, &sc, &n8};
  const void* fn = in_bits == 32 ? reinterpret_cast<const void*>(quant_mxfp4<IN_F32>)
                   : bf16        ? reinterpret_cast<const void*>(quant_mxfp4<IN_BF16>)
                                 : reinterpret_cast<const void*>(quant_mxfp4<IN_F16>);
  return launched(hipLaunchKernel(fn, dim3((unsigned)blocks), dim3(kThreads), args, 0,
                                  reinterpret_cast<hipStream_t>(stream)));
}

int g9_quantize_e5m2(const void* x, int in_bits, int bf16, int64_t n, void* codes, void* scale, void* scratch,
                     void* stream) {
  if (in_bits != 16 && in_bits != 32) return G9_ERR_DTYPE;
  if (n <= 0) return G9_ERR_SHAPE;
  if (!x || !codes || !scale || !scratch || !aligned16(x) || !aligned16(codes)) return G9_ERR_LAYOUT;
  if (((uintptr_t)scale & 3) || ((uintptr_t)scratch & 3)) return G9_ERR_LAYOUT;
  // Four blocks per CU at most, one per 8 values of each of its threads at least.
  const size_t want = ((size_t)n / 8 + kThreads - 1) / kThreads;
  int parts = (int)(want < 1 ? 1 : want < G9_QUANT_SCRATCH_WORDS ? want : G9_QUANT_SCRATCH_WORDS);
  size_t sn = (size_t)n;
  u32* part = static_cast<u32*>(scratch);
  unsigned char* cd = static_cast<unsigned char*>(codes);
  float* so = static_cast<float*>(scale);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int in = in_bits == 32 ? IN_F32 : bf16 ? IN_BF16 : IN_F16;
  static const void* const kAmax[3] = {reinterpret_cast<const void*>(quant_amax<IN_F16>),
                                       reinterpret_cast<const void*>(quant_amax<IN_BF16>),
                                       reinterpret_cast<const void*>(quant_amax<IN_F32>)};
  static const void* const kQuant[3] = {reinterpret_cast<const void*>(quant_e5m2<IN_F16>),
                                        reinterpret_cast<const void*>(quant_e5m2<IN_BF16>),
                                        reinterpret_cast<const void*>(quant_e5m2<IN_F32>)};
  void* a1[] = {&x, &sn, &part};
  if (hipLaunchKernel(kAmax[in], dim3(parts), dim3(kThreads), a1, 0, s) != hipSuccess) return G9_ERR_HIP;
  void* a2[] = {&x, &sn, &part, &parts, &cd, &so};
  return launched(hipLaunchKernel(kQuant[in], dim3(parts), dim3(kThreads), a2, 0, s));
}

}  // extern "C"
