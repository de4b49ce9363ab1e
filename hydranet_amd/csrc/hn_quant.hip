// INT4 dequantise and quantise kernels (gfx950).
//
// Dequantise follows the reference's dequantisers, which are bit-identical
// to one another: preprocess/pack_weights.py:230-268,
// cache/packed_expert_store.py:287-315, kernels/expert_mlp.py:305-330:
//   W[n, k] = fp16( (nibble(n, k) - 8) * scale[n, k / group] ).
// (nibble - 8) is exact in fp16 and the product is rounded once (RNE), which
// is what v_pk_mul_f16 does with fp16 denormals enabled (the gfx9 default).
//
// Quantise restates two reference quantisers in their own arithmetic:
//   mode 0  ExpertWeightPacker.quantize_tensor  (preprocess/pack_weights.py:133-181)
//   mode 1  Int4Linear.quantize_weight          (kernels/int4_linear.py:68-107)
#include "hn_common.h"

// One thread handles 32 consecutive k of one row: 16 packed bytes in,
// 32 fp16 (64 bytes) out.
__global__ __launch_bounds__(256) void hn_dequant_kernel(
    const uint8_t* __restrict__ packed, long ld_p,
    const h16* __restrict__ scales, long ld_s,
    h16* __restrict__ out, long ld_o,
    int N, int K, int group) {
  const int chunks = K >> 5;  // K % 32 == 0 checked on the host
  const long tid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (tid >= (long)N * chunks) return;
  const int n = (int)(tid / chunks);
  const int c = (int)(tid % chunks);
  const int k0 = c << 5;
  const u32x4 w = *reinterpret_cast<const u32x4*>(packed + n * ld_p + (k0 >> 1));
  const h16* srow = scales + n * ld_s;
  h16* orow = out + n * ld_o + k0;
  h16 res[32];
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    half2_t p[4];
    hn_unpack8_centered(w[d], p);
    const int kb = k0 + 8 * d;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      // p[i] = (k_i, k_{i+4}) relative to kb
      const h16 s_lo = srow[(kb + i) / group];
      const h16 s_hi = srow[(kb + i + 4) / group];
      const half2_t s2 = {s_lo, s_hi};
      const half2_t v = p[i] * s2;
      res[8 * d + i] = v[0];
      res[8 * d + i + 4] = v[1];
    }
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    u32x4 o;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      half2_t h2 = {res[8 * q + 2 * j], res[8 * q + 2 * j + 1]};
      o[j] = __builtin_bit_cast(uint32_t, h2);
    }
    *reinterpret_cast<u32x4*>(orow + 8 * q) = o;
  }
}

// fp16 -> uint8 conversion of the shifted code, as torch's CPU cast does on
// x86 for the values that occur here: exact for 0..15, and NaN (an all-zero
// group gives scale 0 and 0/0) becomes 0 (observed with torch 2.10 on x86).
__device__ __forceinline__ uint32_t hn_code_u8(float q_plus8) {
  if (!(q_plus8 == q_plus8)) return 0u;
  return (uint32_t)(int)q_plus8 & 0xFFu;
}

template <typename T>
__device__ __forceinline__ float hn_load_f(const T* p);
template <>
__device__ __forceinline__ float hn_load_f<h16>(const h16* p) { return (float)*p; }
template <>
__device__ __forceinline__ float hn_load_f<float>(const float* p) { return *p; }

// Mode 0 (ExpertWeightPacker, fp16 input, arithmetic in fp16 with fp32 opmath):
//   absmax = max |w|                      (exact)
//   s      = fp16(float(absmax) / 7.0f)   (pack_weights.py:157, scalar divisor)
//   s      = clamp(s, min=fp16(1e-10)=0)  (:158, a no-op for s >= 0)
//   q      = rint(fp16(float(w) / float(s))), clamped to [-8, 7]   (:161)
//   code   = q + 8                        (:162)
// Mode 1 (Int4Linear.quantize_weight, arithmetic in the input dtype T):
//   absmax = max(max |w|, T(1e-8))        (int4_linear.py:92)
//   s      = fp16(absmax / 7)             (:94)
//   q      = rint(T(T(w / absmax) * 7)), clamped to [-8, 7]        (:97)
template <typename T, int MODE>
__global__ __launch_bounds__(256) void hn_quantize_kernel(
    const T* __restrict__ w, long ld_w,
    uint8_t* __restrict__ packed, long ld_p,
    h16* __restrict__ scales, long ld_s,
    int N, int K, int group) {
  const int groups = K / group;
  const long tid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (tid >= (long)N * groups) return;
  const int n = (int)(tid / groups);
  const int g = (int)(tid % groups);
  const T* row = w + n * ld_w + (long)g * group;
  float amax = 0.0f;
  bool nan_seen = false;
  for (int i = 0; i < group; ++i) {
    const float v = hn_load_f<T>(row + i);
    nan_seen |= !(v == v);
    amax = fmaxf(amax, fabsf(v));
  }
  if (nan_seen) amax = __builtin_nanf("");
  float absmax_t;  // absmax in the arithmetic dtype
  h16 s16;
  if (MODE == 0) {
    absmax_t = amax;  // fp16 value, exact in float
    s16 = (h16)(absmax_t / 7.0f);
  } else {
    if (sizeof(T) == 2) {
      // clamp(min=1e-8) with the scalar cast to fp16 first: fp16(1e-8) == 0
      absmax_t = fmaxf(amax, 0.0f);
      s16 = (h16)(float)(h16)(absmax_t / 7.0f);
    } else {
      absmax_t = fmaxf(amax, 1e-8f);
      s16 = (h16)(absmax_t / 7.0f);
    }
  }
  scales[n * ld_s + g] = s16;
  const float s = (float)s16;
  uint8_t* prow = packed + n * ld_p + ((long)g * group >> 1);
  for (int i = 0; i < group; i += 2) {
    uint32_t code[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const float v = hn_load_f<T>(row + i + j);
      float q;
      if (MODE == 0) {
        q = (float)(h16)(v / s);           // fp16 tensor / fp16 tensor
      } else if (sizeof(T) == 2) {
        const float r = (float)(h16)(v / absmax_t);  // fp16 / fp16
        q = (float)(h16)(r * 7.0f);                  // fp16 * python scalar
      } else {
        q = (v / absmax_t) * 7.0f;                   // fp32 throughout
      }
      q = rintf(q);                                  // round half to even
      if (q == q) q = fminf(fmaxf(q, -8.0f), 7.0f);  // clamp keeps NaN
      if (MODE == 0) {
        code[j] = hn_code_u8(q + 8.0f);              // fp16 (q + 8) -> uint8
      } else {
        // q -> int8 first (NaN -> 0 on x86 torch), then int8 + 8 -> uint8
        code[j] = (uint32_t)(((q == q) ? (int)q : 0) + 8) & 0xFFu;
      }
    }
    prow[i >> 1] = (uint8_t)((code[1] << 4) | (code[0] & 0xFu));
  }
}

// Quantise with the rows contiguous (the usual case): a lane takes 8 consecutive
// elements (16 or 32 bytes), so L = group / 8 lanes hold a group, its absmax is a
// butterfly over them, and the eight codes leave as one dword per lane; kChunks
// such per lane, their loads in flight together.  Every access is coalesced and
// read once (one thread per group, as the general kernel below, read each
// group twice, an element at a time: fp16 14336 x 4096, 1108 us against 33, which
// is 4.5 TB/s of the 117 MB read and 31 MB written).
// fp16 quotients: v and d are fp16 values (11-bit significands), and fl32(v / d)
// comes exactly from one Newton step on v * rcp(d): the quotient of two 11-bit
// integers is at least 2^-36 (relative) away from any midpoint of two fp32 values it
// is not equal to, and q0 + (v - q0 d) rcp(d) is within 2^-44 before its single
// rounding (v - q0 d is exact in the fma).  Divisors that are not finite and
// positive take the plain division.  fp32 inputs always do.
constexpr int kChunks = 4;

template <typename T> struct QLoad;
template <> struct QLoad<h16> {
  u32x4 a;
  __device__ void load(const h16* p) { a = *reinterpret_cast<const u32x4*>(p); }
  __device__ float at(int i) const {
    return (float)__builtin_bit_cast(h16, (uint16_t)(a[i >> 1] >> (16 * (i & 1))));
  }
  // max over the 8 elements of the bits without the sign: NaN above infinity
  __device__ uint32_t amax() const {
    uint32_t m = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) m = max(m, (a[i >> 1] >> (16 * (i & 1))) & 0x7fffu);
    return m;
  }
  static __device__ float value(uint32_t bits) {
    return (float)__builtin_bit_cast(h16, (uint16_t)bits);
  }
};
template <> struct QLoad<float> {
  u32x4 a, b;
  __device__ void load(const float* p) {
    a = *reinterpret_cast<const u32x4*>(p);
    b = *reinterpret_cast<const u32x4*>(p + 4);
  }
  __device__ float at(int i) const { return __builtin_bit_cast(float, i < 4 ? a[i & 3] : b[i & 3]); }
  __device__ uint32_t amax() const {
    uint32_t m = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) m = max(m, max(a[i] & 0x7fffffffu, b[i] & 0x7fffffffu));
    return m;
  }
  static __device__ float value(uint32_t bits) { return __builtin_bit_cast(float, bits); }
};

// The codes of 8 elements against divisor d (the scale in mode 0, the absmax in
// mode 1), nibble i = element i.
template <typename T, int MODE, bool FAST>
__device__ __forceinline__ uint32_t quant8(const QLoad<T>& v, float d) {
  const float rd = FAST ? __builtin_amdgcn_rcpf(d) : 0.f;
  uint32_t word = 0;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float x = v.at(i);
    float r;
    if (FAST) {
      const float q0 = x * rd;
      r = __builtin_fmaf(__builtin_fmaf(-q0, d, x), rd, q0);
    } else {
      r = x / d;
    }
    float q;
    if (MODE == 0) q = (float)(h16)r;                                     // fp16 / fp16
    else if (sizeof(T) == 2) q = (float)(h16)((float)(h16)r * 7.0f);      // fp16, then * 7
    else q = r * 7.0f;                                                    // fp32 throughout
    q = rintf(q);
    if (!FAST) {
      if (q == q) q = fminf(fmaxf(q, -8.0f), 7.0f);
      const uint32_t c = MODE == 0 ? hn_code_u8(q + 8.0f)
                                   : (uint32_t)(((q == q) ? (int)q : 0) + 8) & 0xFFu;
      word |= (c & 0xFu) << (4 * i);
    } else {
      q = fminf(fmaxf(q, -8.0f), 7.0f);
      word |= (uint32_t)((int)q + 8) << (4 * i);
    }
  }
  return word;
}

template <typename T, int MODE>
__global__ __launch_bounds__(256) void hn_quantize_rows_kernel(
    const T* __restrict__ w, uint32_t* __restrict__ packed, h16* __restrict__ scales, long chunks,
    int lshift) {
  const long base = (long)blockIdx.x * (256 * kChunks) + threadIdx.x;
  QLoad<T> v[kChunks];
#pragma unroll
  for (int u = 0; u < kChunks; ++u) v[u].load(w + 8 * min(base + 256 * u, chunks - 1));
#pragma unroll
  for (int u = 0; u < kChunks; ++u) {
    const long c = base + 256 * u;
    uint32_t m = v[u].amax();
    for (int off = (1 << lshift) >> 1; off > 0; off >>= 1)
      m = max(m, (uint32_t)__shfl_xor((int)m, off, 64));
    const float amax = QLoad<T>::value(m);
    float d;
    h16 s16;
    if (MODE == 0) {
      s16 = (h16)(amax / 7.0f);
      d = (float)s16;
    } else {
      // clamp(min=1e-8): 0 in fp16
      d = fmaxf(amax, sizeof(T) == 2 ? 0.0f : 1e-8f);
      s16 = (h16)(d / 7.0f);
    }
    uint32_t word;
    // a divisor that is zero (or whose quotients are), infinite or NaN: as the
    // plain division has it
    if (sizeof(T) == 2 && d > 0.f && d < __builtin_inff() && amax < __builtin_inff())
      word = quant8<T, MODE, true>(v[u], d);
    else
      word = quant8<T, MODE, false>(v[u], d);
    if (c < chunks) {
      packed[c] = word;
      if ((c & ((1 << lshift) - 1)) == 0) scales[c >> lshift] = s16;
    }
  }
}

extern "C" int hn_int4_dequant(const void* packed, long ld_p, const void* scales, long ld_s,
                               void* out, long ld_o, long N, long K, long group,
                               void* stream) {
  HN_ARG_CHECK(N >= 0 && K >= 0, "hn_int4_dequant: negative dims");
  HN_ARG_CHECK(K % 32 == 0, "hn_int4_dequant: K=%ld must be a multiple of 32", K);
  HN_ARG_CHECK(group > 0 && K % group == 0, "hn_int4_dequant: group=%ld must divide K=%ld",
               group, K);
  HN_ARG_CHECK(((uintptr_t)packed % 16 == 0) && (ld_p % 16 == 0),
               "hn_int4_dequant: packed rows must be 16-byte aligned");
  HN_ARG_CHECK(((uintptr_t)out % 16 == 0) && (ld_o % 8 == 0),
               "hn_int4_dequant: output rows must be 16-byte aligned");
  if (N == 0 || K == 0) return 0;
  const long threads = N * (K / 32);
  hipLaunchKernelGGL(hn_dequant_kernel, dim3(hn_cdiv(threads, 256)), dim3(256), 0,
                     (hipStream_t)stream, (const uint8_t*)packed, ld_p, (const h16*)scales,
                     ld_s, (h16*)out, ld_o, (int)N, (int)K, (int)group);
  HN_LAUNCH_CHECK("hn_int4_dequant");
  return 0;
}

// dtype: 0 = fp16 input, 1 = fp32 input.  mode: 0 = expert packer, 1 = Int4Linear.
extern "C" int hn_int4_quantize(const void* w, long ld_w, int dtype, int mode, void* packed,
                                long ld_p, void* scales, long ld_s, long N, long K, long group,
                                void* stream) {
  HN_ARG_CHECK(N >= 0 && K >= 0, "hn_int4_quantize: negative dims");
  HN_ARG_CHECK(group > 0 && group % 2 == 0 && K % group == 0,
               "hn_int4_quantize: group=%ld must be even and divide K=%ld", group, K);
  HN_ARG_CHECK(dtype == 0 || dtype == 1, "hn_int4_quantize: dtype must be 0 (fp16) or 1 (fp32)");
  HN_ARG_CHECK(mode == 0 || mode == 1, "hn_int4_quantize: mode must be 0 or 1");
  HN_ARG_CHECK(!(mode == 0 && dtype == 1),
               "hn_int4_quantize: the expert packer takes fp16 weights (loaders cast to fp16)");
  if (N == 0 || K == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  // contiguous rows, groups of 8 to 512 elements in whole lanes of 8: the
  // coalesced kernel; anything else a thread per group
  const long lanes = group / 8, chunks = N * (K / 8);
  if (group % 8 == 0 && lanes <= 64 && (lanes & (lanes - 1)) == 0 && ld_w == K && ld_p == K / 2 &&
      ld_s == K / group && (uintptr_t)w % 16 == 0 && (uintptr_t)packed % 4 == 0 &&
      (chunks + 256 * kChunks - 1) / (256 * kChunks) < (1L << 31)) {
    int lshift = 0;
    while ((1L << lshift) < lanes) ++lshift;
    dim3 grid(hn_cdiv(chunks, 256 * kChunks)), block(256);
    if (dtype == 0 && mode == 0)
      hipLaunchKernelGGL((hn_quantize_rows_kernel<h16, 0>), grid, block, 0, s, (const h16*)w,
                         (uint32_t*)packed, (h16*)scales, chunks, lshift);
    else if (dtype == 0)
      hipLaunchKernelGGL((hn_quantize_rows_kernel<h16, 1>), grid, block, 0, s, (const h16*)w,
                         (uint32_t*)packed, (h16*)scales, chunks, lshift);
    else
      hipLaunchKernelGGL((hn_quantize_rows_kernel<float, 1>), grid, block, 0, s, (const float*)w,
                         (uint32_t*)packed, (h16*)scales, chunks, lshift);
    HN_LAUNCH_CHECK("hn_int4_quantize");
    return 0;
  }
  const long threads = N * (K / group);
  dim3 grid(hn_cdiv(threads, 256)), block(256);
  if (dtype == 0 && mode == 0)
    hipLaunchKernelGGL((hn_quantize_kernel<h16, 0>), grid, block, 0, s, (const h16*)w, ld_w,
                       (uint8_t*)packed, ld_p, (h16*)scales, ld_s, (int)N, (int)K, (int)group);
  else if (dtype == 0)
    hipLaunchKernelGGL((hn_quantize_kernel<h16, 1>), grid, block, 0, s, (const h16*)w, ld_w,
                       (uint8_t*)packed, ld_p, (h16*)scales, ld_s, (int)N, (int)K, (int)group);
  else
    hipLaunchKernelGGL((hn_quantize_kernel<float, 1>), grid, block, 0, s, (const float*)w,
                       ld_w, (uint8_t*)packed, ld_p, (h16*)scales, ld_s, (int)N, (int)K,
                       (int)group);
  HN_LAUNCH_CHECK("hn_int4_quantize");
  return 0;
}
