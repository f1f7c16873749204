// Shared device helpers for the gfx950 kernels of this library.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ffa {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr float kLog2e = 1.4426950408889634f;

// ---------------------------------------------------------------------------
// scalar conversions
// ---------------------------------------------------------------------------
__device__ __forceinline__ float bf16_bits_to_f32(uint32_t b) { return __uint_as_float(b << 16); }

__device__ __forceinline__ uint32_t f32_to_bf16_bits(float f) {
  // round-to-nearest-even, NaN kept quiet (same rule as torch's bf16 cast)
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return ((u >> 16) | 0x40u) & 0xffffu;
  u += 0x7fffu + ((u >> 16) & 1u);
  return u >> 16;
}

__device__ __forceinline__ float f16_bits_to_f32(uint32_t b) {
  return (float)__builtin_bit_cast(_Float16, (uint16_t)b);
}

__device__ __forceinline__ uint32_t f32_to_f16_bits(float f) {
  return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)f);
}

// fp16(a) in the low half and fp16(b) in the high half, each rounded to nearest even as
// f32_to_f16_bits rounds it: gfx950 converts the pair with one v_cvt_pk_f16_f32 (two conversions,
// a shift and an OR otherwise)
__device__ __forceinline__ uint32_t pk_f16_bits(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, f16x2));
}

// the same for bf16 (v_cvt_pk_bf16_f32: the bits of f32_to_bf16_bits for every input)
__device__ __forceinline__ uint32_t pk_bf16_bits(float a, float b) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, bf16x2));
}

// load element i of a float tensor of runtime dtype (0=f16, 1=bf16, 2=f32)
__device__ __forceinline__ float load_any(const void *p, size_t i, int dt) {
  if (dt == 2) return ((const float *)p)[i];
  uint32_t b = ((const uint16_t *)p)[i];
  return dt == 1 ? bf16_bits_to_f32(b) : f16_bits_to_f32(b);
}

__device__ __forceinline__ void store_any(void *p, size_t i, int dt, float v) {
  if (dt == 2) {
    ((float *)p)[i] = v;
  } else if (dt == 1) {
    ((uint16_t *)p)[i] = (uint16_t)f32_to_bf16_bits(v);
  } else {
    ((uint16_t *)p)[i] = (uint16_t)f32_to_f16_bits(v);
  }
}

// round a float to the given float dtype and back (0=f16, 1=bf16, 2=f32)
__device__ __forceinline__ float round_to(float v, int dt) {
  if (dt == 2) return v;
  if (dt == 1) return bf16_bits_to_f32(f32_to_bf16_bits(v));
  return (float)(_Float16)v;
}

// ---------------------------------------------------------------------------
// fp8 (OCP e4m3fn / e5m2) encode with torch's rules: RNE, e4m3fn overflow -> NaN, e5m2 overflow ->
// inf, a NaN's byte its sign and 0x7f.  gfx950 converts a pair with one v_cvt_pk_fp8_f32 /
// v_cvt_pk_bf8_f32; over all 2^32 fp32 patterns its bytes are these for everything but NaN inputs
// (always 0xff / 0xfe), which are put right.  A conversion in integer arithmetic from the format
// definitions is some 25 instructions an element with two branches: with it the nvfp4 quantizer of
// 20K x 1024 bf16 keys took 124.6 us a call, with this 103.8 (the 2-bit one of 32K x 1024: 337 -> 311).
// ---------------------------------------------------------------------------
template <bool E4M3>
__device__ __forceinline__ uint32_t fp8_pair_hw(float a, float b) {  // bytes of a (low) and b; NaN signs not kept
  if constexpr (E4M3) return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false) & 0xffffu;
  else return (uint32_t)__builtin_amdgcn_cvt_pk_bf8_f32(a, b, 0, false) & 0xffffu;
}
__device__ __forceinline__ uint32_t f32_to_fp8(float x, int e4m3) {
  const uint32_t u = __float_as_uint(x);
  const uint32_t b = (e4m3 ? fp8_pair_hw<true>(x, x) : fp8_pair_hw<false>(x, x)) & 0xffu;
  return (u & 0x7fffffffu) > 0x7f800000u ? ((u >> 24) & 0x80u) | 0x7fu : b;
}

// Eight floats to eight fp8 bytes in memory order.  A NaN among them (seen in the sum, which other
// than for NaNs is only a NaN for infinities of both signs) takes the element-wise conversion, which
// keeps its sign.
template <bool E4M3>
__device__ __forceinline__ uint2 f32x8_to_fp8(const float *x) {
  uint2 w;
  if constexpr (E4M3) {
    w.x = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(x[2], x[3], __builtin_amdgcn_cvt_pk_fp8_f32(x[0], x[1], 0, false), true);
    w.y = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(x[6], x[7], __builtin_amdgcn_cvt_pk_fp8_f32(x[4], x[5], 0, false), true);
  } else {
    w.x = (uint32_t)__builtin_amdgcn_cvt_pk_bf8_f32(x[2], x[3], __builtin_amdgcn_cvt_pk_bf8_f32(x[0], x[1], 0, false), true);
    w.y = (uint32_t)__builtin_amdgcn_cvt_pk_bf8_f32(x[6], x[7], __builtin_amdgcn_cvt_pk_bf8_f32(x[4], x[5], 0, false), true);
  }
  const float any = ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
  if (__builtin_isnan(any)) [[unlikely]] {
    w = make_uint2(0u, 0u);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      w.x |= f32_to_fp8(x[e], E4M3) << (8 * e);
      w.y |= f32_to_fp8(x[4 + e], E4M3) << (8 * e);
    }
  }
  return w;
}

// Eight consecutive elements of a float tensor of dtype DT (0=f16, 1=bf16, 2=f32) at an address that is
// a multiple of their size: one or two 16-byte loads, then conversions that need no dtype test.
template <int DT>
struct Raw8 {
  uint4 v[DT == 2 ? 2 : 1];
};
template <int DT>
__device__ __forceinline__ Raw8<DT> load8(const void *p, size_t i) {
  Raw8<DT> r;
  const uint4 *s = (const uint4 *)((const uint8_t *)p + i * (DT == 2 ? 4 : 2));
  r.v[0] = s[0];
  if constexpr (DT == 2) r.v[1] = s[1];
  return r;
}
template <int DT>
__device__ __forceinline__ void raw8_to_f32(const Raw8<DT> &r, float *x) {
  if constexpr (DT == 2) {
    const uint32_t w[8] = {r.v[0].x, r.v[0].y, r.v[0].z, r.v[0].w, r.v[1].x, r.v[1].y, r.v[1].z, r.v[1].w};
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = __uint_as_float(w[e]);
  } else {
    const uint32_t w[4] = {r.v[0].x, r.v[0].y, r.v[0].z, r.v[0].w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      x[2 * e] = DT == 1 ? __uint_as_float(w[e] << 16) : f16_bits_to_f32(w[e] & 0xffffu);
      x[2 * e + 1] = DT == 1 ? __uint_as_float(w[e] & 0xffff0000u) : f16_bits_to_f32(w[e] >> 16);
    }
  }
}
// eight floats rounded to dtype DT and back (the hardware's paired conversions: RNE)
template <int DT>
__device__ __forceinline__ void round8(float *x) {
  if constexpr (DT != 2) {
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      if constexpr (DT == 1) {
        const uint32_t w = pk_bf16_bits(x[e], x[e + 1]);
        x[e] = __uint_as_float(w << 16);
        x[e + 1] = __uint_as_float(w & 0xffff0000u);
      } else {
        const uint32_t w = pk_f16_bits(x[e], x[e + 1]);
        x[e] = f16_bits_to_f32(w & 0xffffu);
        x[e + 1] = f16_bits_to_f32(w >> 16);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// lane exchange
// ---------------------------------------------------------------------------
template <int CTRL>
__device__ __forceinline__ float dpp(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xF, 0xF, false));
}
constexpr int kRowRor4 = 0x124;
constexpr int kRowRor8 = 0x128;

// Lane i combined with lane i ^ m.  For m = 16 and 32 a single register-to-register exchange:
// v_permlane16_swap / v_permlane32_swap (gfx950) of x with itself leaves x_i in one result and
// x_(i^m) in the other; other distances go through __shfl_xor (an LDS-pipe permute).
template <int M>
__device__ __forceinline__ void xor_pair(float x, float &a, float &b) {
  if constexpr (M == 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
  } else if constexpr (M == 32) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
  } else {
    a = x;
    b = __shfl_xor(x, M);
  }
}
__device__ __forceinline__ float xor_max(float x, int m) {
  float a, b;
  if (m == 16) xor_pair<16>(x, a, b);
  else if (m == 32) xor_pair<32>(x, a, b);
  else { a = x; b = __shfl_xor(x, m); }
  return fmaxf(a, b);
}
__device__ __forceinline__ float xor_sum(float x, int m) {
  float a, b;
  if (m == 16) xor_pair<16>(x, a, b);
  else if (m == 32) xor_pair<32>(x, a, b);
  else { a = x; b = __shfl_xor(x, m); }
  return a + b;
}

// Whole-wave max / sum with register-to-register exchanges: lane i with i ^ 32 and i ^ 16,
// then DPP row rotations by 8, 4, 2, 1 inside each 16-lane row.  Every lane ends with the
// result.
constexpr int kRowRor1 = 0x121;
constexpr int kRowRor2 = 0x122;
__device__ __forceinline__ float wave_max(float x) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto c = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(c[0]), __uint_as_float(c[1]));
  x = fmaxf(x, dpp<kRowRor8>(x));
  x = fmaxf(x, dpp<kRowRor4>(x));
  x = fmaxf(x, dpp<kRowRor2>(x));
  return fmaxf(x, dpp<kRowRor1>(x));
}
__device__ __forceinline__ float wave_sum(float x) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto c = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(c[0]) + __uint_as_float(c[1]);
  x += dpp<kRowRor8>(x);
  x += dpp<kRowRor4>(x);
  x += dpp<kRowRor2>(x);
  return x + dpp<kRowRor1>(x);
}
// lane i + lane (i ^ 32), for every lane
__device__ __forceinline__ float swap32_sum(float x) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(a[0]) + __uint_as_float(a[1]);
}

// Raw buffer resource over [base, base + bytes) (gfx9 word 3: 32-bit data format, no
// swizzle).  A load at an offset past `bytes` returns zeros without a memory access, so a
// load group can be issued on every path with its validity carried by the size; the
// compiler then counts outstanding loads exactly and waits for one group at a time.
typedef __amdgpu_buffer_rsrc_t brsrc;
__device__ __forceinline__ brsrc make_rsrc(const void *base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ uint4 bload16(brsrc r, uint32_t off) {
  const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0);
  return make_uint4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ uint32_t bload4(brsrc r, uint32_t off) {
  return __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0);
}
__device__ __forceinline__ uint2 bload8(brsrc r, uint32_t off) {
  const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0);
  return make_uint2(v[0], v[1]);
}
__device__ __forceinline__ uint64_t bload8u(brsrc r, uint32_t off) {
  const uint2 v = bload8(r, off);
  return ((uint64_t)v.y << 32) | v.x;
}
// The same loads with the non-temporal hint (cache-policy bit 1, `nt` on gfx950), for data one
// workgroup reads once in whole cache lines per load: the paged (page, KV head) blocks of codes,
// scales, residual and V, and the contiguous layouts' V rows.  Data that several workgroups read
// keeps the default policy: q, probe windows, page ids, and the reference layout's code rows, whose
// cache lines hold several KV heads' codes; so do the other-format decoder's contiguous residual
// rows, which a wave reads in two loads of alternate 16-byte pieces of each line (with the hint, a
// load-only probe of config 1's reads took 4.55 against 4.10 us; the q2 decoder's contiguous
// residual, read for about a tenth of the chunks at config 2, measured 0.15 us slower without it).
constexpr int kNonTemporal = 2;
__device__ __forceinline__ uint4 bload16_nt(brsrc r, uint32_t off) {
  const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, kNonTemporal);
  return make_uint4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ uint2 bload8_nt(brsrc r, uint32_t off) {
  const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, kNonTemporal);
  return make_uint2(v[0], v[1]);
}
__device__ __forceinline__ uint64_t bload8u_nt(brsrc r, uint32_t off) {
  const uint2 v = bload8_nt(r, off);
  return ((uint64_t)v.y << 32) | v.x;
}

}  // namespace ffa
