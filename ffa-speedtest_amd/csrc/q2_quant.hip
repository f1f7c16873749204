// 2-bit K quantizers and the fused K-projection + RoPE producers for gfx950.
//
//  * per-channel quantizer, bit-exact with the reference's torch op sequence
//    (ffa-q2fp8/run_attn_bench_q2.py:78-105): every op that torch runs in the
//    K dtype tau is rounded to tau here; no FMA contraction (the file is built
//    with `fp contract(off)`); divisions are IEEE round-to-nearest.
//  * fused K-proj + RoPE (ffa-q2fp8/fused_kproj_rope_q2fp8.py:103-399, which
//    runs the GEMM twice): one MFMA GEMM pass writes the rotated K, then the
//    per-channel quantizer runs on it.
//  * fused K-proj + RoPE + g32 quantize + append into the paged cache
//    (the decode-time producer): per-token groups make the append local, so GEMM,
//    RoPE, quantization and the page writes are one kernel.
#include "decode_common.h"
#include "ffa_common.h"
#include "ffa_mi355x.h"
#include "page_tile.h"

#include <stdio.h>
#include <type_traits>

#pragma clang fp contract(off)

namespace ffa {

// ---------------------------------------------------------------------------
// per-channel quantizer
// ---------------------------------------------------------------------------
constexpr int kQTok = 256;  // tokens per min/max split

__global__ __launch_bounds__(256) void q2_minmax_kernel(const void *k, int kdt, int T, int C, int nsplit,
                                                         float *minmax) {
  // grid (nsplit, B, ceil(C/256)); thread = column
  const int split = blockIdx.x, b = blockIdx.y;
  const int c = blockIdx.z * 256 + threadIdx.x;
  if (c >= C) return;
  const int tper = (T + nsplit - 1) / nsplit;
  const int ta = split * tper, tb = min(T, ta + tper);
  float mn = INFINITY, mx = -INFINITY;
  for (int t = ta; t < tb; ++t) {
    const float v = load_any(k, ((size_t)b * T + t) * C + c, kdt);
    mn = fminf(mn, v);
    mx = fmaxf(mx, v);
  }
  const int B = gridDim.y;
  minmax[((size_t)b * nsplit + split) * C + c] = mn;
  minmax[((size_t)(B + b) * nsplit + split) * C + c] = mx;
}

// 32 columns per workgroup, 8 threads a column: the splits' extrema are read 8 at a time instead of one
// after the other (64 splits of 1024 columns: 17.5 us as a chain of dependent reads by 4 workgroups)
__global__ __launch_bounds__(256) void q2_scale_kernel(const float *minmax, int B, int nsplit, int C, int kdt,
                                                        void *scale, void *zero) {
  const int b = blockIdx.y;
  const int col = threadIdx.x & 31, r = threadIdx.x >> 5;
  const int c = blockIdx.x * 32 + col;
  float mn = INFINITY, mx = -INFINITY;
  if (c < C) {
#pragma unroll 8
    for (int s = r; s < nsplit; s += 8) {
      mn = fminf(mn, minmax[((size_t)b * nsplit + s) * C + c]);
      mx = fmaxf(mx, minmax[((size_t)(B + b) * nsplit + s) * C + c]);
    }
  }
  __shared__ float s_m[2][8][32];
  s_m[0][r][col] = mn;
  s_m[1][r][col] = mx;
  __syncthreads();
  if (r != 0 || c >= C) return;
#pragma unroll
  for (int i = 1; i < 8; ++i) mn = fminf(mn, s_m[0][i][col]), mx = fmaxf(mx, s_m[1][i][col]);
  // scale = tau(tau(tau(max - min).clamp_min(1e-6)) / 3.0)   (run_attn_bench_q2.py:82)
  const float diff = round_to(mx - mn, kdt);
  const float cl = round_to(fmaxf(diff, 1e-6f), kdt);
  const float sc = round_to(__fdiv_rn(cl, 3.0f), kdt);
  store_any(scale, (size_t)b * C + c, kdt, sc);
  store_any(zero, (size_t)b * C + c, kdt, mn);
}

// one thread per (token, packed byte) of a [B, T, HKV, D] tensor
// One packed byte (channels 4 byte .. 4 byte + 3) of one K row under per-channel scale / zero
// (tau values at sz_off + d): codes and residuals with the reference's per-element ops.  The
// full quantizer runs it with K's own scale / zero, the per-channel append with the cache's.
__device__ __forceinline__ void quant_channel_byte(const void *k, int kdt, size_t k_row, int D, int byte,
                                                   const void *scale, const void *zero, size_t sz_off,
                                                   uint8_t *kq_byte, uint8_t *res_row, int res_e4m3) {
  uint32_t packed = 0;
  for (int e = 0; e < 4; ++e) {
    const int d = 4 * byte + e;
    if (d >= D) break;
    const float kv = load_any(k, k_row * D + d, kdt);
    const float sc = load_any(scale, sz_off + d, kdt);
    const float zr = load_any(zero, sz_off + d, kdt);
    const float xs = round_to(kv - zr, kdt);               // (k - zero) in tau
    const float xd = round_to(__fdiv_rn(xs, sc), kdt);     // / scale in tau
    const float cq = fminf(fmaxf(__builtin_rintf(xd), 0.f), 3.f);  // round (RNE), clamp(0,3)
    const float deq = (cq * sc) + zr;                      // two fp32 roundings
    res_row[d] = (uint8_t)f32_to_fp8(kv - deq, res_e4m3);
    packed |= ((uint32_t)cq) << (2 * e);
  }
  *kq_byte = (uint8_t)packed;
}

__global__ __launch_bounds__(256) void q2_quant_channel_kernel(const void *k, int kdt, int B, int T, int HKV,
                                                                int D, const void *scale, const void *zero,
                                                                uint8_t *kq, uint8_t *res, int res_e4m3) {
  const int DP = (D + 3) / 4;
  const size_t total = (size_t)B * T * HKV * DP;
  const size_t id = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (id >= total) return;
  const int byte = (int)(id % DP);
  const size_t row = id / DP;  // (b, t, hkv)
  const int hkv = (int)(row % HKV);
  const int b = (int)(row / ((size_t)HKV * T));
  quant_channel_byte(k, kdt, row, D, byte, scale, zero, ((size_t)b * HKV + hkv) * D, kq + row * DP + byte,
                     res + row * D, res_e4m3);
}

// ---- the same quantizer over vectors of 8 columns (D a multiple of 4, HKV * D a multiple of 8, aligned
// pointers): columns of a [B, T, C = HKV * D] tensor are quantized independently, so the kernels see C
// only.  Both passes are bound by reading K and writing codes and residual once; what kept the scalar
// kernels from it were 2-byte loads one after the other (minimum / maximum of 32K x 1024 bf16: 150 us)
// and, per element, an IEEE division and two roundings in software (112 us).  A call on 32K x 1024 bf16 keys
// (109 MB read and written once) took 341 us with the scalar kernels and takes 38 with these.

// Minimum and maximum per column of one split of the tokens: a workgroup covers 128 columns (256 or 512
// bytes of a row, 16 lanes), 16 token rows at a time, 8 of them in flight per lane.
constexpr int kMmCols = 128, kMmRows = 16, kMmFly = 8;
template <int KDT>
__global__ __launch_bounds__(256) void q2_minmax8_kernel(const void *k, int T, int C, int nsplit, float *minmax) {
  const int split = blockIdx.x, b = blockIdx.y, B = gridDim.y;
  const int cl = (threadIdx.x & 15) * 8, c = blockIdx.z * kMmCols + cl, r = threadIdx.x >> 4;
  const int tper = (T + nsplit - 1) / nsplit;
  const int ta = split * tper, tb = min(T, ta + tper);
  float mn[8], mx[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) mn[e] = INFINITY, mx[e] = -INFINITY;
  if (c < C) {
    for (int t = ta + r; t < tb; t += kMmRows * kMmFly) {
      Raw8<KDT> w[kMmFly];
#pragma unroll
      for (int u = 0; u < kMmFly; ++u)  // rows past the split repeat its last: no effect on an extremum
        w[u] = load8<KDT>(k, ((size_t)b * T + min(t + kMmRows * u, tb - 1)) * C + c);
#pragma unroll
      for (int u = 0; u < kMmFly; ++u) {
        float x[8];
        raw8_to_f32<KDT>(w[u], x);
#pragma unroll
        for (int e = 0; e < 8; ++e) mn[e] = fminf(mn[e], x[e]), mx[e] = fmaxf(mx[e], x[e]);
      }
    }
  }
  __shared__ float s_mn[kMmRows][kMmCols + 4], s_mx[kMmRows][kMmCols + 4];
#pragma unroll
  for (int e = 0; e < 8; ++e) s_mn[r][cl + e] = mn[e], s_mx[r][cl + e] = mx[e];
  __syncthreads();
  const int col = threadIdx.x & (kMmCols - 1), cc = blockIdx.z * kMmCols + col;
  const bool lo = threadIdx.x < kMmCols;
  float m = lo ? s_mn[0][col] : s_mx[0][col];
#pragma unroll
  for (int i = 1; i < kMmRows; ++i) m = lo ? fminf(m, s_mn[i][col]) : fmaxf(m, s_mx[i][col]);
  if (cc < C) minmax[((size_t)(lo ? b : B + b) * nsplit + split) * C + cc] = m;
}

// Smallest float x with code(x) >= i + 1 for a scale sc > 0, where code(x) = clamp(rne(tau(x / sc)), 0, 3),
// the quotient in fp32 first (one division per element in the reference, run_attn_bench_q2.py:84-85).
// The code is monotone in x, and it turns where tau(x / sc) passes 0.5, 1.5, 2.5 (ties to even: above 0.5,
// at 1.5, above 2.5), i.e. where x / sc passes the middle of the tau values around: q = 0.5 + u/2 (above),
// 1.5 - u'/2 (at or above), 2.5 + u''/2 (above), with the ulps u of tau there.  q * sc is exact in
// double, and for fp16 / bf16 the fp32 quotient does not cross q (x and sc have at most 11 bits, so x / sc
// is q or at least 2^-24 away from it).  A scale that is not finite gives a NaN, which no x passes, as
// x / inf = 0 and inf / inf = NaN take code 0.
template <int KDT>
__device__ __forceinline__ float q2_turn(float sc, int i) {
  constexpr int p = KDT == 2 ? 24 : (KDT == 1 ? 8 : 11);  // significant bits of tau
  constexpr double h = 1.0 / (double)(1u << p);           // an ulp of tau in [1/2, 1)
  const double q = i == 0 ? 0.5 + 0.5 * h : (i == 1 ? 1.5 - h : 2.5 + 2.0 * h);
  const double v = (double)sc * q;
  float f = (float)v;
  const bool up = i == 1 ? (double)f < v : (double)f <= v;
  if (up) f = __uint_as_float(__float_as_uint(f) + 1u);
  return sc < INFINITY ? f : __builtin_nanf("");
}

// Codes and residual: a lane keeps the scale, zero point and the three turning points of its 8 columns and
// walks down the tokens, so an element costs a subtraction, a rounding, three compares and half an fp8
// conversion.  A wave reads 64 consecutive vectors (1 or 2 KB) and writes 512 residual and 128 code bytes.
template <int KDT, bool E4M3>
__global__ __launch_bounds__(256) void q2_quant8_kernel(const void *k, int T, int C, int lw, int per, const void *scale,
                                                        const void *zero, uint8_t *kq, uint8_t *res) {
  const int b = blockIdx.z;
  const int chunk = (blockIdx.y << lw) + (threadIdx.x & ((1 << lw) - 1));
  const int rows = 256 >> lw, c = chunk * 8;
  if (c >= C) return;
  float sc[8], zr[8], turn[3][8];
  raw8_to_f32<KDT>(load8<KDT>(scale, (size_t)b * C + c), sc);
  raw8_to_f32<KDT>(load8<KDT>(zero, (size_t)b * C + c), zr);
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int e = 0; e < 8; ++e) turn[i][e] = q2_turn<KDT>(sc[e], i);
  const int ta = blockIdx.x * per, tb = min(T, ta + per);
  constexpr int kFly = KDT == 2 ? 2 : 4;  // token rows in flight per lane
  for (int t = ta + (threadIdx.x >> lw); t < tb; t += rows * kFly) {
    Raw8<KDT> w[kFly];
#pragma unroll
    for (int u = 0; u < kFly; ++u) w[u] = load8<KDT>(k, ((size_t)b * T + min(t + rows * u, tb - 1)) * C + c);
#pragma unroll
    for (int u = 0; u < kFly; ++u) {
      if (t + rows * u >= tb) break;
      float kv[8], xs[8], d[8];
      raw8_to_f32<KDT>(w[u], kv);
#pragma unroll
      for (int e = 0; e < 8; ++e) xs[e] = kv[e] - zr[e];  // (k - zero) in tau
      round8<KDT>(xs);
      uint32_t packed = 0;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const uint32_t cq = xs[e] >= turn[2][e] ? 3u : (xs[e] >= turn[1][e] ? 2u : (xs[e] >= turn[0][e] ? 1u : 0u));
        d[e] = kv[e] - ((float)cq * sc[e] + zr[e]);  // two fp32 roundings of the dequantized value
        packed |= cq << (2 * e);
      }
      const size_t row = (size_t)b * T + t + rows * u;
      *(uint2 *)(res + row * C + c) = f32x8_to_fp8<E4M3>(d);
      *(uint16_t *)(kq + row * (C >> 2) + 2 * chunk) = (uint16_t)packed;
    }
  }
}

// Reference-layout append: token n of sequence b (k_new [B, Tn, HKV, D]) is quantized with the
// cache's per-channel scale / zero [B, HKV, D] and written at position pos[b] + n of
// k_q [B, T_cap, HKV, ceil(D/4)] and residual [B, T_cap, HKV, D]; positions outside
// [0, T_cap) are not written.
__global__ __launch_bounds__(256) void q2_append_channel_kernel(const void *k_new, int kdt, int B, int Tn, int HKV,
                                                                 int D, const int32_t *pos, int T_cap,
                                                                 const void *scale, const void *zero, uint8_t *kq,
                                                                 uint8_t *res, int res_e4m3) {
  const int DP = (D + 3) / 4;
  const size_t total = (size_t)B * Tn * HKV * DP;
  const size_t id = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (id >= total) return;
  const int byte = (int)(id % DP);
  const size_t row = id / DP;  // (b, n, hkv) of k_new
  const int hkv = (int)(row % HKV);
  const int n = (int)((row / HKV) % Tn);
  const int b = (int)(row / ((size_t)HKV * Tn));
  const int t = pos[b] + n;
  if (t < 0 || t >= T_cap) return;
  const size_t dst = ((size_t)b * T_cap + t) * HKV + hkv;
  quant_channel_byte(k_new, kdt, row, D, byte, scale, zero, ((size_t)b * HKV + hkv) * D, kq + dst * DP + byte,
                     res + dst * D, res_e4m3);
}

// K projection GEMM tile: 16 tokens x 32 output channels per 512-thread workgroup.  The 32-wide k
// steps are dealt round-robin to the 8 waves (wave w takes steps w, w + 8, ...), so even a handful of
// tokens keeps 8 waves per tile streaming W; each wave accumulates its steps with MFMA 16x16x32 into
// two 16x16 tiles, and the 8 partial tiles are summed in wave order through LDS, so the result does
// not depend on timing.  Returns the fp32 product for row threadIdx.x >> 5 (token m0 + row) and
// column threadIdx.x & 31 (output channel n0 + column).  w is [N, H] (out, in), rows of H elements.
// ---------------------------------------------------------------------------
constexpr int kKpWaves = 8;

template <int HDT>
__device__ __forceinline__ f32x4 kp_mfma(uint4 a, uint4 b, f32x4 c) {
  const u32x4 av = {a.x, a.y, a.z, a.w}, bv = {b.x, b.y, b.z, b.w};
  if constexpr (HDT == FFA_DT_BF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, av), __builtin_bit_cast(bf16x8, bv), c,
                                                   0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, av), __builtin_bit_cast(f16x8, bv), c, 0,
                                                  0, 0);
}

// Operand loads read 4 lanes per row (lane L: row L >> 2, 16-byte piece L & 3 of the step's
// 64 bytes), so a 16-lane quarter of the wave touches 4 rows; the MFMA layout (lane L: row
// L & 15, piece L >> 4) puts 16 rows in each quarter, which the memory pipeline serves about
// twice as slowly.  A cross-lane permute then moves each piece to its MFMA lane.
__device__ __forceinline__ uint4 kp_to_mfma_layout(uint4 v) {
  const int lane = threadIdx.x & 63;
  const int src = (4 * (lane & 15) + (lane >> 4)) << 2;  // byte address of the source lane
  return make_uint4((uint32_t)__builtin_amdgcn_ds_bpermute(src, (int)v.x),
                    (uint32_t)__builtin_amdgcn_ds_bpermute(src, (int)v.y),
                    (uint32_t)__builtin_amdgcn_ds_bpermute(src, (int)v.z),
                    (uint32_t)__builtin_amdgcn_ds_bpermute(src, (int)v.w));
}

// NB k steps of one wave: all 3 * NB loads are issued before the first MFMA waits.  The column tiles of an XCD begin at
// different steps, a quarter of the batch apart: the rows' pitch is a power of two as a rule, and workgroups that walk
// it in step ask the same few L2 channels at a time (16 layers with the append, 1024 channels: 64 tokens of H = 2048
// 167 -> 153 us, of H = 4096 227 -> 225, 256 tokens 403 -> 361; another start for each wave, which parts the
// neighbours that share 128-byte lines, is slower).  The start depends on the output channels alone: with the token
// tile in it as well 64 tokens of H = 4096 took 214, but a token's sums then depend on its row of the batch, and so
// do its bytes in the cache.
template <int NB, int HDT, bool kFirst>
__device__ __forceinline__ void kp_steps(const uint16_t *hp, const uint16_t *wp0, const uint16_t *wp1, int wv, int i,
                                         int xcol, f32x4 &acc0, f32x4 &acc1) {
  uint4 a[NB], b0[NB], b1[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int k0 = 32 * (wv + kKpWaves * (i + (kFirst ? j : (j + NB / 4 * xcol) & (NB - 1))));
    a[j] = *(const uint4 *)(hp + k0);
    b0[j] = *(const uint4 *)(wp0 + k0);
    b1[j] = *(const uint4 *)(wp1 + k0);
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const uint4 aj = kp_to_mfma_layout(a[j]);
    acc0 = kp_mfma<HDT>(aj, kp_to_mfma_layout(b0[j]), acc0);
    acc1 = kp_mfma<HDT>(aj, kp_to_mfma_layout(b1[j]), acc1);
  }
}

template <int HDT>
__device__ __forceinline__ float kproj_tile32(const void *h, const void *w, int M, int H, int m0, int n0,
                                              float (*red)[16][33]) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  // load layout: lane L reads row L >> 2, elements 8 (L & 3) .. + 8 of each 32-wide k step
  const int mrow = min(m0 + (lane >> 2), M - 1);
  const int kq = 8 * (lane & 3);
  const uint16_t *hp = (const uint16_t *)h + (size_t)mrow * H + kq;
  const uint16_t *wp0 = (const uint16_t *)w + (size_t)(n0 + (lane >> 2)) * H + kq;
  const uint16_t *wp1 = wp0 + (size_t)16 * H;
  f32x4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
  const int nsteps = H / 32;
  const int mine = (nsteps - wv + kKpWaves - 1) / kKpWaves;  // steps of this wave (16 at H = 4096)
  const int xcol = n0 >> 8;  // which of its XCD's column tiles (they go round-robin to the 8 XCDs)
  // the first column tile of an XCD begins at step 0: addresses without arithmetic (1024 x 4096 -> 64 10.1 -> 9.7 us)
  auto steps = [&](auto first) {
    constexpr bool kFirst = decltype(first)::value;
    int i = 0;
    for (; i + 16 <= mine; i += 16) kp_steps<16, HDT, kFirst>(hp, wp0, wp1, wv, i, xcol, acc0, acc1);
    for (; i + 4 <= mine; i += 4) kp_steps<4, HDT, kFirst>(hp, wp0, wp1, wv, i, xcol, acc0, acc1);
    for (; i < mine; ++i) kp_steps<1, HDT, true>(hp, wp0, wp1, wv, i, 0, acc0, acc1);
  };
  if (xcol == 0) steps(std::true_type());
  else steps(std::false_type());
  // MFMA 16x16 result: acc[u] is row 4 * (lane >> 4) + u, column lane & 15
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    red[wv][4 * (lane >> 4) + u][lane & 15] = acc0[u];
    red[wv][4 * (lane >> 4) + u][16 + (lane & 15)] = acc1[u];
  }
  __syncthreads();
  const int row = threadIdx.x >> 5, col = threadIdx.x & 31;
  float sum = red[0][row][col];
#pragma unroll
  for (int x = 1; x < kKpWaves; ++x) sum += red[x][row][col];
  return sum;
}

// blockIdx.x -> (column tile ct, token tile mt).  Workgroups go to the 8 XCDs round-robin; when the
// column tiles split evenly over the XCDs, all token tiles of one column tile run on one XCD and share
// its L2, so each slice of W is read from HBM once.
__device__ __forceinline__ void kproj_tile_of(int bid, int nct, int &ct, int &mt) {
  if ((nct & 7) == 0) {
    const int per = nct >> 3, j = bid >> 3;
    ct = (bid & 7) + 8 * (j % per);
    mt = j / per;
  } else {
    ct = bid % nct;
    mt = bid / nct;
  }
}

// g32 quantization of one (token, KV head, group) held by the 32 lanes of a half wave (lane e of the
// half holds channel 32 g + e), and its page writes:
//   zero = fp16(min), scale = fp16(max(max - zero, 1e-6) / 3), c = clamp(rne((k - zero)/scale), 0, 3),
//   residual = fp8(k - (c*scale + zero)) with two fp32 roundings;
// min / max by shuffles, 2-bit codes OR-reduced over 16 lanes, residual bytes stored by each lane.
// All 64 lanes must call it; `store` masks the writes.
__device__ __forceinline__ void g32_quantize_lanes(float x, bool store, int page, int slot, int hkv, int HKV, int g,
                                                   uint8_t *kq_pages, uint16_t *s_pages, uint16_t *z_pages,
                                                   uint8_t *r_pages, int res_e4m3) {
  constexpr int D = 128;
  const int e = threadIdx.x & 31;
  float mn = x, mx = x;
#pragma unroll
  for (int m = 1; m < 32; m <<= 1) {
    mn = fminf(mn, __shfl_xor(mn, m));
    mx = fmaxf(mx, __shfl_xor(mx, m));
  }
  const float zr = (float)(_Float16)mn;
  const float sc = (float)(_Float16)__fdiv_rn(fmaxf(mx - zr, 1e-6f), 3.0f);
  const float cq = fminf(fmaxf(__builtin_rintf(__fdiv_rn(x - zr, sc)), 0.f), 3.f);
  const float deq = (cq * sc) + zr;
  const uint32_t rb = f32_to_fp8(x - deq, res_e4m3);
  uint32_t word = ((uint32_t)cq) << (2 * (e & 15));
#pragma unroll
  for (int m = 1; m < 16; m <<= 1) word |= (uint32_t)__shfl_xor((int)word, m);
  if (!store) return;
  const size_t blk = (size_t)page * HKV + hkv;
  r_pages[blk * (64 * D) + res_off(slot, 32 * g + e)] = (uint8_t)rb;
  if ((e & 15) == 0) *(uint32_t *)(kq_pages + blk * (4 * 64 * 8) + codes_off(g, slot) + 4 * (e >> 4)) = word;
  if (e == 0) {
    const int ss = 16 * (slot >> 4) + 4 * (slot & 3) + ((slot >> 2) & 3);  // tile-major scale slot
    const size_t so = blk * (4 * 64) + gscale_off(g, ss);
    s_pages[so] = (uint16_t)f32_to_f16_bits(sc);
    z_pages[so] = (uint16_t)f32_to_f16_bits(zr);
  }
}

// RoPE of one element given its pair partner (fused_kproj_rope_q2fp8.py:26-37):
//   out[2i]   = x[2i]  *cos[2i]   + (-x[2i+1])*sin[2i]
//   out[2i+1] = x[2i+1]*cos[2i+1] +   x[2i]   *sin[2i+1]
// each product and the sum are rounded to the promoted dtype `odt`.
__device__ __forceinline__ float rope_one(float x, float partner, bool odd, float c, float s, int odt) {
  const float t1 = round_to(x * c, odt);
  const float rot = odd ? partner : -partner;
  const float t2 = round_to(rot * s, odt);
  return round_to(t1 + t2, odt);
}

// Rotated K of the reference producer -> k_scratch [M, N] in dtype odt.  One 512-thread workgroup per
// (16 tokens, 32 output channels); grid = (N / 32) * ceil(M / 16).
template <int HDT>
__global__ __launch_bounds__(512) void kproj_rope_kernel(const void *h, const void *w, const void *bias, const void *cos,
                                                         const void *sin, int csdt, int M, int T, int H, int N, int D,
                                                         void *kout, int odt) {
  __shared__ float red[kKpWaves][16][33];
  int ct, mt;
  kproj_tile_of(blockIdx.x, N / 32, ct, mt);
  const int m0 = mt * 16, n0 = ct * 32;
  const float acc = kproj_tile32<HDT>(h, w, M, H, m0, n0, red);
  const int m = m0 + (threadIdx.x >> 5), col = n0 + (threadIdx.x & 31);
  const float bv = bias ? load_any(bias, col, HDT) : 0.f;
  const float x = round_to(acc + bv, HDT);  // F.linear output in the h dtype
  const float partner = __shfl_xor(x, 1);   // channel col ^ 1 (D is even, so the RoPE pair)
  if (m < M) {
    const int d = col % D, t = m % T;
    const float c = load_any(cos, (size_t)t * D + d, csdt);
    const float s = load_any(sin, (size_t)t * D + d, csdt);
    store_any(kout, (size_t)m * N + col, odt, rope_one(x, partner, (d & 1) != 0, c, s, odt));
  }
}

// The same for many tokens: a tile of TM tokens x TN output channels per 256-thread workgroup, operands
// staged through LDS.  (The kernel above keeps few tokens' W stream spread over the chip; with many it
// reads h and W from the caches once per 32 channels and 16 tokens: 4096 tokens x 4096 -> 1024 take 249 us
// there and 53 here, 0.65 PFLOP/s; the matrix cores need 23 at the rate a large product reaches.  What is
// left: of a wave's 104 K cycles over 64 steps 33 K are products, LDS is busy for another 33 K with 96 KB a
// step, partly under them (no bank conflicts), and a wave has its SIMD to itself, so that every wait shows;
// 8 us are the first loads and the end.)
//   * Four waves in 2 x 2 quarters; MFMA rows are channels and columns are tokens, so that a lane ends with
//     four consecutive channels of one token: RoPE pairs need no exchange, stores are 16 bytes (fp32).
//   * K in steps of 64: 16-byte pieces go to registers four steps ahead and to one of three LDS buffers two
//     steps ahead, one barrier a step; a step's operands are read under the products before them (with two
//     buffers, and the reads and writes between the products, 57 us).  A row's eight pieces are stored at
//     piece ^ (row & 7), so that the 16 rows an operand read touches spread over the banks (no conflicts).
//   * Accumulators are folded into a second set every eighth of K (512 of it at most): chains as long as the
//     split over eight waves gives, and its rounding error (fp16 values that round otherwise than the 64-bit
//     product, 4096 tokens: H = 1024 7.2e-4 of them with the split, 7.3e-4 here; H = 2048 9.4e-4 both, where
//     folds every 512 gave 11.5e-4; H = 4096 12.3e-4 and 12.4e-4).
//   * Workgroups go round-robin to the 8 XCDs; each XCD takes a run of consecutive tiles, channel tiles
//     fastest, so that its L2 serves a tile row's tokens to every channel tile.
constexpr int kGemmK = 64, kGemmMinH = 1024;

template <int HDT, bool CS32, int TM, int TN>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1))) void kproj_rope_tile_kernel(
    const void *h, const void *w, const void *bias, const void *cos, const void *sin, int M, int T, int H, int N, int D,
    void *kout) {
  constexpr int kRow = kGemmK * 2;                    // bytes of a staged row
  constexpr int kPa = TN * 8 / 256, kPb = TM * 8 / 256;  // 16-byte pieces per thread and step: W, h
  constexpr int kMi = TN / 32, kNi = TM / 32;         // MFMA tiles of a wave: channels, tokens
  constexpr int kBuf = (TM + TN) * kRow;
  __shared__ __attribute__((aligned(16))) uint8_t s_t[3 * kBuf];
  const int nct = (N + TN - 1) / TN;
  int tile = blockIdx.x;
  if ((gridDim.x & 7) == 0) tile = (int)(blockIdx.x & 7) * (int)(gridDim.x >> 3) + (int)(blockIdx.x >> 3);
  const int n0 = (tile % nct) * TN, m0 = (tile / nct) * TM;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int wn = (wv & 1) * (TN / 2), wm = (wv >> 1) * (TM / 2);

  // pieces of this thread: piece i of an operand is row (threadIdx.x + 256 i) / 8, 16-byte column % 8; rows
  // past the end read zeros (never stored)
  const int pr = threadIdx.x >> 3, pc = threadIdx.x & 7;
  const brsrc rw = make_rsrc((const uint16_t *)w + (size_t)n0 * H, (uint32_t)(min(TN, N - n0) * H * 2));
  const brsrc rh = make_rsrc((const uint16_t *)h + (size_t)m0 * H, (uint32_t)(min(TM, M - m0) * H * 2));
  const uint32_t src = (uint32_t)(pr * H * 2 + pc * 16), src32 = (uint32_t)(64 * H);  // bytes of 32 rows
  const uint32_t dst = (uint32_t)(pr * kRow + ((pc ^ (pr & 7)) * 16));  // + 32 rows per piece (32 is a multiple of 8)
  u32x4 a0[kPa], b0[kPb], a1[kPa], b1[kPb];  // steps of even and odd number
  const int steps = H / kGemmK;
  auto fetch = [&](u32x4(&a)[kPa], u32x4(&b)[kPb], int step) {
    const int k = min(step, steps - 1) * kRow;
#pragma unroll
    for (int i = 0; i < kPa; ++i) a[i] = __builtin_amdgcn_raw_buffer_load_b128(rw, (int)(src + src32 * i), k, 0);
#pragma unroll
    for (int i = 0; i < kPb; ++i) b[i] = __builtin_amdgcn_raw_buffer_load_b128(rh, (int)(src + src32 * i), k, 0);
  };
  auto stage = [&](const u32x4(&a)[kPa], const u32x4(&b)[kPb], uint8_t *to) {
#pragma unroll
    for (int i = 0; i < kPa; ++i) *(u32x4 *)(to + dst + 32 * kRow * i) = a[i];
#pragma unroll
    for (int i = 0; i < kPb; ++i) *(u32x4 *)(to + TN * kRow + dst + 32 * kRow * i) = b[i];
  };
  // LDS traffic only (lgkmcnt 0, the loads of later steps stay in flight), and with the builtin wait, so
  // that the compiler counts on from it
  auto lds_barrier = []() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  f32x4 acc[kMi][kNi], sum[kMi][kNi];
#pragma unroll
  for (int i = 0; i < kMi; ++i)
#pragma unroll
    for (int j = 0; j < kNi; ++j) acc[i][j] = sum[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int fr = lane & 15, fq = lane >> 4;
  const uint32_t fo[2] = {(uint32_t)((fq ^ (fr & 7)) * 16), (uint32_t)(((4 + fq) ^ (fr & 7)) * 16)};
  uint4 fa[2][kMi], fb[2][kNi];  // operands of the two 32-wide halves of a step
  auto read = [&](int kk, const uint8_t *from) {
    const uint8_t *ta = from + (wn + fr) * kRow + fo[kk], *tb = from + TN * kRow + (wm + fr) * kRow + fo[kk];
#pragma unroll
    for (int i = 0; i < kMi; ++i) fa[kk][i] = *(const uint4 *)(ta + 16 * kRow * i);
#pragma unroll
    for (int j = 0; j < kNi; ++j) fb[kk][j] = *(const uint4 *)(tb + 16 * kRow * j);
  };
  auto product = [&](int kk) {
#pragma unroll
    for (int i = 0; i < kMi; ++i)
#pragma unroll
      for (int j = 0; j < kNi; ++j) acc[i][j] = kp_mfma<HDT>(fa[kk][i], fb[kk][j], acc[i][j]);
  };
  auto fold = [&]() {
#pragma unroll
    for (int i = 0; i < kMi; ++i)
#pragma unroll
      for (int j = 0; j < kNi; ++j) {
        sum[i][j] += acc[i][j];
        acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
  };
  // one step: its first half's operands are in registers; the second half's are read and step + 2 is staged
  // under the first half's products, the next step's first half is read under the second's
  uint8_t *cur = s_t, *nxt = s_t + kBuf, *free = s_t + 2 * kBuf;
  auto step = [&](u32x4(&a)[kPa], u32x4(&b)[kPb], int i) {
    read(1, cur);
    __builtin_amdgcn_sched_barrier(0);
    stage(a, b, free);  // step i + 2, into the buffer step i - 1 was read from
    product(0);
#pragma unroll
    for (int g = 0; g < kPa + kPb; ++g) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // a product,
      __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);  // a staging write
    }
    __builtin_amdgcn_sched_barrier(0);
    read(0, nxt);
    fetch(a, b, i + 4);
    product(1);
#pragma unroll
    for (int g = 0; g < kMi + kNi; ++g) {
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // an operand read,
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // a product
    }
#pragma unroll
    for (int g = 0; g < kPa + kPb; ++g) {
      __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // a load,
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // a product
    }
    lds_barrier();
    uint8_t *t = cur;
    cur = nxt, nxt = free, free = t;
  };
  fetch(a0, b0, 0);
  fetch(a1, b1, 1);
  __builtin_amdgcn_sched_barrier(0);
  stage(a0, b0, cur);
  fetch(a0, b0, 2);
  __builtin_amdgcn_sched_barrier(0);
  stage(a1, b1, nxt);
  fetch(a1, b1, 3);
  lds_barrier();
  read(0, cur);
  const int fold_mask = steps >= 64 ? 7 : (steps >= 32 ? 3 : 1);  // steps of a chain, less one
  int i = 0;
  for (; i + 1 < steps; i += 2) {
    step(a0, b0, i);
    step(a1, b1, i + 1);
    if (((i + 2) & fold_mask) == 0) fold();
  }
  if (i < steps) step(a0, b0, i);
  fold();

  // bias, rounding to the h dtype (F.linear's output), RoPE, store: channels n .. n + 3 of token m (D and
  // n are multiples of 4, so the four lie within a head and their angles are one vector)
  constexpr int ODT = CS32 ? FFA_DT_F32 : HDT;
  auto load4 = [](const void *p, size_t i, float *x) {
    if constexpr (CS32) {
      const float4 v = *(const float4 *)((const float *)p + i);
      x[0] = v.x, x[1] = v.y, x[2] = v.z, x[3] = v.w;
    } else {
      const uint2 v = *(const uint2 *)((const uint16_t *)p + i);
      const uint32_t b[4] = {v.x & 0xffffu, v.x >> 16, v.y & 0xffffu, v.y >> 16};
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = HDT == FFA_DT_BF16 ? bf16_bits_to_f32(b[e]) : f16_bits_to_f32(b[e]);
    }
  };
#pragma unroll
  for (int i = 0; i < kMi; ++i) {
    const int n = n0 + wn + 16 * i + 4 * fq;
    if (n >= N) continue;
    float bv[4] = {0.f, 0.f, 0.f, 0.f};
    if (bias != nullptr)
#pragma unroll
      for (int e = 0; e < 4; ++e) bv[e] = load_any(bias, n + e, HDT);
    const int d = n % D;
#pragma unroll
    for (int j = 0; j < kNi; ++j) {
      const int m = m0 + wm + 16 * j + fr;
      if (m >= M) continue;
      float c[4], sn[4], o[4];
      load4(cos, (size_t)(m % T) * D + d, c);
      load4(sin, (size_t)(m % T) * D + d, sn);
#pragma unroll
      for (int e = 0; e < 4; e += 2) {
        const float x0 = round_to(sum[i][j][e] + bv[e], HDT), x1 = round_to(sum[i][j][e + 1] + bv[e + 1], HDT);
        o[e] = rope_one(x0, x1, false, c[e], sn[e], ODT);
        o[e + 1] = rope_one(x1, x0, true, c[e + 1], sn[e + 1], ODT);
      }
      const size_t at = (size_t)m * N + n;
      if constexpr (CS32)
        *(float4 *)((float *)kout + at) = make_float4(o[0], o[1], o[2], o[3]);
      else if constexpr (HDT == FFA_DT_BF16)
        *(uint2 *)((uint16_t *)kout + at) = make_uint2(f32_to_bf16_bits(o[0]) | (f32_to_bf16_bits(o[1]) << 16),
                                                       f32_to_bf16_bits(o[2]) | (f32_to_bf16_bits(o[3]) << 16));
      else
        *(uint2 *)((uint16_t *)kout + at) = make_uint2(pk_f16_bits(o[0], o[1]), pk_f16_bits(o[2], o[3]));
    }
  }
}

// K-proj + RoPE (fp32 cos/sin rows per token) + g32 quantize + paged append; the 32 channels of a
// workgroup are one g32 group of one KV head, so quantization needs no other workgroup.
template <int HDT>
__global__ __launch_bounds__(512) void kproj_append_kernel(const void *h, const void *w, const void *bias,
                                                           const float *cos, const float *sin, int M, int Tn, int H,
                                                           int HKV, const int32_t *pos, const int32_t *bt, int bt_stride,
                                                           int num_pages, uint8_t *kq_pages, uint16_t *s_pages,
                                                           uint16_t *z_pages, uint8_t *r_pages, int res_e4m3,
                                                           const void *v_new, void *v_pages) {
  constexpr int D = 128;
  __shared__ float red[kKpWaves][16][33];
  int ct, mt;
  kproj_tile_of(blockIdx.x, HKV * (D / 32), ct, mt);
  const int m0 = mt * 16, n0 = ct * 32;
  const int hkv = n0 / D, g = (n0 % D) / 32;
  const int e = threadIdx.x & 31, d = 32 * g + e;
  const int m = m0 + (threadIdx.x >> 5), mc = min(m, M - 1);
  // the epilogue's inputs are fetched before the GEMM so their latency hides behind it
  const float bv = bias ? load_any(bias, n0 + e, HDT) : 0.f;
  const float cv = cos[(size_t)mc * D + d], sv = sin[(size_t)mc * D + d];
  const int b = mc / Tn, nn = mc % Tn;
  const int P = pos[b] + nn;
  const uint16_t vv = v_new != nullptr ? ((const uint16_t *)v_new)[((size_t)mc * HKV + hkv) * D + d] : 0;
  const float acc = kproj_tile32<HDT>(h, w, M, H, m0, n0, red);
  const float x = round_to(acc + bv, HDT);
  const float partner = __shfl_xor(x, 1);
  // fp32 cos / sin promote the rotation to fp32
  const float k = rope_one(x, partner, (d & 1) != 0, cv, sv, FFA_DT_F32);
  const int page = append_page(bt, bt_stride, num_pages, b, P);
  const int slot = P & 63;
  const bool wr = m < M && page >= 0;  // uniform over the 32 lanes of a token's group
  g32_quantize_lanes(k, wr, page, slot, hkv, HKV, g, kq_pages, s_pages, z_pages, r_pages, res_e4m3);
  if (v_new != nullptr && wr)  // V^T pages: this workgroup's 32 channels of each token
    ((uint16_t *)v_pages)[((size_t)page * HKV + hkv) * (D * 64) + vt_off(d, slot)] = vv;
}


// g32 quantize + append of given K rows (no projection): 128 threads per (token row, KV head),
// one channel each (coalesced loads; the quantization of a 32-channel group runs across the 32
// lanes of a half wave, g32_quantize_lanes).  k [B, Tn, HKV, 128] (dtype kdt).
__global__ __launch_bounds__(256) void q2_g32_append_kernel(const void *k, int kdt, int M, int Tn, int HKV,
                                                             const int32_t *pos, const int32_t *bt, int bt_stride,
                                                             int num_pages, uint8_t *kq_pages, uint16_t *s_pages,
                                                             uint16_t *z_pages, uint8_t *r_pages, int res_e4m3,
                                                             const void *v_new, int vmode, void *v_pages) {
  constexpr int D = 128;
  const size_t rowid = (size_t)blockIdx.x * 2 + (threadIdx.x >> 7);  // (token row, head)
  if (rowid >= (size_t)M * HKV) return;  // whole waves (a row is two waves)
  const int c = threadIdx.x & 127, g = c >> 5;
  const int hkv = (int)(rowid % HKV);
  const int m = (int)(rowid / HKV);
  const int b = m / Tn, nn = m % Tn;
  const int P = pos[b] + nn;
  const int page = append_page(bt, bt_stride, num_pages, b, P);
  const int slot = P & 63;
  const float x = load_any(k, rowid * D + c, kdt);
  g32_quantize_lanes(x, page >= 0, page, slot, hkv, HKV, g, kq_pages, s_pages, z_pages, r_pages, res_e4m3);
  if (v_new != nullptr && page >= 0)
    ((uint16_t *)v_pages)[((size_t)page * HKV + hkv) * (D * 64) + vt_off(c, slot)] = v_element(v_new, vmode, rowid * D + c);
}


// The same append for many tokens, a (page, KV head) block per workgroup (page_tile.h): a thread holds a whole
// 32-channel group, so extrema, scale, codes and residual are its own; codes by the scale's turning points
// (q2_turn, of the fp32 quotient) instead of 32 divisions.  grid (KV head, tile, sequence).
template <int KDT, bool E4M3>
__global__ __launch_bounds__(256) void q2_g32_page_kernel(const void *k, int Tn, int HKV, const int32_t *pos,
                                                          const int32_t *bt, int bt_stride, int num_pages,
                                                          uint8_t *kq_pages, uint16_t *s_pages, uint16_t *z_pages,
                                                          uint8_t *r_pages, const void *v_new, int vmode, void *v_pages) {
  __shared__ __attribute__((aligned(16))) uint8_t s_t[page_tile_lds<KDT>()];
  const int hkv = blockIdx.x, b = blockIdx.z;
  const PageTile pt = page_tile(pos, bt, bt_stride, num_pages, b, blockIdx.y, Tn);
  if (pt.page < 0) return;  // the whole workgroup
  const size_t row0 = (size_t)b * Tn * HKV + hkv, blk = (size_t)pt.page * HKV + hkv;
  float x[32];
  page_tile_k<KDT>(k, row0, HKV, pt, s_t, x);
  const int m = threadIdx.x & 15, g = (threadIdx.x >> 4) & 3, tau = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int t = 4 * m + tau;
  float mn = x[0], mx = x[0];
#pragma unroll
  for (int e = 1; e < 32; ++e) mn = fminf(mn, x[e]), mx = fmaxf(mx, x[e]);
  const float zr = (float)(_Float16)mn;
  const float sc = (float)(_Float16)__fdiv_rn(fmaxf(mx - zr, 1e-6f), 3.0f);
  const float t1 = q2_turn<FFA_DT_F32>(sc, 0), t2 = q2_turn<FFA_DT_F32>(sc, 1), t3 = q2_turn<FFA_DT_F32>(sc, 2);
  uint32_t cw[2] = {0u, 0u};
#pragma unroll
  for (int e = 0; e < 32; ++e) {
    const float y = x[e] - zr;
    const uint32_t cq = y >= t3 ? 3u : (y >= t2 ? 2u : (y >= t1 ? 1u : 0u));
    cw[e >> 4] |= cq << (2 * (e & 15));
    x[e] -= (float)cq * sc + zr;
  }
  if (t >= pt.lo && t < pt.hi) {
    uint4 *rp = (uint4 *)(r_pages + blk * (64 * 128)) + tau * 128 + lane;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint2 r0 = f32x8_to_fp8<E4M3>(x + 16 * h), r1 = f32x8_to_fp8<E4M3>(x + 16 * h + 8);
      rp[64 * h] = make_uint4(r0.x, r0.y, r1.x, r1.y);
    }
    *(uint2 *)(kq_pages + blk * (4 * 64 * 8) + codes_off(g, t)) = make_uint2(cw[0], cw[1]);
    const int ss = 16 * (t >> 4) + 4 * (t & 3) + ((t >> 2) & 3);  // tile-major scale slot
    const size_t so = blk * (4 * 64) + gscale_off(g, ss);
    s_pages[so] = (uint16_t)f32_to_f16_bits(sc);
    z_pages[so] = (uint16_t)f32_to_f16_bits(zr);
  }
  if (v_new != nullptr) page_tile_v(v_new, vmode, row0, HKV, pt, s_t, (uint16_t *)v_pages + blk * (128 * 64));
}

// eight floats to eight consecutive elements of dtype DT in registers: one 16-byte word, or two (f32)
template <int DT>
__device__ __forceinline__ Raw8<DT> pack8(const float *x) {
  Raw8<DT> r;
  if constexpr (DT == 2) {
    r.v[0] = make_uint4(__float_as_uint(x[0]), __float_as_uint(x[1]), __float_as_uint(x[2]), __float_as_uint(x[3]));
    r.v[1] = make_uint4(__float_as_uint(x[4]), __float_as_uint(x[5]), __float_as_uint(x[6]), __float_as_uint(x[7]));
  } else {
    uint32_t w[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = DT == 1 ? pk_bf16_bits(x[2 * e], x[2 * e + 1]) : pk_f16_bits(x[2 * e], x[2 * e + 1]);
    r.v[0] = make_uint4(w[0], w[1], w[2], w[3]);
  }
  return r;
}

// 16 bytes of consecutive elements of kEs bytes at an address that is a multiple of 16 (WHOLE) or of kEs
template <int kEs, bool WHOLE>
__device__ __forceinline__ void store16(void *p, uint4 w) {
  if constexpr (WHOLE) {
    *(uint4 *)p = w;
  } else {
    const uint32_t v[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (kEs == 4) {
        ((uint32_t *)p)[i] = v[i];
      } else {
        ((uint16_t *)p)[2 * i] = (uint16_t)(v[i] & 0xffffu);
        ((uint16_t *)p)[2 * i + 1] = (uint16_t)(v[i] >> 16);
      }
    }
  }
}

// Paged g32 cache -> contiguous K and V (the exact-attention path of the HF integration, which the
// reference feeds with dequantized keys: ffa-fp8fp8/e2e/fp8fp8_cache.py:60-69, returned by update at
// :84-89).  One workgroup per (sequence, page of the sequence, KV head): K = c * s + z + r in fp32
// (c * s is exact, so the fma rounds once, as the sum does), then one rounding to the output dtype.
// Tokens at or past the sequence's length are written as zeros; block-table entries outside the pool
// read page 0.
// Bound by the bytes (24 read, 27 KB or more written per page and head).  Everything is read in the
// pool's own order, 1 KB a wave and load: wave tau, lane (group g, m) holds all 32 channels of group g of
// token 4 m + tau (residual blocks (tau, 0) and (tau, 1)), and V^T pieces of 8 tokens of one column.
// Rows are put together in LDS and written 16 bytes a lane, whole rows at a time; V is turned by the
// transposing LDS read (4 tokens x 32 columns per 16 lanes).  Written 2 bytes a lane at 64-byte distances,
// as K and V were before, the cache of 4 sequences of 3K to 8K tokens, 214 MB, took 300 us; 56 now.  Outputs at
// addresses that are no multiple of 16 bytes are written element by element (WHOLE = false).
template <bool E4M3, int VDT, int ODT, bool WHOLE>
__global__ __launch_bounds__(256) void q2_paged_dequant_kernel(const uint8_t *kq_pages, const uint16_t *s_pages,
                                                               const uint16_t *z_pages, const uint8_t *r_pages,
                                                               const uint16_t *v_pages, const int32_t *bt, int bt_stride,
                                                               int num_pages, const int32_t *seq_lens, int T, int HKV,
                                                               void *k_out, void *v_out) {
  constexpr int D = 128;
  constexpr int kEs = ODT == 2 ? 4 : 2, kRow = D * kEs, kPcs = kRow / 16;  // output row: bytes, 16-byte pieces
  constexpr int kVPitch = 144;  // LDS bytes of a V^T column (64 tokens), 16 past 128 to spread the banks
  constexpr int kLds = 64 * kRow > D * kVPitch ? 64 * kRow : D * kVPitch;
  __shared__ __attribute__((aligned(16))) uint8_t s_t[kLds];
  const int j = blockIdx.x, hkv = blockIdx.y, b = blockIdx.z;
  const int Tb = seq_lens ? min(max(seq_lens[b], 0), T) : T;
  const int nv = min(max(Tb - 64 * j, 0), 64);  // tokens of the page that the sequence holds
  int page = bt[(size_t)b * bt_stride + j];
  page = (unsigned)page < (unsigned)num_pages ? page : 0;
  const size_t blk = (size_t)page * HKV + hkv;
  const int lane = threadIdx.x & 63, tau = threadIdx.x >> 6;
  const int m = lane & 15, g = lane >> 4, t = 4 * m + tau;
  const uint2 cw = *(const uint2 *)(kq_pages + blk * (4 * 64 * 8) + codes_off(g, t));
  const int ss = 16 * (t >> 4) + 4 * (t & 3) + ((t >> 2) & 3);  // tile-major scale slot, as appended
  const float sc = f16_bits_to_f32(s_pages[blk * (4 * 64) + gscale_off(g, ss)]);
  const float zr = f16_bits_to_f32(z_pages[blk * (4 * 64) + gscale_off(g, ss)]);
  const uint4 *rp = (const uint4 *)(r_pages + blk * (64 * D)) + tau * 128 + lane;
  const uint4 r0 = rp[0], r1 = rp[64];
  // V^T: 1024 16-byte pieces (8 tokens of one column); piece P holds column 16 (P >> 7) + (P & 15),
  // tokens 16 ((P >> 4) & 3) + 8 ((P >> 6) & 1) + (0..7)
  const uint4 *vp = (const uint4 *)(v_pages + blk * (D * 64));
  uint4 vw[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) vw[i] = vp[threadIdx.x + 256 * i];

  const uint32_t rw[8] = {r0.x, r0.y, r0.z, r0.w, r1.x, r1.y, r1.z, r1.w};
  const uint32_t cwords[2] = {cw.x, cw.y};
#pragma unroll
  for (int a = 0; a < 4; ++a) {  // channels 32 g + 8 a + (0..7)
    const f16x8 rv = fp8x8_to_f16x8<E4M3 ? kResE4M3 : kResE5M2>(rw[2 * a], rw[2 * a + 1]);  // exact
    float k[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t code = (cwords[a >> 1] >> (2 * ((8 * a + e) & 15))) & 3u;
      const float x = __builtin_fmaf((float)code, sc, zr) + (float)rv[e];
      k[e] = t < nv ? x : 0.f;
    }
    const Raw8<ODT> o = pack8<ODT>(k);
    // piece q of row t at q ^ (m & 7): the 16 rows that a write touches start at different banks
#pragma unroll
    for (int h = 0; h < kEs / 2; ++h) {
      const int q = (kPcs / 4) * g + (kEs / 2) * a + h;
      *(uint4 *)(s_t + t * kRow + ((q ^ (m & 7)) * 16)) = o.v[h];
    }
  }
  __syncthreads();
  const size_t orow = ((size_t)b * T + 64 * j) * HKV + hkv;  // row of the page's token 0
#pragma unroll
  for (int i = 0; i < 64 * kPcs / 256; ++i) {
    const int tk = (threadIdx.x + 256 * i) / kPcs, q = threadIdx.x & (kPcs - 1);
    const uint4 w = *(const uint4 *)(s_t + tk * kRow + ((q ^ ((tk >> 2) & 7)) * 16));
    store16<kEs, WHOLE>((uint8_t *)k_out + (orow + (size_t)tk * HKV) * kRow + 16 * q, w);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int P = threadIdx.x + 256 * i;
    const int c = 16 * (P >> 7) + (P & 15), t0 = 16 * ((P >> 4) & 3) + 8 * ((P >> 6) & 1);
    *(uint4 *)(s_t + c * kVPitch + 2 * t0) = vw[i];
  }
  __syncthreads();
  // lane x of a 16-lane group addresses 4 tokens of column 32 grp + 8 (x % 4) + x / 4 and receives, of token
  // x % 4 of those, the columns that lanes x / 4 + 4 e address: 32 grp + 8 (x / 4) + e (e = 0..3); a second read
  // 4 columns on completes its 8
  typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
  const int x = lane & 15, col = 32 * g + 8 * (x & 3) + (x >> 2);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int tk0 = 16 * tau + 4 * i, tk = tk0 + (x & 3);
    const auto *p0 = (const lds_s16x4 *)((__attribute__((address_space(3))) const uint8_t *)s_t + col * kVPitch + 2 * tk0);
    const auto *p1 = (const lds_s16x4 *)((__attribute__((address_space(3))) const uint8_t *)s_t + (col + 4) * kVPitch + 2 * tk0);
    const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)p0));
    const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)p1));
    Raw8<VDT> in;
    in.v[0] = make_uint4(lo[0], lo[1], hi[0], hi[1]);
    float v[8];
    raw8_to_f32<VDT>(in, v);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = tk < nv ? v[e] : 0.f;
    const Raw8<ODT> o = pack8<ODT>(v);
#pragma unroll
    for (int h = 0; h < kEs / 2; ++h)
      store16<kEs, WHOLE>((uint8_t *)v_out + (orow + (size_t)tk * HKV) * kRow + (32 * g + 8 * (x >> 2)) * kEs + 16 * h,
                          o.v[h]);
  }
}
}  // namespace ffa

// ============================================================================
// C ABI
// ============================================================================
// errors of this translation unit are reported through the decode unit's buffer
extern "C" __attribute__((visibility("hidden"))) int ffa_set_error_internal(int code, const char *msg);

extern "C" int ffa_q2_quantize_nsplit(int T) {
  int s = (T + ffa::kQTok - 1) / ffa::kQTok;
  return s < 1 ? 1 : (s > 64 ? 64 : s);
}

// the vector kernels of one K dtype
template <int KDT>
static void launch_quant8(const void *k, int B, int T, int C, int nsplit, uint8_t *k_q, void *scale, void *zero,
                          uint8_t *residual, bool e4m3, float *minmax, hipStream_t st) {
  hipLaunchKernelGGL(ffa::q2_minmax8_kernel<KDT>, dim3(nsplit, B, (C + ffa::kMmCols - 1) / ffa::kMmCols), dim3(256), 0,
                     st, k, T, C, nsplit, minmax);
  hipLaunchKernelGGL(ffa::q2_scale_kernel, dim3((C + 31) / 32, B), dim3(256), 0, st, (const float *)minmax, B, nsplit,
                     C, KDT, scale, zero);
  // a workgroup covers 2^lw vectors of a row and 256 >> lw rows at a time; its tokens: enough that a lane's
  // turning points are paid over 16 rows, but no fewer than 1024 workgroups while rows remain
  const int c8 = C / 8;
  int lw = 0;
  while (lw < 6 && (1 << lw) < c8) ++lw;
  const int rows = 256 >> lw, ny = (c8 + (1 << lw) - 1) >> lw;
  const long units = (long)B * ny * ((T + rows - 1) / rows);  // row steps of all workgroups
  long steps = units / 1024;
  steps = steps < 1 ? 1 : (steps > 16 ? 16 : steps);
  const int per = (int)steps * rows;
  const dim3 grid((unsigned)((T + per - 1) / per), (unsigned)ny, (unsigned)B);
  if (e4m3)
    hipLaunchKernelGGL((ffa::q2_quant8_kernel<KDT, true>), grid, dim3(256), 0, st, k, T, C, lw, per,
                       (const void *)scale, (const void *)zero, k_q, residual);
  else
    hipLaunchKernelGGL((ffa::q2_quant8_kernel<KDT, false>), grid, dim3(256), 0, st, k, T, C, lw, per,
                       (const void *)scale, (const void *)zero, k_q, residual);
}

static bool aligned(const void *p, size_t n) { return (reinterpret_cast<uintptr_t>(p) & (n - 1)) == 0; }

static int launch_quant_channel(const void *k, int kdt, int B, int T, int HKV, int D, uint8_t *k_q, void *scale,
                                void *zero, uint8_t *residual, int res_dtype, float *minmax, hipStream_t st) {
  const int C = HKV * D;
  const int nsplit = ffa_q2_quantize_nsplit(T);
  const int e4m3 = res_dtype == FFA_DT_FP8_E4M3 ? 1 : 0;
  // vectors of 8 columns: whole code bytes (D), whole vectors (C), aligned loads and stores, grid limits
  if (D % 4 == 0 && C % 8 == 0 && B <= 65535 && C <= 65535 * ffa::kMmCols && aligned(k, 16) && aligned(scale, 16) &&
      aligned(zero, 16) && aligned(residual, 8) && aligned(k_q, 2)) {
    if (kdt == FFA_DT_F16)
      launch_quant8<FFA_DT_F16>(k, B, T, C, nsplit, k_q, scale, zero, residual, e4m3 != 0, minmax, st);
    else if (kdt == FFA_DT_BF16)
      launch_quant8<FFA_DT_BF16>(k, B, T, C, nsplit, k_q, scale, zero, residual, e4m3 != 0, minmax, st);
    else
      launch_quant8<FFA_DT_F32>(k, B, T, C, nsplit, k_q, scale, zero, residual, e4m3 != 0, minmax, st);
  } else {
    hipLaunchKernelGGL(ffa::q2_minmax_kernel, dim3(nsplit, B, (C + 255) / 256), dim3(256), 0, st, k, kdt, T, C, nsplit,
                       minmax);
    hipLaunchKernelGGL(ffa::q2_scale_kernel, dim3((C + 31) / 32, B), dim3(256), 0, st, (const float *)minmax, B,
                       nsplit, C, kdt, scale, zero);
    const size_t total = (size_t)B * T * HKV * ((D + 3) / 4);
    hipLaunchKernelGGL(ffa::q2_quant_channel_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, k, kdt,
                       B, T, HKV, D, (const void *)scale, (const void *)zero, k_q, residual, e4m3);
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return ffa_set_error_internal(FFA_E_LAUNCH, hipGetErrorString(e));
  return FFA_OK;
}

extern "C" int ffa_q2_append_channel(const void *k_new, int k_dtype, int B, int Tn, int HKV, int D, const int32_t *pos,
                                     int T_cap, const void *scale, const void *zero, uint8_t *k_q, uint8_t *residual,
                                     int res_dtype, void *stream) {
  if (B <= 0 || Tn <= 0 || HKV <= 0 || D <= 0 || T_cap <= 0) return ffa_set_error_internal(FFA_E_INVALID, "bad dims");
  if (!(k_dtype >= FFA_DT_F16 && k_dtype <= FFA_DT_F32)) return ffa_set_error_internal(FFA_E_INVALID, "k dtype");
  if (!(res_dtype == FFA_DT_FP8_E4M3 || res_dtype == FFA_DT_FP8_E5M2))
    return ffa_set_error_internal(FFA_E_INVALID, "residual dtype");
  if (!k_new || !pos || !scale || !zero || !k_q || !residual) return ffa_set_error_internal(FFA_E_INVALID, "null pointer");
  const size_t total = (size_t)B * Tn * HKV * ((D + 3) / 4);
  hipLaunchKernelGGL(ffa::q2_append_channel_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, k_new, k_dtype, B, Tn, HKV, D, pos, T_cap, scale, zero, k_q, residual,
                     res_dtype == FFA_DT_FP8_E4M3 ? 1 : 0);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? FFA_OK : ffa_set_error_internal(FFA_E_LAUNCH, hipGetErrorString(e));
}

extern "C" int ffa_q2_quantize_channel(const void *k, int k_dtype, int B, int T, int HKV, int D, uint8_t *k_q,
                                       void *scale, void *zero, uint8_t *residual, int res_dtype, float *minmax,
                                       void *stream) {
  if (B <= 0 || T <= 0 || HKV <= 0 || D <= 0) return ffa_set_error_internal(FFA_E_INVALID, "bad dims");
  if (!(k_dtype >= FFA_DT_F16 && k_dtype <= FFA_DT_F32)) return ffa_set_error_internal(FFA_E_INVALID, "k dtype");
  if (!(res_dtype == FFA_DT_FP8_E4M3 || res_dtype == FFA_DT_FP8_E5M2))
    return ffa_set_error_internal(FFA_E_INVALID, "residual dtype must be fp8");
  return launch_quant_channel(k, k_dtype, B, T, HKV, D, k_q, scale, zero, residual, res_dtype, minmax,
                              (hipStream_t)stream);
}

template <int HDT, int TM, int TN>
static void launch_kproj_tile(const void *h, const void *w, const void *bias, const void *cos, const void *sin, int csdt,
                              int M, int T, int H, int N, int D, void *k_out, hipStream_t st) {
  const dim3 grid((unsigned)((size_t)((N + TN - 1) / TN) * ((M + TM - 1) / TM)));
  if (csdt == FFA_DT_F32)
    hipLaunchKernelGGL((ffa::kproj_rope_tile_kernel<HDT, true, TM, TN>), grid, dim3(256), 0, st, h, w, bias, cos, sin, M,
                       T, H, N, D, k_out);
  else
    hipLaunchKernelGGL((ffa::kproj_rope_tile_kernel<HDT, false, TM, TN>), grid, dim3(256), 0, st, h, w, bias, cos, sin, M,
                       T, H, N, D, k_out);
}

template <int HDT>
static void launch_kproj_rope(const void *h, const void *w, const void *bias, const void *cos, const void *sin, int csdt,
                              int M, int T, int H, int N, int D, void *k_out, int odt, hipStream_t st) {
  // Vector loads and stores need D and the pointers aligned, the K loop H a multiple of 64 (and a tile's rows
  // within a buffer resource's 31 bits).  Below H = 1024 the split's chains are shorter than two steps.
  if (H % ffa::kGemmK == 0 && H >= ffa::kGemmMinH && H < (1 << 22) && D % 4 == 0 && aligned(h, 16) && aligned(w, 16) &&
      aligned(k_out, 16) && aligned(cos, 16) && aligned(sin, 16)) {
    switch (ffa::kproj_route(M, N, ffa::device_cus() > 0 ? ffa::device_cus() : 256)) {
      case ffa::kKproj128x128: return launch_kproj_tile<HDT, 128, 128>(h, w, bias, cos, sin, csdt, M, T, H, N, D, k_out, st);
      case ffa::kKproj128x64: return launch_kproj_tile<HDT, 128, 64>(h, w, bias, cos, sin, csdt, M, T, H, N, D, k_out, st);
      case ffa::kKproj64x64: return launch_kproj_tile<HDT, 64, 64>(h, w, bias, cos, sin, csdt, M, T, H, N, D, k_out, st);
      case ffa::kKproj32x64: return launch_kproj_tile<HDT, 32, 64>(h, w, bias, cos, sin, csdt, M, T, H, N, D, k_out, st);
    }
  }
  hipLaunchKernelGGL(ffa::kproj_rope_kernel<HDT>, dim3((unsigned)((N / 32) * ((M + 15) / 16))), dim3(512), 0, st, h, w,
                     bias, cos, sin, csdt, M, T, H, N, D, k_out, odt);
}

extern "C" int ffa_kproj_rope(const void *h, const void *w_k, const void *bias, int h_dtype, const void *cos,
                              const void *sin, int cs_dtype, int B, int T, int H, int HKV, int D, void *k_out,
                              void *stream) {
  if (B <= 0 || T <= 0 || H <= 0 || HKV <= 0 || D <= 0) return ffa_set_error_internal(FFA_E_INVALID, "bad dims");
  if (!(h_dtype == FFA_DT_F16 || h_dtype == FFA_DT_BF16))
    return ffa_set_error_internal(FFA_E_UNSUPPORTED, "h must be fp16 or bf16");
  if (!(cs_dtype == FFA_DT_F32 || cs_dtype == h_dtype))
    return ffa_set_error_internal(FFA_E_UNSUPPORTED, "cos/sin must be fp32 or the dtype of h");
  if (D % 2 || (HKV * D) % 32 || H % 32)
    return ffa_set_error_internal(FFA_E_UNSUPPORTED, "needs even D, HKV*D % 32 == 0, H % 32 == 0");
  const int M = B * T, N = HKV * D;
  const int odt = cs_dtype == FFA_DT_F32 ? FFA_DT_F32 : h_dtype;
  hipStream_t st = (hipStream_t)stream;
  if (h_dtype == FFA_DT_BF16)
    launch_kproj_rope<FFA_DT_BF16>(h, w_k, bias, cos, sin, cs_dtype, M, T, H, N, D, k_out, odt, st);
  else
    launch_kproj_rope<FFA_DT_F16>(h, w_k, bias, cos, sin, cs_dtype, M, T, H, N, D, k_out, odt, st);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return ffa_set_error_internal(FFA_E_LAUNCH, hipGetErrorString(e));
  return FFA_OK;
}

extern "C" int ffa_kproj_rope_q2_channel(const void *h, const void *w_k, const void *bias, int h_dtype, const void *cos,
                                         const void *sin, int cs_dtype, int B, int T, int H, int HKV, int D,
                                         void *k_scratch, uint8_t *k_q, void *scale, void *zero, uint8_t *residual,
                                         int res_dtype, float *minmax, void *stream) {
  if (!(res_dtype == FFA_DT_FP8_E4M3 || res_dtype == FFA_DT_FP8_E5M2))
    return ffa_set_error_internal(FFA_E_INVALID, "residual dtype must be fp8");
  const int rc = ffa_kproj_rope(h, w_k, bias, h_dtype, cos, sin, cs_dtype, B, T, H, HKV, D, k_scratch, stream);
  if (rc != FFA_OK) return rc;
  const int odt = cs_dtype == FFA_DT_F32 ? FFA_DT_F32 : h_dtype;
  return launch_quant_channel(k_scratch, odt, B, T, HKV, D, k_q, scale, zero, residual, res_dtype, minmax,
                              (hipStream_t)stream);
}

extern "C" int ffa_kproj_rope_q2_append(const void *h, const void *w_k, const void *bias, int h_dtype, const float *cos,
                                        const float *sin, int B, int Tn, int H, int HKV, const int32_t *pos,
                                        const int32_t *block_table, int bt_stride, int num_pages,
                                        uint8_t *k_q_pages, void *scale_pages, void *zero_pages, uint8_t *res_pages,
                                        int res_dtype, const void *v_new, void *v_pages, int v_dtype, void *stream) {
  if (B <= 0 || Tn <= 0 || H <= 0 || HKV <= 0) return ffa_set_error_internal(FFA_E_INVALID, "bad dims");
  if (bt_stride <= 0 || num_pages <= 0) return ffa_set_error_internal(FFA_E_INVALID, "empty block table or pool");
  if (!(h_dtype == FFA_DT_F16 || h_dtype == FFA_DT_BF16))
    return ffa_set_error_internal(FFA_E_UNSUPPORTED, "h must be fp16 or bf16");
  if (H % 32) return ffa_set_error_internal(FFA_E_UNSUPPORTED, "H must be a multiple of 32");
  if (!(res_dtype == FFA_DT_FP8_E4M3 || res_dtype == FFA_DT_FP8_E5M2))
    return ffa_set_error_internal(FFA_E_INVALID, "residual dtype must be fp8");
  if (v_new != nullptr && !(v_dtype == FFA_DT_F16 || v_dtype == FFA_DT_BF16))
    return ffa_set_error_internal(FFA_E_UNSUPPORTED, "V pages must be fp16 or bf16");
  const int M = B * Tn;
  hipStream_t st = (hipStream_t)stream;
  const dim3 grid((unsigned)(HKV * 4 * ((M + 15) / 16)));
  if (h_dtype == FFA_DT_BF16)
    hipLaunchKernelGGL(ffa::kproj_append_kernel<FFA_DT_BF16>, grid, dim3(512), 0, st, h, w_k, bias, cos, sin, M, Tn, H,
                       HKV, pos, block_table, bt_stride, num_pages, k_q_pages, (uint16_t *)scale_pages,
                       (uint16_t *)zero_pages,
                       res_pages, res_dtype == FFA_DT_FP8_E4M3 ? 1 : 0, v_new, v_pages);
  else
    hipLaunchKernelGGL(ffa::kproj_append_kernel<FFA_DT_F16>, grid, dim3(512), 0, st, h, w_k, bias, cos, sin, M, Tn, H,
                       HKV, pos, block_table, bt_stride, num_pages, k_q_pages, (uint16_t *)scale_pages,
                       (uint16_t *)zero_pages,
                       res_pages, res_dtype == FFA_DT_FP8_E4M3 ? 1 : 0, v_new, v_pages);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return ffa_set_error_internal(FFA_E_LAUNCH, hipGetErrorString(e));
  return FFA_OK;
}

static int q2_g32_append(const void *k, int k_dtype, int B, int Tn, int HKV, const int32_t *pos,
                         const int32_t *block_table, int bt_stride, int num_pages, uint8_t *k_q_pages,
                         void *scale_pages, void *zero_pages, uint8_t *res_pages, int res_dtype, const void *v_new,
                         int vmode, void *v_pages, void *stream) {
  if (B <= 0 || Tn <= 0 || HKV <= 0) return ffa_set_error_internal(FFA_E_INVALID, "bad dims");
  if (bt_stride <= 0 || num_pages <= 0) return ffa_set_error_internal(FFA_E_INVALID, "empty block table or pool");
  if (!(k_dtype >= FFA_DT_F16 && k_dtype <= FFA_DT_F32)) return ffa_set_error_internal(FFA_E_INVALID, "k dtype");
  if (!(res_dtype == FFA_DT_FP8_E4M3 || res_dtype == FFA_DT_FP8_E5M2))
    return ffa_set_error_internal(FFA_E_INVALID, "residual dtype must be fp8");
  const bool e4m3 = res_dtype == FFA_DT_FP8_E4M3;
  // Whole pages where the sizes favour them (q2_whole_pages); the pieces need aligned rows and pools, the tiles are a
  // grid dimension
  if (ffa::q2_whole_pages(B, Tn, HKV) && ffa::page_tiles(Tn) <= 65535 && B <= 65535 && aligned(k, 16) &&
      aligned(v_new, 16) && aligned(res_pages, 16) && aligned(v_pages, 16) && aligned(k_q_pages, 8)) {
    const dim3 grid((unsigned)HKV, (unsigned)ffa::page_tiles(Tn), (unsigned)B);
#define FFA_CASE(KK, EE)                                                                                            \
  if (k_dtype == KK && e4m3 == EE)                                                                                  \
    hipLaunchKernelGGL((ffa::q2_g32_page_kernel<KK, EE>), grid, dim3(256), 0, (hipStream_t)stream, k, Tn, HKV, pos, \
                       block_table, bt_stride, num_pages, k_q_pages, (uint16_t *)scale_pages, (uint16_t *)zero_pages, \
                       res_pages, v_new, vmode, v_pages);
    FFA_CASE(FFA_DT_F16, true)
    FFA_CASE(FFA_DT_F16, false)
    FFA_CASE(FFA_DT_BF16, true)
    FFA_CASE(FFA_DT_BF16, false)
    FFA_CASE(FFA_DT_F32, true)
    FFA_CASE(FFA_DT_F32, false)
#undef FFA_CASE
  } else {
    const size_t rows = (size_t)B * Tn * HKV;
    hipLaunchKernelGGL(ffa::q2_g32_append_kernel, dim3((unsigned)((rows + 1) / 2)), dim3(256), 0,
                       (hipStream_t)stream, k, k_dtype, B * Tn, Tn, HKV, pos, block_table, bt_stride, num_pages,
                       k_q_pages, (uint16_t *)scale_pages, (uint16_t *)zero_pages, res_pages, e4m3 ? 1 : 0, v_new,
                       vmode, v_pages);
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return ffa_set_error_internal(FFA_E_LAUNCH, hipGetErrorString(e));
  return FFA_OK;
}

extern "C" int ffa_q2_quantize_g32_append(const void *k, int k_dtype, int B, int Tn, int HKV, const int32_t *pos,
                                          const int32_t *block_table, int bt_stride, int num_pages,
                                          uint8_t *k_q_pages, void *scale_pages, void *zero_pages, uint8_t *res_pages,
                                          int res_dtype, const void *v_new, void *v_pages, void *stream) {
  return q2_g32_append(k, k_dtype, B, Tn, HKV, pos, block_table, bt_stride, num_pages, k_q_pages, scale_pages,
                       zero_pages, res_pages, res_dtype, v_new, ffa::kVSame, v_pages, stream);
}

extern "C" int ffa_q2_quantize_g32_append_cast(const void *k, int k_dtype, int B, int Tn, int HKV, const int32_t *pos,
                                               const int32_t *block_table, int bt_stride, int num_pages,
                                               uint8_t *k_q_pages, void *scale_pages, void *zero_pages,
                                               uint8_t *res_pages, int res_dtype, const void *v_new, int v_new_dtype,
                                               void *v_pages, int v_dtype, void *stream) {
  const int vmode = v_new ? ffa::v_mode(v_new_dtype, v_dtype) : ffa::kVSame;
  if (vmode < 0) return ffa_set_error_internal(FFA_E_INVALID, "v dtypes (rows fp16, bf16 or fp32, pool fp16 or bf16)");
  return q2_g32_append(k, k_dtype, B, Tn, HKV, pos, block_table, bt_stride, num_pages, k_q_pages, scale_pages,
                       zero_pages, res_pages, res_dtype, v_new, vmode, v_pages, stream);
}

extern "C" int ffa_q2_paged_dequant(const uint8_t *k_q_pages, const void *scale_pages, const void *zero_pages,
                                    const uint8_t *res_pages, int res_dtype, const void *v_pages, int v_dtype,
                                    const int32_t *block_table, int bt_stride, int num_pages, const int32_t *seq_lens,
                                    int B, int T, int HKV, void *k_out, void *v_out, int out_dtype, void *stream) {
  if (B <= 0 || T <= 0 || HKV <= 0) return ffa_set_error_internal(FFA_E_INVALID, "bad dims");
  if (B > 65535 || HKV > 65535) return ffa_set_error_internal(FFA_E_UNSUPPORTED, "B and HKV are grid dimensions");
  if (bt_stride <= 0 || num_pages <= 0) return ffa_set_error_internal(FFA_E_INVALID, "empty block table or pool");
  if ((long)bt_stride * ffa::kPage < T) return ffa_set_error_internal(FFA_E_INVALID, "block table has fewer than ceil(T/64) columns");
  if (!(res_dtype == FFA_DT_FP8_E4M3 || res_dtype == FFA_DT_FP8_E5M2))
    return ffa_set_error_internal(FFA_E_INVALID, "residual dtype must be fp8");
  if (!(v_dtype == FFA_DT_F16 || v_dtype == FFA_DT_BF16)) return ffa_set_error_internal(FFA_E_INVALID, "v dtype");
  if (!(out_dtype >= FFA_DT_F16 && out_dtype <= FFA_DT_F32)) return ffa_set_error_internal(FFA_E_INVALID, "out dtype");
  if (!k_q_pages || !scale_pages || !zero_pages || !res_pages || !v_pages || !block_table || !k_out || !v_out)
    return ffa_set_error_internal(FFA_E_INVALID, "null pointer");
  if (T % ffa::kPage) return ffa_set_error_internal(FFA_E_INVALID, "T must be a multiple of the 64-token page");
  const dim3 grid((unsigned)(T / ffa::kPage), (unsigned)HKV, (unsigned)B);
  const bool whole = aligned(k_out, 16) && aligned(v_out, 16);
#define FFA_CASE(EE, VV, OO, WW)                                                                                     \
  if ((res_dtype == FFA_DT_FP8_E4M3) == EE && v_dtype == VV && out_dtype == OO && whole == WW)                       \
    hipLaunchKernelGGL((ffa::q2_paged_dequant_kernel<EE, VV, OO, WW>), grid, dim3(256), 0, (hipStream_t)stream,      \
                       k_q_pages, (const uint16_t *)scale_pages, (const uint16_t *)zero_pages, res_pages,            \
                       (const uint16_t *)v_pages, block_table, bt_stride, num_pages, seq_lens, T, HKV, k_out, v_out);
#define FFA_CASES(EE, VV)                                                      \
  FFA_CASE(EE, VV, FFA_DT_F16, true) FFA_CASE(EE, VV, FFA_DT_F16, false)       \
  FFA_CASE(EE, VV, FFA_DT_BF16, true) FFA_CASE(EE, VV, FFA_DT_BF16, false)     \
  FFA_CASE(EE, VV, FFA_DT_F32, true) FFA_CASE(EE, VV, FFA_DT_F32, false)
  FFA_CASES(true, FFA_DT_F16)
  FFA_CASES(true, FFA_DT_BF16)
  FFA_CASES(false, FFA_DT_F16)
  FFA_CASES(false, FFA_DT_BF16)
#undef FFA_CASES
#undef FFA_CASE
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? FFA_OK : ffa_set_error_internal(FFA_E_LAUNCH, hipGetErrorString(e));
}
