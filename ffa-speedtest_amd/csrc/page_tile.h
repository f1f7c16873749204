// Whole pages of a paged cache written at once: what the many-token appends of the 2-bit, nvfp4 and nf4
// caches share.  A 256-thread workgroup takes one (page, KV head) block: 64 token slots x 128 channels.
//
// Bound by the bytes: K and V are read once, codes, scales, residual and V^T written once.  K rows come in
// 16 bytes a lane, whole rows, go through LDS, and wave tau, lane (g, m) = (lane >> 4, lane & 15) gets the 32
// channels of group g of token slot 4 m + tau: the order of the pool's residual and 4-bit code pieces, so that
// every store instruction of a wave writes one contiguous KB.  A thread holds its quantization group alone or
// with one neighbour, so minima, maxima and scales need no chain of shuffles.  V goes through LDS too and leaves
// by the transposing read, already in the order of the V^T pieces.  (One thread per channel, 1-byte stores and
// five shuffles per extremum before: 16K tokens x 8 heads took 112 us, 129 for nf4.)
#pragma once

#include "decode_common.h"
#include "routes.h"

namespace ffa {

// V rows given with an append: how they are brought to the pool's 16-bit type (the conversions of a torch cast:
// through fp32, round to nearest even, a NaN to bf16's 0x7fc0).  Cast by the caller instead, 16K x 1024 bf16 values for an fp16 pool were
// 67 MB more to move, a launch and an allocation.
enum { kVSame = 0, kVBf16ToF16 = 1, kVF16ToBf16 = 2, kVF32ToF16 = 3, kVF32ToBf16 = 4 };
// element types (0 = f16, 1 = bf16, 2 = f32) of the rows and of the pool; -1: not one of the above
inline int v_mode(int from, int to) {
  if (to != 0 && to != 1) return -1;
  if (from == to) return kVSame;
  if (from == 2) return to == 0 ? kVF32ToF16 : kVF32ToBf16;
  return from == 1 ? kVBf16ToF16 : (from == 0 ? kVF16ToBf16 : -1);
}
// a and b as the bf16 halves of a word, as a cast leaves them
__device__ __forceinline__ uint32_t cast_pk_bf16(float a, float b) {
  uint32_t w = pk_bf16_bits(a, b);
  if (__builtin_isnan(a)) w = (w & 0xffff0000u) | 0x7fc0u;
  if (__builtin_isnan(b)) w = (w & 0xffffu) | 0x7fc00000u;
  return w;
}
__device__ __forceinline__ uint16_t v_element(const void *v, int vmode, size_t i) {
  if (vmode == kVSame) return ((const uint16_t *)v)[i];
  const float x = load_any(v, i, vmode == kVF16ToBf16 ? 0 : (vmode == kVBf16ToF16 ? 1 : 2));
  return (uint16_t)(vmode == kVF16ToBf16 || vmode == kVF32ToBf16 ? cast_pk_bf16(x, x) : f32_to_f16_bits(x));
}

struct PageTile {
  int page;    // pool page, or -1: nothing to write
  int P0;      // position of the page's slot 0 in the sequence
  int n0;      // row of slot 0 among the sequence's new tokens (negative: the page starts before them)
  int lo, hi;  // slots [lo, hi) are new tokens
};
// tile i of sequence b: page (pos >> 6) + i of the sequence, for new tokens at positions pos .. pos + Tn - 1
__device__ __forceinline__ PageTile page_tile(const int32_t *pos, const int32_t *bt, int bt_stride, int num_pages, int b,
                                              int i, int Tn) {
  PageTile t;
  const int p = pos[b];
  t.P0 = ((p >> 6) + i) * 64;
  t.n0 = t.P0 - p;
  t.lo = max(-t.n0, 0);
  t.hi = min(64, Tn - t.n0);
  t.page = t.lo < t.hi ? append_page(bt, bt_stride, num_pages, b, t.P0) : -1;
  return t;
}

constexpr int kVTilePitch = kVRow;  // LDS bytes of a V row
template <int KDT>
constexpr int page_tile_lds() {
  return 64 * 128 * (KDT == 2 ? 4 : 2) > 64 * kVTilePitch ? 64 * 128 * (KDT == 2 ? 4 : 2) : 64 * kVTilePitch;
}

// K of the tile into x: the 32 channels of group g of slot 4 m + tau (zeros in slots without a new token).
// Two barriers; lds may be reused after the call.  rows: the sequence's new tokens [Tn, HKV, 128] at head hkv.
template <int KDT>
__device__ __forceinline__ void page_tile_k(const void *k, size_t row0, int HKV, const PageTile &pt, uint8_t *lds,
                                            float (&x)[32]) {
  constexpr int kEs = KDT == 2 ? 4 : 2, kRow = 128 * kEs, kPcs = kRow / 16, kN = 64 * kPcs / 256;
  const int th = threadIdx.x;
  uint4 w[kN];
#pragma unroll
  for (int i = 0; i < kN; ++i) {
    const int t = (th + 256 * i) / kPcs, q = th & (kPcs - 1);
    w[i] = make_uint4(0u, 0u, 0u, 0u);
    if (t >= pt.lo && t < pt.hi)
      w[i] = *(const uint4 *)((const uint8_t *)k + (row0 + (size_t)((long)(pt.n0 + t) * HKV)) * kRow + 16 * q);
  }
#pragma unroll
  for (int i = 0; i < kN; ++i) {  // piece q of row t at q ^ (t / 4 % 8): reads and writes spread over the banks
    const int t = (th + 256 * i) / kPcs, q = th & (kPcs - 1);
    *(uint4 *)(lds + t * kRow + ((q ^ ((t >> 2) & 7)) * 16)) = w[i];
  }
  __syncthreads();
  const int m = th & 15, g = (th >> 4) & 3, t = 4 * m + (th >> 6);
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    Raw8<KDT> r;
#pragma unroll
    for (int h = 0; h < kEs / 2; ++h)
      r.v[h] = *(const uint4 *)(lds + t * kRow + ((((kPcs / 4) * g + (kEs / 2) * a + h) ^ (m & 7)) * 16));
    raw8_to_f32<KDT>(r, x + 8 * a);
  }
  __syncthreads();
}

// V of the tile from rows [Tn, HKV, 128] into the page's V^T block.  One barrier; lds free on entry.
__device__ __forceinline__ void page_tile_v(const void *v, int vmode, size_t row0, int HKV, const PageTile &pt,
                                            uint8_t *lds, uint16_t *dst) {
  const int th = threadIdx.x, lane = th & 63, wv = th >> 6;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int t = (th + 256 * i) >> 4, q = th & 15;
    uint4 w = make_uint4(0u, 0u, 0u, 0u);
    if (t >= pt.lo && t < pt.hi) {
      const size_t at = (row0 + (size_t)((long)(pt.n0 + t) * HKV)) * 128 + 8 * q;
      if (vmode == kVSame) {
        w = *(const uint4 *)((const uint16_t *)v + at);
      } else {
        float x[8];
        if (vmode == kVBf16ToF16) raw8_to_f32<1>(load8<1>(v, at), x);
        else if (vmode == kVF16ToBf16) raw8_to_f32<0>(load8<0>(v, at), x);
        else raw8_to_f32<2>(load8<2>(v, at), x);
        const bool bf = vmode == kVF16ToBf16 || vmode == kVF32ToBf16;
        uint32_t o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = bf ? cast_pk_bf16(x[2 * e], x[2 * e + 1]) : pk_f16_bits(x[2 * e], x[2 * e + 1]);
        w = make_uint4(o[0], o[1], o[2], o[3]);
      }
    }
    *(uint4 *)(lds + t * kVTilePitch + 16 * q) = w;
  }
  __syncthreads();
  const int n = lane & 15, kc = lane >> 4;
#pragma unroll
  for (int i = 0; i < 4; ++i) {  // piece (nu, kap), lane (kc, n): tokens 16 kc + 8 kap + (0..7) of column 16 nu + n
    const int nu = 2 * wv + (i >> 1), kap = i & 1;
    const u32x4 w = vt_operand_lds(lds, kVTilePitch, nu, kap, kc, n);
    const int t0 = 16 * kc + 8 * kap, at = ((nu * 2 + kap) * 64 + lane) * 8;
    if (t0 >= pt.lo && t0 + 8 <= pt.hi) {
      *(u32x4 *)(dst + at) = w;
    } else {  // a piece that holds older tokens or slots not yet written: the new ones alone
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (t0 + e >= pt.lo && t0 + e < pt.hi) dst[at + e] = (uint16_t)(w[e >> 1] >> (16 * (e & 1)));
    }
  }
}

}  // namespace ffa
