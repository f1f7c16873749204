// Which kernel or build a call takes where several compute the same (the same bytes, or sums in another order) and the
// sizes decide: plain host functions.
#pragma once

namespace ffa {

// pages that Tn tokens at any position can touch: workgroups of an append by whole pages, per sequence and KV head
inline int page_tiles(int Tn) { return (int)(((long)Tn + 126) >> 6); }

// nvfp4 quantizer of the reference layout by vectors of 8 channels, a page of a KV head per workgroup: pages of more than
// 256 values.  Smaller ones leave most of its threads without a vector (time over the element-wise kernel's, 16-bit keys
// of 30K tokens: 64 values 1.3-1.5, 128 1.2-1.4, 256 0.9-1.06, 384 0.8-0.9, 8192 0.3).
inline bool nvfp4_by_vectors(int D, int page) { return D % 8 == 0 && (long)D * page > 256; }

// 2-bit appends by whole (page, KV head) blocks rather than 128 threads per (token, head): for whole pages' worth of
// tokens, from some 4600 rows (tokens x heads) on; below that a launch of either is all latency, 6 us against 3.5.  us,
// per row against whole pages, fp16 V:
//   rows 1024 (one head of 1024 tokens, 40 x 33)   4.5 / 6.5      2048   5.0 / 6.2      8192   9.1-11.6 / 6.6-8.3
//   rows 4096 (16 heads of 4 x 64, 4 of 1024 tokens, 2 of 2048)   6.0 / 7.0, 6.5 / 6.8, 7.4 / 6.3
//   16K tokens x 8 heads   120 / 29      16 tokens a sequence, 8 and 16 heads   equal from 8192 rows on
inline bool q2_whole_pages(int B, int Tn, int HKV) { return Tn >= 32 && (long)B * Tn * HKV >= 4608; }

// nvfp4 / nf4 appends by whole (page, KV head) blocks rather than a thread per 16 channels of a token.  A workgroup of
// the first costs some 6 ns (nvfp4; nf4 9) however few of its 64 slots it fills, past the 7 us that the smallest launch
// takes; the second needs 14 us up to 8K rows (tokens x heads).  us, per token against whole pages, bf16 keys:
//   one token, B x HKV = 512    nvfp4 14 / 8, nf4 14 / 10      1024    14 / 11, 14 / 14      2048    15 / 15, 15 / 23
//   4096    16 / 24, 16 / 40      8 tokens of 256 sequences, 8 heads (4096 workgroups)    26 / 30, 26 / 40
//   16 tokens of 256 sequences, 8 heads   41 / 30, 41 / 41     of 4 heads   21 / 20, 20 / 25
//   32 tokens of 1024 sequences, 1 head   27 / 19, 27 / 25     of 256, 8 heads   75 / 31, 71 / 42
// (2 tokens of 2048 sequences with 4 heads took 106 us by pages, fp32 keys, and 23 per token.)
inline bool k4_whole_pages(bool nf4, int B, int Tn, int HKV) {
  const long workgroups = (long)B * HKV * page_tiles(Tn);
  return workgroups <= (nf4 ? 512 : 1024) || Tn >= 32 || (!nf4 && Tn >= 16 && HKV >= 8);
}

// Paged 2-bit decode with nq quads of query rows per KV head: whether the quads' loads keep the default cache policy and
// pass 2 decides before it loads (the SHARE builds).  With a multiple of 8 KV heads the quads of one run on one XCD; one
// head's few workgroups gain as well.  Elsewhere the quads meet in the last-level cache only, which pays where rounds of
// workgroups queue up: time over that of the other builds, groups of 8, at a usual and a full share of kept blocks
//   4 heads  one a CU (16K tokens) 0.98, 1.05    2.25 (4 x 3K-9K) 1.02, 1.02    3 (50K) 0.92, 0.97    6 (100K) 0.81, 0.95
//   2 heads  one a CU (32K) 0.96, 1.04 (groups of 5 1.00, 1.10)    1.5 (50K) 0.95, 1.02    3 (100K) 0.93, 1.00
//   3 heads  0.75 a CU (16K) 0.97, 1.06    2.3 (50K) 0.94, 0.98    2.6 (4 x 14K) 0.91, 0.98
//   1 head   up to 1.5 a CU 0.96-1.00      8 heads  2 a CU (32K) 0.92, 0.77 of the build without this unit order
inline bool quads_share(int nq, int HKV, long workgroups, int cus) {
  return nq > 1 && (HKV % 8 == 0 || HKV == 1 || 2 * workgroups > 5 * (long)cus);
}

// Contiguous per-channel 2-bit decode: whether the build for three workgroups per CU is taken (V staged a quarter of its
// columns at a time) or that for two.
// Several quads per KV head, from more than two workgroups a CU: 8 x 16K tokens, 64 query heads of 8, 175 -> 139 us,
// 4 x 64K 246 -> 175, and faster at every share of kept blocks (0.80-0.99); with at most two a CU the sharing that comes
// with it gave 1-2 %, and lost as much with mean values.
// One quad, from five a CU: below that a third round of workgroups that is nearly empty costs more than the third
// resident one hides (4 layers of 2 x 30K, 944 workgroups: 127 -> 131 us; of 3 x 30K, 1416: 167 either way).  It pays
// while pruned chunks leave the CUs waiting: 8 x 16K to 32 x 16K tokens, 32 query heads of 8, 0.94-0.95 of the time at
// 40 % of the blocks kept, 0.99-1.02 at 70 %, but 1.06-1.10 with all of them, where the narrower staging shows (with
// mean values 0.94-0.95, 0.95-0.98, 0.97-1.04).  The threshold's distance from the probes' maximum is what a launch
// knows of that: with the usual 5 or less the three-per-CU build (at 8 the ratios are 0.89 to 1.03).
inline bool three_per_cu(int nq, long workgroups, int cus, float delta) {
  return nq > 1 ? workgroups > 2 * (long)cus : workgroups > 5 * (long)cus && delta <= 5.f;
}

// K projection + RoPE of M tokens onto N channels: the split kernel (16 tokens x 32 channels a workgroup) or a tile of
// the LDS-staged one.  us at H = 4096, bf16 (from H = 1024 to 8192 the order is the same but for
// differences of a few per cent):
//   N = 1024, tiles 128x128 / 128x64 / 64x64 / 32x64, split
//     M = 256  - / - / 21 / 18, 18    512  45 / 31 / 22 / 18, 36    1024  45 / 32 / 22 / 26, 67
//     2048  45 / 32 / 36 / -, 128
//     4096  53 / 57 / 72 / -, 249    4100  87 / 70 / 70 / -, 230    5200  89 / 73 / 85 / -, 287
//     8200  130 / 112 / - / -, 447
//   N = 32 (half of a tile's channels unused)   M = 4096  32x64 17.3, split 11.7    4224  17.2, 18.8    5200  17.7, 19.5
//   N = 2048   M = 100  32x64 18.0, split 16.5    128  18.1, 17.3      N = 8192   M = 32  17.8, 26.6    100  42.6, 80.6
// So: the split kernel while its workgroups are one round (a few more than one a CU run beside the others), for short
// prompts up to N = 2048, and where the smallest tiles fill less than half the chip; then the largest tile that gives
// every CU a workgroup.  A 128x128 workgroup has its CU to itself, so a last round of them that is at most half full
// costs as much as a full one: 128x64 tiles take it, two a CU, where their number is whole in XCD order (elsewhere they
// were the slower ones: M = 12000, N = 384 95 -> 109).
enum { kKprojSplit = 0, kKproj32x64, kKproj64x64, kKproj128x64, kKproj128x128 };
inline int kproj_route(int M, int N, int cus) {
  auto tiles = [&](int tm, int tn) { return (long)((M + tm - 1) / tm) * ((N + tn - 1) / tn); };
  const long split = (long)((M + 15) / 16) * (N / 32);
  if (tiles(32, 64) < cus / 2 || split < cus + cus / 32 || (M <= 128 && N <= 2048)) return kKprojSplit;
  const long large = tiles(128, 128), over = large % cus;
  if (large >= cus) return over > 0 && 2 * over <= cus && tiles(128, 64) % 8 == 0 ? kKproj128x64 : kKproj128x128;
  return tiles(128, 64) >= cus ? kKproj128x64 : (tiles(64, 64) >= cus ? kKproj64x64 : kKproj32x64);
}

}  // namespace ffa
