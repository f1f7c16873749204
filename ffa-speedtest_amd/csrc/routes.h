// Which of two kernels a call takes, where both give the same bytes and the sizes decide: plain host functions.
#pragma once

namespace ffa {

// pages that Tn tokens at any position can touch: workgroups of an append by whole pages, per sequence and KV head
inline int page_tiles(int Tn) { return (int)(((long)Tn + 126) >> 6); }

// 2-bit appends by whole (page, KV head) blocks rather than 128 threads per (token, head): for whole pages' worth of
// tokens, from some 4600 rows (tokens x heads) on; below that a launch of either is all latency, 6 us against 3.5.  us,
// per row against whole pages, fp16 V:
//   rows 1024 (one head of 1024 tokens, 40 x 33)   4.5 / 6.5      2048   5.0 / 6.2      4096 (16 heads of 4 x 64, 4 of
//   1024 tokens, 2 of 2048)   6.0 / 7.0, 6.5 / 6.8, 7.4 / 6.3     8192   9.1-11.6 / 6.6-8.3      16K tokens x 8 heads 120 / 29
//   16 tokens a sequence, 8 and 16 heads   equal from 8192 rows on
inline bool q2_whole_pages(int B, int Tn, int HKV) { return Tn >= 32 && (long)B * Tn * HKV >= 4608; }

// nvfp4 / nf4 appends by whole (page, KV head) blocks rather than a thread per 16 channels of a token.  A workgroup of
// the first costs some 6 ns (nvfp4; nf4 9) however few of its 64 slots it fills, past the 7 us that the smallest launch
// takes; the second needs 14 us up to 8K rows (tokens x heads).  us, per token against whole pages, bf16 keys:
//   one token, B x HKV = 512    nvfp4 14 / 8, nf4 14 / 10      1024    14 / 11, 14 / 14      2048    15 / 15, 15 / 23
//                     4096            16 / 24,     16 / 40     8 tokens, 2048 (4096 workgroups)    26 / 30,     26 / 40
//   16 tokens of 256 sequences, 8 heads   41 / 30, 41 / 41     of 4 heads   21 / 20, 20 / 25
//   32 tokens of 1024 sequences, 1 head   27 / 19, 27 / 25     of 256, 8 heads   75 / 31, 71 / 42
// (2 tokens of 2048 sequences with 4 heads took 106 us by pages, fp32 keys, and 23 per token.)
inline bool k4_whole_pages(bool nf4, int B, int Tn, int HKV) {
  const long workgroups = (long)B * HKV * page_tiles(Tn);
  return workgroups <= (nf4 ? 512 : 1024) || Tn >= 32 || (!nf4 && Tn >= 16 && HKV >= 8);
}

}  // namespace ffa
