// Tuning policy of the kernels: cache hints, rows per thread, tile order.  Every value here
// was chosen by measurement on MI355X with cold inputs (buffers rotated beyond the memory-side
// cache); results are identical whatever the values.  One table for the whole library.
//
// A sweep build may replace the table: compile with -DFQ_POLICY_HEADER='"my_policy.hpp"', a
// header that defines fq::Policy with the same members.
#pragma once

#ifdef FQ_POLICY_HEADER
#include FQ_POLICY_HEADER
#else
namespace fq {

struct Policy {
  // ---- which code stores carry the non-temporal hint (bit 0: transposed codes, bit 1: row-wise
  // codes).  With it the outputs do not displace inputs from L2 and the memory-side cache:
  // gather+pad+quant 75 -> 55 us, RMSNorm+quant after the statistic pass 25 -> 21 us
  // (8192 x 2048) and 146 -> 122 us (16384 x 7168).  The SwiGLU backward is 3-7 % slower when its
  // transposed stores carry it; the plain blockwise quantiser takes none (13.2 us at 8192 x 2048
  // against 14.2-16.1 with any), its per-expert form the row-wise codes only, so that an L2 merges the pieces of lines that two
  // row blocks share (us with none / the transposed stores / the row-wise ones / both: 33040 x 2048 in 32 experts 53.4 / 50.0 / 46.8 /
  // 57.2, 16000 x 4096 in 16 53.2 / 53.1 / 45.8 / 62.7, 16000 x 7168 in 64 104.9 / 122.0 / 90.2 / 124.5, 28500 x 1408 in 128 33.3 / 33.1 /
  // 32.2 / 36.4, 65536 x 1024 in 256 55.7 / 53.6 / 51.0 / -; with a plan 65536 x 512 in 256 33.2 / 29.8 / 27.8 / 33.5); the RMSNorm tile kernel
  // with the statistic given (transposed output only, x read once: nothing to protect) none
  // (16384 x 7168: 66.6 -> 59.5 us).  Transposed rows that do not start on 16-byte boundaries
  // (M or a per-expert count that is not a multiple of 16) are where the hint on the transposed
  // stores costs most: the SwiGLU forward takes 100 instead of 70 us at 16300 x 3584 with it (and
  // gains 3 % at 8192 x 2048), so it keeps the hint on the row-wise codes only; the RMSNorm tile
  // kernel gains 18 % from it on rows that start on lines and loses on others, which go out in pieces from two row blocks that
  // an L2 would merge: 14160 x 5120 46.0 us without / 68.9 with it, 9104 x 4096 24.2 / 32.3, 14160 x 5632 49.8 / 66.0; rows on half
  // lines are level (14144 x 4096 36.7 / 36.6, 4160 x 2048 8.5 / 7.7).
  static constexpr int kStoreHintBlockwise = 0;
  static constexpr int kStoreHintBlockwiseBatched = 2;
  static constexpr int kStoreHintPermute = 3;
  static constexpr int kStoreHintSiluFwd = 2;        // both layouts, single matrix
  static constexpr int kStoreHintSiluFwdRows = 2;    // row-wise layout only
  static constexpr int kStoreHintSiluFwdCols = 1;    // transposed layout only
  static constexpr int kStoreHintSiluFwdBatched = 2;
  static constexpr int kStoreHintSiluBwd = 2;
  static constexpr int kStoreHintSiluBwdBatched = 2;
  static constexpr int kStoreHintRmsnorm = 3;        // both layouts (x is read again: protect it)
  static constexpr int kStoreHintRmsnormCols = 0;    // transposed output only, statistic given

  // ---- the bulk loads carry the hint (3-5 % on the SwiGLU kernels and the RMSNorm tile kernel,
  // 12 % on the plain blockwise quantiser, 6 % on its per-expert form; the gathered rows, which
  // several experts read, are 27 % slower with it)
  static constexpr bool kLoadHintBlockwise = true;
  static constexpr bool kLoadHintBlockwiseBatched = true;
  static constexpr bool kLoadHintPermute = false;
  static constexpr bool kLoadHintSiluFwd = true;
  static constexpr bool kLoadHintSiluFwdBatched = true;
  static constexpr bool kLoadHintSiluBwd = true;
  static constexpr bool kLoadHintSiluBwdBatched = true;
  static constexpr bool kLoadHintRmsnorm = true;

  // ---- the lean form of the quantiser and of the tile loads (scalar bases, paired
  // column-maximum reduction; every other tile kernel uses it, -3 to -9 %) in the PLAIN
  // blockwise quantiser, which is 7 % slower with it (48 -> 51 us at 65536 x 1024); the
  // per-expert form takes it (Zipf counts: 60.6 -> 57.9 us)
  static constexpr bool kLeanBlockwise = false;

  // ---- rows per thread (workgroup = 2048 / rows threads).  8 rows per thread spread the
  // per-thread overhead over twice the elements, 4 rows per thread put twice the waves on a CU.
  // The SwiGLU forward needs 135 registers with 8 and loses 5-9 %.  The RMSNorm tile kernel
  // measured 3-4 % ahead with 8 (93 registers, five 256-thread workgroups per CU) when its
  // division took three operations per element; with the current two it is level at
  // 16384 x 7168 (110.5 us either way, 58.9 / 58.5 us with the statistic given) and 2 % behind at
  // 8192 x 2048 (18.3 / 18.0 us), so it runs with 4.
  static constexpr int kRowsPerThreadSiluFwd = 4;
  // Rows of a 128x128 tile per thread in the plain blockwise quantiser: 8 (256 threads) for the
  // dense form (4 rows: 13.2 -> 13.9 us on 8192x4096), 4 (512 threads) for the per-expert form,
  // which waits on its lookup and gains from more waves per CU (31.3 -> 30.9 us, 32 experts).
  static constexpr int kRowsPerThreadBlockwise = 8;
  static constexpr int kRowsPerThreadBlockwiseBatched = 4;
  static constexpr int kRowsPerThreadRmsnorm = 4;
  // waves (one row each) per workgroup of the statistic pass: 18.10 / 18.00 / 18.00 / 18.04 us at 8192 x 2048 and
  // 107.8 / 108.0 / 107.4 / 107.6 at 16384 x 7168 with 1 / 2 / 4 / 8
  static constexpr int kRowstatWaves = 4;
  // per-expert launches that read their tiles from a plan: the packed tiles (last row blocks of at most 64
  // rows) before or behind the others.  65536 rows in 256 experts (Zipf counts), packed first / last:
  // SwiGLU forward 44.2 / 43.2 us, backward 77.7 / 77.4, blockwise quantiser 30.9 / 31.8
  static constexpr bool kPlanPackedFirstSiluFwd = false;
  static constexpr bool kPlanPackedFirstSiluBwd = false;
  static constexpr bool kPlanPackedFirstBlockwise = true;
  static constexpr bool kPlanPackedFirstPermute = false;  // 43.8 / 43.3 us first / last (33040 x 2048 gathered from 16384 rows)
  // One matrix, M no multiple of 128: neighbouring row blocks share lines of the transposed rows, which one L2 merges and two
  // write out twice. In grid order a column block stays on its XCD where their number is a multiple of 8; elsewhere every XCD
  // takes an eighth of the tiles counted column block after column block. us of the tile kernel in grid order / so: RMSNorm
  // 15935 x 5248 62.8 / 52.8, 8120 x 2176 14.8 / 11.8, 3046 x 1408 7.4 / 6.8, 6537 x 768 7.7 / 7.2, 1303 x 6272 8.4 / 7.7, plain
  // quantiser 9040 x 3968 31.4 / 27.6, 4720 x 6528 27.8 / 25.4.
  // RMSNorm with both outputs, rows on half lines, 4096 columns and 3072 tiles or more: eighths of the tiles in grid order (us of
  // a call, so / by columns: 11328 x 5504 64.7 / 68.7, 15040 x 5504 84.2 / 90.0, 12352 x 4992 63.7 / 65.7, 14144 x 6528 91.8 / 94.2,
  // 18496 x 6016 109.6 / 112.3, 16320 x 5248 92.1 / 86.9 and 84.7 / 88.9; fewer tiles 8256 x 3456 31.9 / 31.2, 4160 x 5248
  // 26.8 / 26.2).
  // Column blocks in eights: rows that share lines anywhere take grid order at all sizes. us of the transposed output, statistic
  // given, eighths / grid order: 14352 x 4096 38.9 / 36.8, x 6144 55.1 / 51.0, x 7168 63.1 / 58.4, x 8192 78.1 / 63.5, x 5120 45.0 / 44.0,
  // but within 80 rows of 16384 16400 x 4096 42.2 / 42.7, 16336 x 5120 47.5 / 51.2, 16464 x 7168 68.5 / 72.9 (x 8192 90.5 / 78.6).
  // One block of columns more or less than a multiple of 16384: rows start 32 KB apart but for 256 bytes, and a walk down a column
  // block is the slower one. us in grid order / by columns: plain quantiser 1040 x 32640 36.2 / 45.0, 2064 x 16256 36.8 / 40.5, 4112 x
  // 16512 56.8 / 68.5 (transposed only 46.3 / 54.4), but 4112 x 16128 54.4 / 50.3, x 16640 56.0 / 53.0, 4112 x 8064 35.8 / 34.0, 2064 x
  // 24448 51.2 / 47.2; SwiGLU forward 2064 x 16256 43.2 / 51.9, 528 x 32640 24.9 / 29.1, but 2064 x 16128 42.9 / 39.6.
  // The plain quantiser, with the least work in a tile, only from so many tiles on; us of a call with a weight's quantiser: 14800 x 1920
  // (1740 tiles) 29.4 / 26.9, x 1664 (1508) 25.2 / 24.3, x 1408 (1276) 20.75 / 20.96, x 1152 (1044) 20.4 / 19.8, x 896 (812) 16.0 / 15.6,
  // x 768 (696) 14.0 / 14.3, x 640 (580) 13.75 / 13.96, 6000 x 1920 (705) 14.55 / 14.69: up to 1276 it goes either way
  static constexpr int kBlockwiseByColumnsTiles = 1408;
  // The SwiGLU forward from so many tiles on, and where rows don't start on half lines. us of the kernel, both layouts [transposed
  // only], grid order / by columns: 3001 x 1408 (264 tiles) 10.4 / 10.3 [9.3 / 9.0], 5000 x 3200 (1000) 21.9 / 20.5 [21.6 / 19.9],
  // 8120 x 2176 (1088) 25.8 / 24.3, 14800 x 1920 (1740) 36.9 / 34.1 [40.3 / 37.1], 16336 x 5248 (5248) 97.4 / 94.8 [135 / 104]; 1040 x
  // 1408 (99) 6.57 / 6.75, 2160 x 1408 (187) 7.41 / 7.56; half lines: 4160 x 2944 15.8 / 16.3 [13.1 / 13.4], 14144 x 1664 27.3 / 28.7
  // [24.6 / 25.2], x 3456 53.1 / 55.3 [51.6 / 52.7], but 16320 x 2944 56.1 / 54.0 [59.3 / 49.5], where rows start 16 KB apart but
  // for one half line. At 9 row blocks and 513 to 567 tiles it loses up to 8 % (1040 x 7552 13.2 / 13.8).
  static constexpr int kSiluByColumnsTiles = 256;
  // row blocks per run that an XCD works on (xcd_runs; 0: every eighth tile).  Same sizes, planned launches with
  // 0 / 2 / 4 / 8 / 16: SwiGLU forward 43.4 / 41.2 / 40.8 / 40.7 / 40.8 us, backward 76.5 / 76.1 / 75.5 / 75.3 / 76.2,
  // blockwise quantiser 30.9 / 30.3 / 29.9 / 29.9 / 29.8.  Launches that scan the counts, 0 / 2 / 4 / 8: forward
  // 44.4 / 45.2 / 45.1 / 45.6, backward 80.4 / 78.4 / 78.4 / 79.4, blockwise 31.1 / 32.2 / 32.4 / 32.7,
  // gather + pad + quant 47.0 / 48.8 / 49.4 / 50.8: only the backward gains there
  static constexpr int kXcdRowsPlanned = 8;
  static constexpr int kXcdRowsSiluBwdCounts = 4;
  // gather + pad + quant with a plan: runs of 8 row blocks per XCD 50.6 us, grid order 44.8, column sweeps (-1:
  // XCD X takes the column blocks X, X + 8, .. one after the other, so that what it gathers from while it works
  // on one of them is a 256-byte strip of the source: 4.2 MB for 16384 source rows, the size of its L2) 43.8;
  // the launch that scans the counts 45.6
  static constexpr int kXcdRowsPermutePlanned = -1;
  static constexpr bool kStartPriorityRmsnorm = true;
  // RMSNorm + quant in two passes, both passes giving XCD X (workgroup number mod 8) the X-th eighth of the rows,
  // the statistic pass walking its eighth from the end and the tile kernel from the start: what the tile kernel
  // reads first is what the same XCD's L2 read last.  Rows a multiple of 128; where
  // an eighth is not a whole number of row blocks the two passes' eighths differ by less than one.
  // us without / with: 2048 x 2048 8.8 / 7.9, 4096 x 2048 11.7 / 10.6, 8192 x 2048 17.9 / 16.6, 3072 x 4096
  // 14.6 / 13.3, 4096 x 7168 30.2 / 27.9, 8192 x 4096 33.0 / 32.0, 16384 x 2048 33.2 / 31.7, 8192 x 7168
  // 55.8 / 52.9, 16384 x 4096 63.4 / 62.7, 32768 x 2048 63.6 / 63.3, 16384 x 7168 108.1 / 109.6: up to this
  // many bytes of input.  Eighths of broken row blocks: 640 x 4096 8.3 / 8.0, 1152 x 2048 8.0 / 7.6, 2176 x 5120
  // 15.0 / 14.1, 4224 x 5120 24.2 / 22.7, 8064 x 2048 17.9 / 16.7, 4992 x 7168 35.8 / 34.0, 10112 x 7168 68.6 / 65.2.
  // With rows that are no multiple of 128 the transposed rows share lines between row blocks and the grid order
  // is better: 1000 x 2048 8.1 / 8.5, 4104 x 5120 26.9 / 28.8, 6001 x 4096 30.4 / 32.6, 5000 x 7168 42.4 / 45.7
  static constexpr long long kRmsnormByXcdMaxBytes = 160ll << 20;
  // 16-byte chunks per lane, matrix and step in the bf16 SwiGLU backward (three matrices are read):
  // 29.0 / 30.4 / 28.7 / 35.5 us with 2 / 3 / 4 / 8 at 8192 x 4096
  static constexpr int kSwigluBwdRowsUnroll = 4;
  // RMSNorm + row-wise quant of more than 2048 columns (us 2 / 3 / 4 chunks a thread, one row at once). Up to so many
  // rows (n <= 3072, <= 6144, above) two chunks a thread: 1 x 7168 2.56 / 2.82 / 2.94, 256 x 5120 3.40 / 3.57 / 3.73,
  // 1500 x 2560 5.12 / 5.47 / 5.70, 700 x 5632 5.46 / 5.33 / 5.81, 1500 x 6656 9.09 / 9.35 / 9.09. Beyond, what leaves
  // few lanes without a chunk: 3001 x 2560 7.48 / 7.42 / 7.80, 3001 x 4096 9.72 / 10.2 / 9.88, 4104 x 4608
  // 15.3 / 13.8 / 14.2, 3001 x 5632 14.0 / 12.6 / 12.8, 4104 x 6656 20.3 / 20.2 / 18.9. From there 256 threads with one row
  // take the kernel of the narrow rows, which unpacks gamma while the row is on its way, where more registers (54 to 84 for
  // 31 to 52) still leave a CU five to eight workgroups (us that one / the other: 4104 x 3968 12.1 / 12.4, 8192 x 4096
  // 21.0 / 22.4, 4104 x 5120 14.7 / 15.6, x 6144 16.9 / 17.9, 3001 x 7168 15.5 / 15.9; fewer rows 1024 x 3584 5.40 / 5.28, and
  // 2000 x 5120 9.43 / 9.26, where a CU holds seven of the eight rows that it has).
  static constexpr int kRowQuantTwoChunksNarrow = 2000, kRowQuantTwoChunks = 512, kRowQuantTwoChunksWide = 1500;
  // Up to so many rows one at once, then two (us one / two). 128 threads of three chunks (n <= 3072): 7000 x 3072 15.2 / 16.2,
  // 8192 x 2560 15.6 / 15.5. 192 of three (4096 < n <= 4608): 4104 x 4608 14.2 / 15.0, 8192 x 4608 25.1 / 24.8. 256 threads:
  // 8192 x 3968 21.0 / 21.8, 8192 x 5120 25.9 / 26.4, 8192 x 6144 29.3 / 30.0, 12288 x 6656 47.0 / 46.2, 16384 x 3968 36.6 / 35.9,
  // 16384 x 5120 48.2 / 46.4, 16384 x 7168 64.7 / 63.3.
  static constexpr int kRowQuantOneRow128 = 8000, kRowQuantOneRow192 = 4500, kRowQuantOneRow256 = 8192;
  // One row at any number of rows where they start a multiple of 4 KB apart (16384 x 4096 38.0 / 40.4, x 6144 57.1 / 57.4, x 8192
  // 73.0 / 78.7, 12288 x 8192 58.2 / 64.3, but x 6144 42.7 / 42.6; their neighbours gain by two: 16384 x 3968 36.6 / 35.9),
  // and beyond this many columns (8192 x 7680 36.3 / 37.9, x 8064 38.6 / 40.5, 12288 x 8064 56.0 / 57.8).
  static constexpr int kRowQuantWidest = 7168, kRowQuantPitch = 2048;
  // Rows of a workgroup of the RMSNorm backward where 512 workgroups are not reached. It writes one partial row of
  // dgamma and walks its rows one after the other, so that eight each (before) left most of the chip idle. Up to 2048
  // columns one row for each of the four waves (us 8 / 4 / 1 rows: 32 x 2048 7.7 / 6.4 / 6.8, 512 x 2048 8.8 / 7.4 /
  // 9.2, 1024 x 640 7.2 / 6.3 / 7.0). Wider rows take the whole workgroup: one workgroup per CU up to 1024 rows, then
  // three rows each (8 / 4 / 3 / 2 / 1 rows: 32 x 7168 16.2 / 10.3 / 9.3 / 7.9 / 6.7, 512 x 2944 13.8 / 9.8 / 8.5 / 8.5 /
  // 9.7, 1024 x 4096 15.7 / 12.3 / 13.0 / 13.3 / 13.3, 1448 x 5120 20.2 / 18.2 / 18.0 / 18.4 / 18.3).
  static constexpr int kRowBwdRowsNarrow = 4, kRowBwdOnePerCu = 1024, kRowBwdRowsWide = 3;
  // the same in the wide-row RMSNorm backward with one chunk per thread (2048 < n <= 4096: 70.4 -> 66.9 us at
  // 16384 x 3072, 78.5 -> 76.4 at 16384 x 4096); with two chunks the second register set spills
  static constexpr bool kPrefetchRowBwdWide = true;
  // 1x128 groups per thread and step of the plain group quantiser (their loads are in flight together):
  // 10.3 / 10.5 / 13.0 us with 1 / 2 / 4 at 8192 x 2048, where a thread has two groups in all
  static constexpr int kGroupQuantUnroll = 1;

  // SwiGLU + row-wise quant, dense: up to so many 1 x 128 groups per row that 16 lanes take, the rows kernel with
  // one row, then with two.  32768 groups are 2048 workgroups of 256 threads: what 256 CUs hold at once.  Past two
  // rows the tile kernel is ahead: 4096 x 4096 (131072 groups) 16.29 us, rows kernel 17.3 / 16.5 / 17.0 with 1 / 2 / 4.
  static constexpr int kSiluRowsGroupsPerRow = 32768;
  static constexpr int kSiluRowsPerTeamMax = 2;

  // ---- the SwiGLU backwards widen row s of their packed inputs after row s-1 is done (fence_values):
  // without it the per-expert form needed 136 registers under its cap of 128 and spilled; with it (and no
  // branch around the arithmetic) 105, the single-matrix form 100
  static constexpr bool kPinBwdRowsBatched = true;
  static constexpr bool kPinBwdRows = true;

  // ---- row kernels: the outputs are written once (-3 to -7 % with the hint on the RMSNorm
  // backward, the bf16 SwiGLU rows and the 128x128 block quantiser); the loads of rows that a
  // kernel reads once carry it too; RMSNorm + row-wise quant gives every XCD one contiguous
  // eighth of the rows (13.0 -> 12.4 us at 8192 x 2048)
  static constexpr bool kStoreHintRows = true;
  static constexpr bool kLoadHintRows = true;
  static constexpr bool kXcdContiguousRowQuant = true;

  // ---- router kernels: hint on the stores of y and the codes
  static constexpr bool kStoreHintRouter = true;
  // Which router kernel, by the number of workgroups of 64 rows x 64 logits the call has; us of the kernel alone, few-rows
  // / 64-logit / 128-logit form.  Up to 80 of them, 256 CUs are mostly idle and the 16-row form spreads the rows further,
  // at every K alike: 1024 x 256 (64 of them) x 1024 7.7 / 11.9 / 16.4, x 2048 13.6 / 18.8 / 26.1, x 7168 33.0 / 52.8 /
  // 74.4; 1536 x 256 (96) x 1024 10.6 / 12.0, x 2048 18.6 / 18.9, x 7168 48.0 / 53.6; 2048 x 256 (128) x 1024 13.2 / 12.3,
  // x 2048 23.3 / 19.1, x 7168 61.7 / 55.0; fp32 weight (no 128-logit form): 64 of them x 2048 18.5 / 22.0, x 7168 48.6 /
  // 62.9, 96 x 2048 26.2 / 22.1, x 7168 72.0 / 64.5.  As long as the 64-logit workgroups fit the chip at once they halve
  // a workgroup's work: 4096 x 256 (256) x 1024 13.1 / 17.2 (64- / 128-logit), x 2048 21.0 / 27.2, x 7168 68.0 / 83.3;
  // beyond, the 128-logit form turns x into operands half as often: 4224 x 256 (264) x 1024 23.1 / 17.2, x 2048
  // 37.2 / 27.3, x 7168 114.9 / 81.9.
  static constexpr int kRouterFewRowsMax = 80;
  static constexpr int kRouterNarrowMax = 256;
  // The 32-row form against these two by rounds (workgroups over 256 CUs, and over what the CUs hold): one of its rounds
  // costs (k blocks + a) / b of a round of 64-row workgroups, with a, b = 25, 20 where one fits a CU (512 logits,
  // 256 of an fp32 weight), 12, 20 with 256 of a bf16 weight, 34, 40 (fp32 10, 12) with 128.
  // One walk over K for all logits is ahead where K is short and where 64 rows are just too many for a round.
  // us 64-row / 32-row form: 4224 x 512 x 1024 29.5 / 22.0, x 2048 48.4 / 43.4, x 4096 84.7 / 86.3, 4096 x 512 x 1024
  // 16.9 / 22.4, 12288 x 512 x 2048 81.0 / 95.6; fp32 4224 x 256 x 1024 26.6 / 21.2, 4096 x 256 x 1024 15.3 / 21.2,
  // 8320 x 128 x 1024 31.6 / 27.0, 8192 x 128 x 1024 18.2 / 22.0; 6144 x 384 x 2048 51.5 / 40.6, 5120 x 384 x 2048
  // 29.0 / 32.2; 16384 x 256 x 1024 39.4 / 33.1, 8192 x 256 x 1024 20.3 / 18.7, x 2048 36.0 / 41.6.
  // k blocks up to which it is ahead in one round of either (4096 x 512 x 128 8.9 / 7.4, x 256 10.0 / 9.6, x 512
  // 12.2 / 13.7; 4096 x 256 x 256 7.7 / 7.4, x 512 9.2 / 9.9)
  static constexpr int kRouter32ShortK = 2;
  // From this K on the 64-row x 128-logit form of a bf16 weight has its waves in two roles where the logits are whole 256s (N = 128:
  // 64 rows for four waves to quantise). us 64-row form / two roles: 8192 x 256 x 1024 18.7 / 19.0, x 1280 23.6 / 23.7, x 1536
  // 26.9 / 25.5, x 2048 34.3 / 32.0, 4224 x 256 x 1280 19.5 / 19.3, x 1536 21.9 / 19.8, x 3072 37.3 / 37.0, 8192 x 512 x 4096
  // 94.5 / 84.6, 8320 x 128 x 2048 35.8 / 37.5, 4096 x 384 x 3072 35.2 / 38.6, x 4096 48.5 / 47.6. K blocks that do not come
  // out even over the four multiplying waves, and rows of a few more than the 16 that are held, are carried by 512 logits and
  // more only: 6144 x 256 x 1664 25.1 / 27.1, x 2176 30.7 / 33.7, 4224 x 256 x 4224 51.4 / 53.2, 8192 x 512 x 2176 60.4 / 57.4, 4224 x
  // 512 x 3200 70.3 / 62.3.
  static constexpr int kRouterTwoRolesMinK = 1536;
  // ... and from this K on it is ahead of the 32-row form too: 16384 x 256 x 1536 45.3 / 48.1 (32-row / two roles), x 2048
  // 65.4 / 60.2, x 3072 83.8 / 80.5, 8320 x 512 x 1536 60.7 / 50.4, x 2048 73.7 / 63.5, 8192 x 1024 x 1536 65.0 / 70.5, x 2048
  // 96.6 / 89.2.
  static constexpr int kRouterTwoRolesAlwaysK = 2048;
};

}  // namespace fq
#endif
