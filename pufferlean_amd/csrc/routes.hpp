// Which form of a kernel a call takes, by sizes and types (host code, no device types). The reasons and the
// measured times on both sides of each line stand here, at the line. All forms of one call compute the
// same values to their tolerance, so a line's place is a matter of time only.
#pragma once

namespace ph {

// ---- GEMM, reductions of k >= 4096 with a small output ------------------------------------------------
// 64x64 split tiles instead of 128x128 ones, for outputs at most 64 wide or tall with fp32 operands (128x128 tiles
// are mostly padding there) and, in fp32 math, where 128x128 splits of >= 512 leave most CUs idle. fp32 math is bound
// by the matrix core, so the smaller tile wins until its tiles outnumber half the CUs and no split is left
// (TN 128x28x32768 69 -> 17 us, 288x96x6699 89 -> 19, 512x64x262144 457 -> 317; but NT 64x8256x16384 397 -> 432).
// With bf16 products the operand reads bound it: 64x64 tiles re-read the wide operand's partner once per tile and
// run fewer, longer splits, so they stay to few tiles or short reductions (64x64x65536 20 -> 12 us, 128x64x262144
// 49 -> 36, 64x1024x8192 20 -> 14.5, 64x4096x8192 38 -> 35; but 64x8256x4096 41 -> 58, 512x64x32768 23 -> 26,
// 512x32x262144 111 -> 131).
inline bool gemm_small_splits(bool f32_math, bool f32_operand, bool trans_b, long M, long N, long K) {
  if (!f32_operand) return false;
  const long tiles64 = ((M + 63) / 64) * ((N + 63) / 64), tiles128 = ((M + 127) / 128) * ((N + 127) / 128);
  if (f32_math && tiles128 * (K / 512) < 256) return true;
  if (M > 64 && N > 64) return false;
  if (f32_math) return tiles64 <= 128 || !trans_b;
  return tiles64 <= 2 || tiles64 * K <= 131072 || (tiles64 <= 64 && K <= 8192);
}

// Threads per element of the split-K fold (each adds a contiguous range of the splits). One thread per element
// has sixteen loads in flight and reads whole rows of a split; more threads shorten its chain of loads but read
// shorter runs of a row. From 64 splits four are faster (64x64 of 128 splits 17.8 -> 14.4 us with the product, 256x256
// of 64 31.6 -> 30.3), sixteen only for outputs of a few blocks and 256 splits (8x8x262144 19.8 -> 17.0, but 128x128 of
// 128 splits 17.0 -> 18.3); at 16 and 32 splits one is (64x64x8192 12.7 against 13.4).
inline int fold_threads(int splits, long MN) {
  if (splits >= 256 && MN <= 4096) return 16;
  return splits >= 64 && MN <= 65536 ? 4 : 1;
}

// ---- Categorical sampler ----------------------------------------------------------------------------------
// Logits of a row held in registers (4, 8, 16 or 32; every one is loaded and exponentiated, so the least that holds
// the row), or 0: the row is read from memory in each pass. That form stays for one action and past 32.
// fp32, 4 actions: 4096 rows 3.7 us in passes, 3.1 in 16 registers, 2.4 in 4; 1048576 rows 12.7, 15.2 and 8.3
// (one action 7.0, 13.4 and 7.6).
inline int sample_registers(long A) {
  if (A <= 1 || A > 32) return 0;
  return A <= 4 ? 4 : A <= 8 ? 8 : A <= 16 ? 16 : 32;
}

// ---- V-trace scan ----------------------------------------------------------------------------------------
// Whether a batch takes the tiles of 16 or 64 segments x chunks of 64 steps staged through LDS, or one lane (two for
// the largest fp32 batches) per segment walking its steps.
// Time-major: from 32768 segments (f64 past 24576) the lanes alone fill the chip and stream whole rows (fp32 65536x64
// 18.6 us against 26.1 tiled). Below that a lane is one chain of dependent load rounds that grows with T, and a
// chunk costs the same whether its 64 steps are real or not: short horizons stay with the lanes (fp32 4096 segments,
// lanes / tiles: T = 4 3.0 / 3.2 us, 8 3.4 / 3.3, 64 13.1 / 6.1; 16384, tiles of 64 segments: 16 5.0 / 5.7, 32 8.0 /
// 6.6; f64 64: 8 3.4 / 3.7, 188: 11 4.5 / 3.9, 8192: 8 4.3 / 4.5, 16384: 12 5.8 / 6.0), and where the two are close a
// chunk that is mostly padding decides (fp32 32767 segments: 64 16.0 / 12.6, 72 16.9 / 17.6, 96 21.5 / 19.5).
// Segment-major: lanes read T elements apart, so tiles win sooner (fp32 64: 4 2.7 / 3.1; 4096: 4 5.3 / 3.3; 16384: 4 5.3 /
// 6.0, 8 9.9 / 6.1; 65536: 8 10.8 / 12.1, 12 15.4 / 12.7; f64 256: 4 3.0 / 3.7, 8 5.9 / 3.8; 32767: 8 8.4 / 9.6).
inline bool vtrace_tiled(bool f64, bool time_major, long B, long T) {
  if (!time_major) return T >= (f64 ? (B <= 16384 ? 8 : 12) : (B > 128 && B <= 8192 ? 4 : B <= 32768 ? 8 : 12));
  const long pad = (T + 63) / 64 * 64 - T;
  if (B <= 8192) return T >= (f64 ? (B <= 4096 ? 10 : 12) : 8);
  if (f64) return B <= 16384 ? T >= 16 : B <= 24576 && 2 * pad <= T;
  return B <= 24576 ? T >= 32 : B < 32768 && 2 * pad <= T;
}

// ---- Prioritised replay, segment-major columns ------------------------------------------------------------
// The gather's tiles of 16 segments x 64 steps: rows of at least 16 steps (shorter ones fill too little of a 64-step
// run, and a whole row is a cache line or less; 64 segments f64: T = 16 10.8 -> 8.9 us, 17 10.3 -> 9.1). The upper bound
// keeps a tile's steps within int.
inline bool gather_tiled(bool time_major, long T) { return !time_major && T >= 16 && T <= 1L << 30; }
// Gather blocks whose (count, mean, M2) partials every normalising block merges itself; past that a launch of one block
// does (1024 partials, time-major f64 256 draws x 4096: merged by every block 25.8 us, by one 26.9; 2048, 4096 x 512:
// 78.0 and 76.0, fp32 1024 x 2048 42.1 and 39.6).
inline bool gather_folds(long blocks) { return blocks <= 1024; }
// The per-segment sums add one row per lane out of the tile, 16 lanes of a block at work: one thread per segment keeps
// up while rows are short, and in fp32 while the segments are few (4096 segments, thread / tile: f64 T = 24 2.4 / 2.8
// us, 32 3.4 / 2.6; fp32 32 2.6 / 2.7, 64 3.4 / 2.8; 65536 x 16 2.2 / 4.4; fp32 16 x 4096 55 / 62, 128 x 2048 35 / 33).
inline bool seg_l1_tiled(bool f64, bool time_major, long N, long T) {
  if (time_major || T > 1L << 30) return false;
  return f64 ? T >= 32 : T >= 64 && N >= 128;
}

// The sampler in one workgroup: few segments and draws, where a second launch (3.7 us of host time) costs more than
// spreading the f64 functions saves (one launch / two: 64 segments, 64 draws 5.6 / 6.7 us, 1024 and 512 7.4 / 8.2, 2048 and
// 512 9.2 / 8.7, 2048 and 1024 10.2 / 8.8; but 1024 and 2048 10.6 / 8.1, 3072 and 1024 11.7 / 9.2).
inline bool prio_one_block(long N, long draws) { return N <= 2048 && draws <= 1024; }

// The value / ratio iterate: tiles of 16 draws x 64 steps that compare their draws with every later one, in one launch,
// or two launches through a last-writer table with a wavefront per draw. The comparison costs each block a pass
// over the draws (so a bound on them), the table a launch (3.7 us of host time, which is what bounds a chain of such
// calls issued one by one); a wavefront per draw reads B apart in the timestep-major inputs and is one chain over T.
// f64, table / tiles, over twenty sets of columns in turn (an update's columns are new to the L2): 64 draws of 16 steps
// 4.1 / 5.5 us, 4096 of 16 6.0 / 7.0, 4096 of 32 7.1 / 7.5, 1024 of 64 5.7 / 5.7, 4096 of 64 9.1 / 7.6, 512 of 256 8.1 /
// 6.3, 4096 of 128 13.5 / 8.3; 8192 of 16 7.3 / 10.0, of 32 9.1 / 9.9, of 48 10.7 / 10.2; 16 of 1024 8.0 / 4.0. The
// replay chain of 1363 segments x 71 steps and 100 draws issued one by one: 39.9 us with the table, 36.2 with the tiles.
inline bool iterate_tiled(bool time_major, long draws, long T) {
  if (time_major || T < 16 || T > 1L << 30) return false;
  return draws <= 4096 || (draws <= 8192 && T >= 48);
}

// ---- Newton-Schulz in fp32 ----------------------------------------------------------------------------------
// Whether a matrix takes the batched launches of 32x32 tiles (one per phase) or the GEMM chain. By its shape alone, so that
// a matrix gives the same result alone and in a batch. A tile's k loop is not split over blocks, so a side past 2048
// leaves one chain of over 7 us per phase, and 32x32 tiles re-read their operands too often once there are thousands of
// them (5 steps, chain / launches: 2048x64 234 / 133 us, 1536x1536 2014 / 1219, 2048x1536 2215 / 1480, but 2048x2048
// 2640 / 2690). Around 1024x1024 the chain's products are 64 whole 128x128 tiles, so two or three matrices run side by side
// on their streams: one 510 / 483 us, two 750 / 810, three 970 / 1132; from 1152 on it does not keep up (one 812 / 623,
// two 1165 / 1108). Four of a size depend on how the runtime maps the side streams to hardware queues (four 1536x1536
// 4093 or 5433 / 4441).
inline bool ns_f32_fits(int rows, int cols) {
  const int lo = rows < cols ? rows : cols, hi = rows < cols ? cols : rows;
  return hi <= 2048 && (long)lo * hi <= 3L << 20 && !(lo >= 1024 && hi < 1152);
}

// ---- MinGRU rollout step ----------------------------------------------------------------------------------
// The layer kernel of N rows and H units (H a multiple of 8): blocks of 32 rows with k split over the wavefronts, of
// 128 or 256 rows with the weights in LDS, or the GEMM chain (products, a cell kernel, a padded head).
// A launch takes rounds of as many blocks as run at a time, and a round costs about the same however full: bf16
// products, bound by operand delivery, 256 blocks of any form, a round of 32 / 128 / 256 rows costing about 10 / 18 / 23
// (below 320 units 10 / 28 / 36; steps of two layers, 512 units: 512 rows 31 / 38 / 44 us, 700 44 / 40 / 45, 2048 71 /
// 42 / 48, 4096 126 / 74 / 57, chain 88; 384: 1500 58 / 37 / 43, chain 46). Past 1280 units few rows go to the chain,
// whose split k keeps the chip busy (2048 units, 48 rows 75, chain 60; 200 rows 128-row blocks 82, chain 100).
// fp32 products, bound by the matrix core, 768 blocks of 32 rows or 256 of 128, the chain 256 tiles of 128x128; 256-row
// blocks are never the faster form. Costs of r rounds: 10 r + 1, 8 r + 12 and 11 r + 14 (512 units: 1300 rows 79 / 94 us,
// chain 128; 2048 104 / 95 / 131; 4096 170 / 152 / 201; 328 units, 7072 rows 163 in 128-row blocks, chain 158; 768: 2600
// rows 243 / 204 / 264, 3300 293 / 294 / 274). A chain of less than two rounds is longer than its tiles say, its gaps
// showing. Past 768 units the chain takes the few rows (896: 256 rows 92, chain 95; 300 101, chain 95; 1024: 100 rows
// 100, chain 94, but 1024 rows in 128-row blocks 165, chain 203).
enum RollForm { kRollChain = 0, kRoll32, kRoll128, kRoll256 };
inline RollForm rollout_form(bool bf16, long N, long H) {
  const auto up = [](long a, long b) { return (a + b - 1) / b; };
  const long cols = up(H, 32), b32 = up(N, 32) * cols, b128 = up(N, 128) * cols, b256 = up(N, 256) * cols;
  if (bf16) {
    if (H > 2048 || (H > 1280 && N <= 128)) return kRollChain;
    const long c32 = 10 * up(b32, 256), c128 = (H >= 320 ? 18 : 28) * up(b128, 256),
               c256 = (H >= 320 ? 23 : 36) * up(b256, 256);
    if (c32 <= c128 && c32 <= c256) return kRoll32;
    return c128 <= c256 ? kRoll128 : kRoll256;
  }
  if (H > 2048) return kRollChain;
  if (H > 768 && N <= 768) return H <= 896 && N <= 256 ? kRoll32 : kRollChain;
  const long r32 = up(b32, 768), r128 = up(b128, 256), rc = up(up(N, 128) * up(3 * H, 128), 256);
  if (H > 768) return 18 * r128 + 6 < 22 * rc + 11 ? kRoll128 : kRollChain;
  const long c32 = 10 * r32 + 1, c128 = 8 * r128 + 12, chain = 11 * rc + 14;
  if ((rc >= 2 || r128 >= 2) && chain <= c32 && chain <= c128) return kRollChain;
  return c32 <= c128 ? kRoll32 : kRoll128;
}

}  // namespace ph
