// Software-pipelined tiled MFMA GEMM for the prompt-pass and encoder projections,
// Y[M, N] = X[M, K] W[N, K]^T with the epilogues of gemm_sk.h and K chunks that all of a tile's workgroups sum up (gemm_pipe_tile.h).
//
// Four waves (2 along the features, 2 along the rows), one per SIMD, own wave tiles of
// up to 128 x 128. What bounds a tile GEMM here is the way from L2 into LDS: 1 KB takes a
// CU 17 - 23 cycles when it comes as whole 128-byte lines (37 as 64-byte pieces), so a K
// step of 64 costs about 1220 cycles of loading against 2048 of MFMA at 256 x 256, 910
// against 1024 at 256 x 128 and 610 against 512 at 128 x 128. Hence the largest tile that
// fills the chip, 128-byte LDS rows, and loads spread evenly over all MFMAs: a burst
// queues up in front of the cache and stalls the wave's in-order MFMA issue.
//
// With one wave per SIMD nothing but this wave's own instruction order hides a latency:
// the fragments of the next K half are read between the MFMAs of the current one (two
// register sets). A stage of 64 K entries runs in two halves:
//
//   half 0 of stage t:  MFMAs | reads of half 1 of t     | W rows of t + NA - 1 -> LDS
//   wait: half 1 read, stage t + 1 landed; barrier (the buffers of stage t are free)
//   half 1 of stage t:  MFMAs | reads of half 0 of t + 1 | X rows of t + NB -> LDS
//
// W and X have rings of their own (NA and NB stages): at 256 x 256 three and two stages of
// 32 KB fill the 160 KB, and half of the loads get a stage and a half to arrive.
// LDS rows are 128 bytes, 16-byte chunk c of row r at place c ^ ((r >> 1) & 7) (swizzled
// on the source address): 16 neighbouring rows of one chunk fall into 16 different
// quarter-banks (no conflicts counted).
//
// Tiles go to the XCDs in contiguous runs, within a run in groups of 4 row blocks with the
// feature block slowest, so the 32 tiles an XCD works on at a time form a 4 x 8 patch:
// 12 tile edges pass its L2 per K step instead of 33 (8192^3: 1290 -> 1365 TFLOP/s against
// groups of 8).
//
// 64 x 64 tiles keep the chip busy where 128 x 64 leave half of it idle: 80 KB of rings, a K step of 16 KB (0.18 us, 128 x
// 64 0.27). 1500 x 512 x 2048 11.1 -> 8.9 us, x 512 5.7 -> 4.7, 300 x 1280 x 1280 9.0 -> 6.6, 200 x 3072 x 2048 11.9 -> 9.0.
//
// Tiles of 160 rows are for what pads the others: 320 rows are five sixths of two tiles of 192. 320 x 28672 x 4096 76.1 -> 73.0 us,
// 640 138 -> 127, 1280 x 4096 x 14336 127 -> 118 in two chunks. Four stages instead of three of 128 x 160: 2 % slower.
//
// Workgroups behind the tiles' (AHEAD: a variant, as the others start 0.15 us sooner without the
// question) bring the weights of later launches into the Infinity Cache.
#include "gemm_pipe_tile.h"

// gemm_pipe_ahead.hip, gemm_pipe_split.hip, gemm_pipe_split_ahead.hip
int gemm_pipe_ahead(const GemmSkCall& p, int layout, hipStream_t st);
int gemm_pipe_split(const GemmSkCall& p, int layout, hipStream_t st);
int gemm_pipe_split_ahead(const GemmSkCall& p, int layout, hipStream_t st);

int gemm_pipe(const GemmSkCall& p, int layout, hipStream_t st) {
  if (p.S > 1) return p.ahead_wgs ? gemm_pipe_split_ahead(p, layout, st) : gemm_pipe_split(p, layout, st);
  return p.ahead_wgs ? gemm_pipe_ahead(p, layout, st) : gp_layout<false, false>(p, layout, st);
}
