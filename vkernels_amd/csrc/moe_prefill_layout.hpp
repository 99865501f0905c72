// moe_prefill_layout.hpp — every byte offset the prefill kernel (moe_prefill.hip) forms, as
// pure functions of integers.  The kernel calls them; tests/test_prefill_layout.py compiles
// them for the host and walks all workgroups, wavefronts, lanes and K steps of a problem,
// checking that every offset stays inside the buffer it indexes and that the bytes a lane
// reads from LDS as its MFMA operand are the bytes of the row and K block it stands for.
#pragma once

#include <stddef.h>
#include <stdint.h>

#ifndef __HIPCC__
#ifndef __host__
#define __host__
#define __device__
#endif
#endif

namespace vk {

constexpr int kMxRows = 128;        // sorted rows per window
constexpr int kMxUnitRows = 128;    // weight rows per unit
constexpr int kMxWaves = 4;
constexpr int kMxRing = 3;          // K steps of split rows in LDS
constexpr int kMxStepBytes = 8704;  // prepacked bytes of one unit's K step: 8 KiB of codes + 512 of scales

// ring slot that holds the rows of K step `step`, register set that holds its weights
__host__ __device__ constexpr inline int mx_ring_slot(int step) { return step % kMxRing; }
__host__ __device__ constexpr inline int mx_weight_set(int step) { return step % 3; }

__host__ __device__ constexpr inline int mx_kp(int K) { return (K + 127) & ~127; }
__host__ __device__ constexpr inline int mx_units(int stage, int ncols) {
  return stage == 0 ? ncols / 64 : (ncols + kMxUnitRows - 1) / kMxUnitRows;
}
// Row of W (within an expert) that lane row n of tile t of `unit` multiplies; the
// caller checks it against the expert's row count (stage 1's last unit may be ragged).
__host__ __device__ constexpr inline int mx_weight_row(int stage, int ncols, int unit, int t, int n) {
  if (stage == 0) return (t >> 1) * ncols + unit * 64 + (t & 1) * 32 + n;
  return unit * kMxUnitRows + t * 32 + n;
}
__host__ __device__ constexpr inline int mx_window_rows(int block_size) {
  if (kMxRows % block_size == 0) return kMxRows;
  for (int rows = kMxRows; rows > 16; rows -= 16)
    if (block_size % rows == 0) return rows;
  return 16;
}

__host__ __device__ constexpr inline size_t mx_align256(size_t n) { return (n + 255) & ~(size_t)255; }

// ---- prepacked weights: [E][units][K steps] blocks of kMxStepBytes, then [E][units] flags ----
__host__ __device__ constexpr inline size_t mx_packed_body_bytes(int num_experts, int units, int nsteps) {
  return mx_align256((size_t)num_experts * (size_t)units * (size_t)nsteps * (size_t)kMxStepBytes);
}
__host__ __device__ constexpr inline size_t mx_packed_bytes(int num_experts, int units, int nsteps) {
  return mx_packed_body_bytes(num_experts, units, nsteps) + mx_align256((size_t)num_experts * (size_t)units);
}
// first byte of (expert, unit)'s K steps; a step past the end reads the last one again
__host__ __device__ constexpr inline size_t mx_unit_offset(int e, int units, int unit, int nsteps) {
  return ((size_t)e * (size_t)units + (size_t)unit) * (size_t)nsteps * (size_t)kMxStepBytes;
}
__host__ __device__ constexpr inline size_t mx_step_offset(int step, int nsteps) {
  return (size_t)(step < nsteps - 1 ? step : nsteps - 1) * (size_t)kMxStepBytes;
}
// byte of a step's block that load j (0 .. 7: the operand tiles, 16 bytes; 8: the scale
// bytes, 8 bytes) of `lane` starts at
__host__ __device__ constexpr inline int mx_weight_load_offset(int j, int lane) {
  return j < 8 ? (j >> 2) * 4096 + (j & 3) * 1024 + lane * 16 : 8192 + lane * 8;
}
__host__ __device__ constexpr inline size_t mx_flag_offset(int num_experts, int units, int nsteps, int e, int unit) {
  return mx_packed_body_bytes(num_experts, units, nsteps) + (size_t)e * (size_t)units + (size_t)unit;
}

// ---- split rows: row r = `terms` planes of kp bytes; 16-byte piece q of a plane's K step ----
// Copy operation (term, g) of a K step, issued by wavefront `wave`: lane (r, c) = (lane / 8,
// lane % 8) copies piece c ^ r of row (32 wave + 8 g + r) of the window to LDS position c
// of that row.  Source offset within the split rows (grow = the row's index there):
__host__ __device__ constexpr inline uint32_t mx_row_copy_lane_offset(size_t grow, int terms, int kp, int lane) {
  const int r = lane >> 3, c = lane & 7;
  return (uint32_t)(grow * (size_t)(terms * kp)) + 16u * (uint32_t)(c ^ r);
}
__host__ __device__ constexpr inline uint32_t mx_row_copy_step_offset(int term, int kp, int step, int nsteps) {
  return (uint32_t)(term * kp + (step < nsteps - 1 ? step : nsteps - 1) * 128);
}
// LDS destination of lane 0 of that copy (lane l lands 16 l bytes further)
__host__ __device__ constexpr inline int mx_slot_bytes(int terms) { return kMxRows * terms * 128; }
__host__ __device__ constexpr inline uint32_t mx_row_copy_lds(int step, int wave, int terms, int term, int g) {
  return (uint32_t)(mx_ring_slot(step) * mx_slot_bytes(terms) + ((wave * terms + term) * 32 + g * 8) * 128);
}
// ---- operand reads: lane (ln, hh) = (lane % 32, lane / 32) takes K block 2 half + hh of
// row ln of row tile m: 16-byte pieces 2 blk and 2 blk + 1, at positions (2 blk) ^ (ln & 7)
// and that ^ 1.  `which` = 2 half + (0: first piece, 1: second piece). ----
__host__ __device__ constexpr inline uint32_t mx_operand_lane_offset(int which, int ln, int hh) {
  const uint32_t pos0 = (uint32_t)(((2 * hh) ^ (ln & 7)) * 16);
  const uint32_t flip = which == 0 ? 0u : which == 1 ? 16u : which == 2 ? 64u : 80u;
  return (uint32_t)(ln * 128) + (pos0 ^ flip);
}
__host__ __device__ constexpr inline uint32_t mx_operand_tile_offset(int slot, int terms, int m, int term) {
  return (uint32_t)(slot * mx_slot_bytes(terms) + ((m * terms + term) * 32) * 128);
}
// ---- the K loop's schedule, as numbers: the kernel's counted waits and the host-side
// model of them (tests/prefill_layout_check.cpp) are built from these ----
// vector-memory operations a wavefront issues per K step: 4 row copies per term (8 rows
// x 128 bytes each, its row tile's 32 rows), 8 weight loads, 1 scale load
__host__ __device__ constexpr inline int mx_row_ops(int terms) { return 4 * terms; }
__host__ __device__ constexpr inline int mx_step_ops(int terms) { return mx_row_ops(terms) + 9; }
// groups of 4 MFMAs (one operand read each) per K step with `live` row tiles
__host__ __device__ constexpr inline int mx_step_groups(int live, int terms) { return 2 * live * terms; }
// The step's one wait (at most mx_step_ops outstanding: step c + 1 has landed, step c + 2 may be
// on its way) and barrier come at the end of group Q - 3.
__host__ __device__ constexpr inline int mx_wait_group(int live, int terms) { return mx_step_groups(live, terms) - 3; }
// MFMA of step c (4 q + t: the t-th of group q) that operation k of step c + 2 is issued behind:
// evenly over the MFMAs of groups 0 .. Q - 3, so that all of them are ahead of the wait
__host__ __device__ constexpr inline int mx_op_slot(int live, int terms, int k) {
  return k * 4 * (mx_step_groups(live, terms) - 2) / mx_step_ops(terms);
}

// ---- raw weights: [E][rows][K / 2] codes and [E][rows][K / 32] scale bytes, as the checkpoint has
// them.  K is a multiple of 512, so that four K steps of a row's scale bytes are 16 aligned bytes.
// A unit is the 128 weight rows it is above; lane (n, hh) of operand load (half, t) takes the 16
// bytes of K block 2 half + hh of row (t, n) itself. ----
constexpr int kMxRawK = 512;
__host__ __device__ constexpr inline int mx_raw_row(int stage, int ncols, int unit, int t, int n) {
  const int row = mx_weight_row(stage, ncols, unit, t, n), rows = stage == 0 ? 2 * ncols : ncols;
  return row < rows ? row : rows - 1;  // (stage 1's last unit may be ragged)
}
__host__ __device__ constexpr inline uint32_t mx_raw_lane_offset(int row, int K, int hh) {
  return (uint32_t)row * (uint32_t)(K / 2) + 16u * (uint32_t)hh;
}
// (a step past the end: the last one again)
__host__ __device__ constexpr inline uint32_t mx_raw_load_offset(int step, int nsteps, int half) {
  return (uint32_t)((step < nsteps - 1 ? step : nsteps - 1) * 64 + half * 32);
}
// Scale bytes come to a wavefront's own 2 KiB of LDS, 16 of each of its 128 rows at a time.
constexpr int kMxRawScaleBytes = 2048;
// The K loop.  K step c is the half steps 2c, 2c + 1 (the halves of its operand tiles), each with
// half of the row copies.  Half step s multiplies the operands that half step s - 1 has moved onto
// the OCP code points, moves those of s + 1, and issues the 4 weight loads of s + 4, into the
// registers whose codes half step s - 1 has moved, then its part of the row copies of K step
// c + 2, spread evenly.  The scale bytes of step c + 1 are read from LDS in the middle of step c;
// behind the first group after the middle of the last but one step of four the two copies for the
// next four are issued (masked off in the other steps).
__host__ __device__ constexpr inline int mx_raw_weight_set(int half_step) { return half_step & 3; }
__host__ __device__ constexpr inline int mx_raw_ops(int terms) { return 4 + mx_row_ops(terms) / 2; }  // of a half step
__host__ __device__ constexpr inline int mx_raw_groups(int live, int terms) { return live * terms; }  // of a half step
__host__ __device__ constexpr inline int mx_raw_op_slot(int live, int terms, int k) {  // MFMA it follows
  return k * 4 * mx_raw_groups(live, terms) / mx_raw_ops(terms);
}
// operations of a half step that are issued by the end of its group g
__host__ __device__ constexpr inline int mx_raw_ops_through(int live, int terms, int g) {
  int n = 0;
  for (int k = 0; k < mx_raw_ops(terms); ++k) n += mx_raw_op_slot(live, terms, k) < 4 * (g + 1) ? 1 : 0;
  return n;
}
// Waits (operations that may be outstanding).  In the middle of a step: those that have followed
// the scale bytes' copies of the step before, which covers the weights the second half step moves
// (three half steps old).  Before the barrier, behind the last group but two, the rows of step
// c + 1 have landed and the weights that its first half step moves: all but the step's own.
__host__ __device__ constexpr inline int mx_raw_middle_wait(int live, int terms) {
  return 2 * mx_raw_ops(terms) - mx_raw_ops_through(live, terms, 0);
}
__host__ __device__ constexpr inline int mx_raw_row_wait(int live, int terms) {
  return mx_raw_ops(terms) + mx_raw_ops_through(live, terms, mx_raw_groups(live, terms) - 3);
}
// MFMA of a half step behind which word w (0 .. 15) of the other half is moved onto the code points
__host__ __device__ constexpr inline int mx_raw_fix_slot(int live, int terms, int w) { return w * live * terms / 4; }

// Where the raw form is ahead of tile_wide_kernel: many rows for the segments (the rows of one
// expert in a window) they are in, as each segment costs the raw loads whatever its rows.  The number
// of experts is not known here: EM is taken for the bound the sorted order is allocated by, block_size
// - 1 rows of padding for each expert, half of it in use.  (An EM of the padded rows themselves makes
// the experts half as many: calls up to a tenth behind are then taken too.)  Figures: a whole layer,
// tile_wide -> raw.
//   Blocks of 128 and more: 50 rows a window of EM.  8 rows a block of 64 experts 233 -> 294 us, 35
//   298 -> 330, 44 340 -> 351, 55 397 -> 389, 77 753 -> 584, 96 1310 -> 1089; of 256 experts 26 2045 ->
//   2153, 43 2557 -> 2438, 64 4157 -> 3803.
//   Blocks of 16, 32, 64, several experts to a window: 64 rows a segment as well.  Without that an
//   expert's 12 rows in blocks of 16 were taken (256 experts of 7168 x 2048 2012 -> 2833 us, 64 of 4096
//   x 1536 436 -> 830); 64 rows in blocks of 16 3142 -> 3292 and 474 -> 484, 96 in blocks of 32 536 ->
//   563, 64 in blocks of 64 428 -> 441; from the line on 144 in blocks of 16 5154 -> 4866 and 735 -> 670,
//   in blocks of 32 713 -> 634, 96 in blocks of 64 3106 -> 2711 and 404 -> 391.
//   Blocks of 48, 80, 96, 112, each a window of its own: 30 rows a block.  36 rows an expert in blocks of
//   48 2158 -> 2222 and 328 -> 332 us; 48 2870 -> 2833 and 400 -> 396, 64 510 -> 426.
// And no round of workgroups of twice tile_wide's columns that is nearly empty (8 experts of 4096 x
// 4096, 4000 rows, second stage 280 workgroups for 256 compute units: 530 -> 548 us); a second stage
// that runs alone is judged as the whole layer is, so it is refused where only the first stage's would be.
constexpr int kMxRawRows = 50, kMxRawSegmentRows = 64, kMxRawBlockRows = 30;
inline bool mx_raw_pays(long long rows, long long EM, int block_size, int ispp, int hidden) {
  const long long padding = EM - rows;
  if (padding < 0 || rows * kMxRows < kMxRawRows * EM) return false;  // (fewer: an expert map drops rows)
  long long windows = rows / kMxRows + padding / (2 * (kMxRows - 1)) + 1;
  if (block_size < kMxRows && padding > 0) {
    const double run = (double)rows * (block_size - 1) / (double)padding;  // an expert's rows
    const double padded = run + (block_size - 1) / 2.0;
    const bool shared = kMxRows % block_size == 0;
    const double segments = shared ? 1.0 + (padded > block_size ? (padded - block_size) / kMxRows : 0.0)
                                   : padded / block_size;  // an expert's
    if (run < segments * (shared ? kMxRawSegmentRows : kMxRawBlockRows)) return false;
    if (shared) windows = (rows + padding / 2) / kMxRows + 1;
  }
  for (int stage = 0; stage < 2; ++stage) {
    const int units = mx_units(stage, stage == 0 ? ispp : hidden);
    const long long tiles = windows * ((units + kMxWaves - 1) / kMxWaves);
    if (5 * tiles < 3 * ((tiles + 255) / 256 * 256)) return false;
  }
  return true;
}

// ---- epilogue staging: a wavefront's own quarter of the ring ----
__host__ __device__ constexpr inline uint32_t mx_stage_base(int wave, int terms) {
  return (uint32_t)(wave * (kMxRing * mx_slot_bytes(terms) / kMxWaves));
}
constexpr int kMxActPitch = 144;  // stage 0: 64 bf16 of a row + 16 bytes (rows stay 16-byte aligned)

}  // namespace vk
