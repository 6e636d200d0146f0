// Stream format of the sweep kernel (spmm_sweep.hip), shared by the kernel, its generated interpreter
// (gen_sweep_loop.py) and the host-side plan builder (sweep_plan.cpp).  No HIP types.
// build_sweep_plan makes the streams as described first; encode_sweep_streams turns them into what the kernel runs (end of
// this file), which asks for A earlier than the 4 positions that the streams of the plan are numbered for.
#pragma once
#include <stdint.h>

namespace smat {

// Geometry (fixed at compile time).
constexpr int SWEEP_TN = 4;      // n-tiles of 16 per workgroup panel -> 64 columns
constexpr int SWEEP_RW = 8;      // block rows per wavefront
constexpr int SWEEP_WAVES = 8;   // wavefronts per workgroup
constexpr int SWEEP_G = SWEEP_RW * SWEEP_WAVES; // 64 block rows per workgroup
constexpr int SWEEP_S = 16;      // block columns (slabs) per K chunk
constexpr int SWEEP_STAGES = 4;  // chunks resident in LDS
constexpr int SWEEP_AHEAD = 4; // an A operand is loaded this many stream positions before its op
constexpr int SWEEP_LDS_AHEAD = 1; // the B operands of an op are read from LDS this many stream positions before it
constexpr int SWEEP_COPIES = 4;  // copy instructions per wavefront and chunk
constexpr int SWEEP_MIN_OPS = SWEEP_AHEAD; // ops per wavefront and chunk: two chunk boundaries are at least AHEAD positions apart (at most one of them between the load of an A operand and its use), and a boundary finds the copies of the boundary before it older than the A loads of the MIN_OPS positions since
constexpr int SWEEP_OP_PAD = 16;   // descriptors after the end of the last stream (loaded ahead, never executed)
constexpr int SWEEP_CHUNK_PAD = 4; // chunk ids after the last list (loaded ahead, never used)

// One stream entry (16 bytes).  The stream of a (row group, wavefront) is
//     ops of chunk 0, ops of chunk 1, ..., ops of the last chunk, end
// where "chunk" counts positions in the row group's chunk list.  Position i in the stream decides the register
// sets its code uses (i % 8).
//   w0  op: byte offset in vals of the first of two neighbouring blocks (q * 512); both are loaded.  End: 0.
//   w1  LDS byte offset of the 16 rows of B that the first block is multiplied with (lanes 0-31)
//   w2  the same for the second block (lanes 32-63), minus w1 (signed)
//   w3  byte offset, from the first code block, of the code that executes the entry:
//         op      ((i % 8 * 8 + local block row) * 2 + v) * SWEEP_BLOCK_BYTES,  v = 1 when the copies of a chunk
//                 boundary were issued after the load of this op's A operand (the op that opens the chunk and the
//                 AHEAD - 1 positions behind it)
//         first op of every chunk but the first:  SWEEP_TRAMP_BASE + (the op's block index) * SWEEP_TRAMP_BYTES: a
//                 trampoline that runs the chunk boundary code (own copies landed, barrier, next copies) and then
//                 the op's block.  A chunk boundary is no stream position: no operand load is spent on it
//         end     SWEEP_END_OFF
// An op is two blocks of one block row (K = 32 of one MFMA per 16 columns) in the chunk the op is listed under or
// the one before.  LDS offset of a block = sweep_lds_offset(chunk position, block column in the chunk); a half
// that must not contribute (unpaired block, filler op, end) points at SWEEP_ZERO_OFF, 16 KiB of zeros.
struct SweepOp {
    uint32_t w0, w1, w2, w3;
};
constexpr uint32_t SWEEP_STAGE_BYTES = 32768;
constexpr uint32_t SWEEP_ZERO_OFF = SWEEP_STAGES * SWEEP_STAGE_BYTES; // 131072
constexpr uint32_t SWEEP_BLOCK_BYTES = 128;
constexpr uint32_t SWEEP_N_BLOCKS = 8 * 8 * 2;                                       // stream position % 8 x block row x v
constexpr uint32_t SWEEP_TRAMP_BASE = SWEEP_N_BLOCKS * SWEEP_BLOCK_BYTES;            // 16384
constexpr uint32_t SWEEP_TRAMP_BYTES = 8;
constexpr uint32_t SWEEP_MARK_OFF = SWEEP_TRAMP_BASE + SWEEP_N_BLOCKS * SWEEP_TRAMP_BYTES; // 17408: the chunk boundary code
constexpr uint32_t SWEEP_MARK_BYTES = 512;
constexpr uint32_t SWEEP_END_OFF = SWEEP_MARK_OFF + SWEEP_MARK_BYTES;               // 17920

// The streams as the kernel runs them.  Each starts with SWEEP_DEV_HEAD entries that hold, one uint32 after the other, the A
// offsets of its first AHEAD ops (0 behind the last op), where AHEAD = SWEEP_DEV_AHEAD; then come the entries of the plan,
// without the fillers that do not open a chunk as far as SWEEP_DEV_MIN_OPS ops of the chunk are left, with
//   w0  the A offset of op i + AHEAD - 1 (0 behind the last op): the position in front asks for it
//   w1, w2 as in the plan; in streams for row-major B the LDS offsets are those of stages of [16 slabs][16 k][64 columns]
//   w3  op      its block, v = 1 when the copies of a chunk boundary were issued after the load of this op's A operand; the
//               block waits until AHEAD + 4 v vector memory operations are under way, with the copies of two boundaries in
//               between (chunks of less than AHEAD ops) for a little more than it has to
//       first op of every chunk but the first:  sweep_tramp_base + (m * SWEEP_N_BLOCKS + the op's block index) *
//               SWEEP_TRAMP_BYTES, m = min(ops of the chunk before, AHEAD) - SWEEP_DEV_MIN_OPS: so many more A loads than
//               SWEEP_DEV_MIN_OPS may be under way when the boundary's own copies have landed
//       end     sweep_end_off
// Light streams, for row groups whose wavefronts have little to do in a chunk: an op runs in the chunk of its later block or the one after,
// so that the copies of a boundary may take two chunks' time.
//       first op of every chunk but the first:  where copies were issued by the boundary before, sweep_light_base + (l * SWEEP_N_BLOCKS +
//               the op's block index) * SWEEP_TRAMP_BYTES, l = min(ops of the two chunks before, AHEAD) - 2 SWEEP_DEV_MIN_OPS: as many A
//               loads and SWEEP_COPIES more may be under way when the copies of the chunk being entered have landed; where not, as above with the ops
//               of both chunks; both blocks of that op are in the chunk before (its LDS reads are issued before the barrier)
// The two loops (column-major and row-major B) have blocks of different sizes.
constexpr int SWEEP_DEV_AHEAD = 7; // with a ring of eight operands the most there is room for
constexpr int SWEEP_DEV_HEAD = 2;
constexpr int SWEEP_DEV_MIN_OPS = 2; // ops per wavefront and chunk
constexpr int SWEEP_DEV_MARKS = SWEEP_DEV_AHEAD - SWEEP_DEV_MIN_OPS + 1;
constexpr uint32_t sweep_block_bytes(bool row_major) { return row_major ? 192 : SWEEP_BLOCK_BYTES; }
constexpr uint32_t sweep_tramp_base(bool row_major) { return SWEEP_N_BLOCKS * sweep_block_bytes(row_major); }
constexpr uint32_t sweep_end_off(bool row_major) { return sweep_tramp_base(row_major) + SWEEP_DEV_MARKS * SWEEP_N_BLOCKS * SWEEP_TRAMP_BYTES + SWEEP_MARK_BYTES; }
constexpr int SWEEP_LIGHT_MARKS = SWEEP_DEV_AHEAD - 2 * SWEEP_DEV_MIN_OPS + 1;
constexpr uint32_t sweep_light_base(bool row_major) { return sweep_end_off(row_major) + 64; }
static_assert(SWEEP_DEV_AHEAD <= 4 * SWEEP_DEV_HEAD && SWEEP_DEV_AHEAD > SWEEP_DEV_MIN_OPS, "the head holds the offsets of the first ops");

inline uint32_t sweep_lds_offset(int32_t chunk_pos, int32_t slab)
{
    const uint32_t slot = (uint32_t)(chunk_pos % SWEEP_STAGES) * SWEEP_S + (uint32_t)slab;
    return (slot >> 3) * 16384u + (slot & 7u) * 32u;
}
// the LDS offset of the same block in a stage of row-major B
inline uint32_t sweep_lds_offset_row_major(uint32_t offset)
{
    return offset >= SWEEP_ZERO_OFF ? offset : ((offset >> 14) * 8u + ((offset >> 5) & 7u)) * 2048u;
}
inline uint32_t sweep_op_code(int pos, int row, int v) { return (uint32_t)(((pos % 8) * 8 + row) * 2 + v) * SWEEP_BLOCK_BYTES; }
// the same op as the first of its chunk: through the chunk boundary code
inline uint32_t sweep_boundary_op_code(int pos, int row, int v) { return SWEEP_TRAMP_BASE + (uint32_t)(((pos % 8) * 8 + row) * 2 + v) * SWEEP_TRAMP_BYTES; }

} // namespace smat
