// Device-side helpers that the backward kernels share (attn_bwd.hip, attn_bwd_head.hip): the per-lane read addresses of
// a tile, the fragments of a row, the stores of a gradient.
#pragma once
#include "attn_common.h"

namespace sma {
namespace {

constexpr float LOG2E = 1.4426950408889634f;

// Chunk swizzle of tiles whose rows are read 16 at a time, 4 chunks each, and transposed, by p = row / 2 % 8.  A 16-byte read serves lanes
// 0-3, 12-15, 20-23 and 24-27 together (then 4-11, 16-19 and 28-31, and the same in the upper half), here rows 0-3 and 12-15 of one chunk and
// 4-11 of its neighbour: the swizzles of these must come in pairs that differ in the last bit.  Transposed reads want the pairs of rows
// 0-7, and those of rows 8-15, different.  (bitrev3 alone: every row read took twice as long.)
__device__ __forceinline__ int swizzle16(int p) { return bitrev3(p ^ ((p & 4) >> 1)); }

// Per-lane LDS read offsets inside a tile (add the tile's base), one for each pattern; l16 = lane % 16, q4 = lane / 16.
//   row     ds_read_b128: row l16, columns 8q4 .. +7; ^ 64: 32 columns further, + 2048: 16 rows          (A operand)
//   col     ds_read_b64_tr_b16: rows 4q4 + (l16 >> 2), columns 4(l16 & 3) .. +3; ^ 32db: 16 columns further, + 2048: 16 rows
//           (A operand = tile^T of which the contraction index 8q4 + 4x + j is row 16x + 4q4 + j, which is what a lane holds of
//           two accumulators of 16 x 16)
struct TileRead {
    uint32_t row, col;
};
__device__ __forceinline__ TileRead make_tile_read(int lane)
{
    const int l16 = lane & 15, q4 = lane >> 4, r = 4 * q4 + (l16 >> 2);
    return TileRead{(uint32_t)(l16 * 128 + ((q4 ^ swizzle16(l16 >> 1)) << 4)),
                      (uint32_t)(r * 128 + ((((l16 & 3) >> 1) ^ swizzle16(r >> 1)) << 4) + ((l16 & 1) << 3))};
}

// The fragments of one row of a matrix (row stride sn elements, D columns): 8 elements at columns
// 32s + 8q4, zeros beyond the row.  `full` (D is the kernel's own head dim) is wave-uniform: the common
// case loads straight.
template <int KS>
__device__ __forceinline__ void load_row(u32x4 (&f)[KS], const uint16_t *mat, uint32_t sn, int row, int q4, int D)
{
    const uint16_t *p = mat + (size_t)row * sn + 8 * q4;
    if (D == 32 * KS) {
#pragma unroll
        for (int s = 0; s < KS; ++s) f[s] = *reinterpret_cast<const u32x4 *>(p + 32 * s);
    } else {
#pragma unroll
        for (int s = 0; s < KS; ++s)
            f[s] = 32 * s + 8 * q4 < D ? *reinterpret_cast<const u32x4 *>(p + 32 * s) : u32x4{0u, 0u, 0u, 0u};
    }
}

// Stores rows row0 .. row0 + 31 of a gradient, in 16 bits or (WIDE) fp32.  A template argument: both ways in
// one kernel, chosen at run time, cost 2 to 4 % of the backward of many short sequences, whose epilogues are a
// large part of it.
template <bool BF16, bool WIDE, int NB>
__device__ __forceinline__ void store_gradient(const f32x4 (&acc)[2][NB], float mult, uint32_t lds_wave, const AttnBwdArgs &a,
                                                 const Rows &r, int bi, int hi, int row0, int lane)
{
    const Rows none = {nullptr, 0u, 0u, 0u};
    const float both[2] = {mult, mult};
    store_rows<BF16>(acc, both, lds_wave, 0, block_dst(WIDE ? none : r, WIDE ? r : none, bi, hi, row0, a.D), !WIDE, WIDE, row0, a.N, lane);
}

}  // namespace
}  // namespace sma
