// f32_tile.h — where k_gemm_f32's loads read (gemm.hip).  Plain constexpr
// functions, so that the bounds are checked on the CPU as well.
#pragma once

namespace ehip {

// A wave loads a 32-input block (128 bytes) of eight rows per instruction,
// eight lanes a row: byte offset of lane `lane`'s 16-byte piece of the i-th
// eight rows in the block, from a buffer's first row of K floats.  The pieces
// of a row are XOR-swizzled over its lanes (LDS banks); a row past the
// buffer's last repeats that one, whose sums are never stored.
constexpr int f32_load_offset(int lane, int i, int K, int rows) {
    const int row = (lane >> 3) * K * 4 + 32 * i * K, last = (rows - 1) * K * 4;
    return (row < last ? row : last) + ((16 * ((lane & 7) ^ (lane >> 4))) ^ (i & 1 ? 64 : 0));
}

}  // namespace ehip
