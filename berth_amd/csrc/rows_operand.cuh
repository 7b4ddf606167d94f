// Where the MFMA kernels of rows and row blocks (exl3_gemm_rows_kernel.cuh, exl3_gemm_block_kernel.cuh)
// find their A operands: a copy of the rotated rows in the order in which a wave reads them.
#pragma once

namespace berth {

// Element offset of the eight values k .. k + 7 (k a multiple of 8) of `row` in the copy with
// `mt` tiles of 16 rows: [k / 64][row / 16][h = k / 8 % 2][(k / 16 % 4) * 16 + row % 16][8].
__host__ __device__ constexpr size_t rows_operand_offset(int row, int k, int mt)
{
    return ((((size_t)(k >> 6) * mt + (row >> 4)) * 2 + ((k >> 3) & 1)) * 64 + ((k >> 4) & 3) * 16 + (row & 15)) * 8;
}
// elements of the copy of one input, or of one block of 16 * mt rows of it
__host__ __device__ constexpr size_t rows_operand_elements(int size_k, int mt) { return (size_t)size_k * 16 * mt; }

}  // namespace berth
