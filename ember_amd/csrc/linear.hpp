// What the linear layers' two kernels (linear.hip: up to 64 rows; gemm.hip:
// more) have in common: W's packed layout, and the order in which a product's
// k steps are summed. Both give a row the same bits, whatever the batch.
//
// K's S 32-wide k steps are 8 runs: run r takes steps r, r + 8, .... A run is
// one chain of v_mfma_f32_16x16x32_f16 from zero; the runs' sums are added in
// run order. A K split in slices (linear.hip's gemv_split) does that in each
// slice, with contiguous runs (of s steps: [r s / 8, (r + 1) s / 8)), and adds
// the slices in slice order.
#pragma once

#include "device.hpp"
#include "kernels.hpp"

namespace ember::hip {

constexpr int kLinearRuns = 8;
// Packed W (ember_hip_gemv_pack): for each 16-feature tile and 32-wide k step,
// the MFMA A operand as the 64 lanes take it, 8 halves per lane (lane 16 g + c:
// row 16 tile + c, k 32 step + 8 g ..): one contiguous 1 KiB per load
// instruction of a wave instead of 16 rows of 64 bytes. Rows past N are zero.
constexpr int kPackBlock = 64 * 8;  // halves per (tile, k step)

__device__ __forceinline__ float silu(float g) { return g / (1.0f + expf(-g)); }

int gemv_split(int N, int K);  // K slices of a launch with a workspace: 1, 2 or 4

}  // namespace ember::hip
