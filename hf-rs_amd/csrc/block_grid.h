// block_grid.h -- launch shape of the block kernels (engine.hip).  (The gradient's
// own, grad.hip, stay at 64 threads: with 256, (fd|dd) asks for a larger private
// segment.)
#pragma once

namespace hfg {

// Workgroups of a block kernel: one thread a block, each workgroup with its own
// 32 KB Boys slice in LDS, five of which fit a CU.  Where the blocks fill the
// chip, 256 threads share a slice (20 waves a CU instead of five) and take
// further blocks in turn; fewer blocks go to workgroups of one wave, so that
// they reach every CU.
struct BlockGrid {
  int blocks, threads;
};
inline BlockGrid block_grid(int ntask) {
  if (ntask < 64 * 2048) return {(ntask + 63) / 64, 64};
  return {ntask / 256 < 2560 ? (ntask + 255) / 256 : 2560, 256};
}

}  // namespace hfg
