// Dense and grouped GEMM on the register-pipelined tile kernels (gemm_tile.hip).
#pragma once

#include "gemm.hpp"

namespace rte {

constexpr int kTileMinK = 128;      // shortest k range of a workgroup: one tile per LDS stage
constexpr int kTileMaxSplits = 32;
// Products over rows of activations (layout-N A) up to this k are never split, whatever M: a
// 1024 x 512 x 512 product takes 8.8 us in one launch, 12.8 in four splits and their sum; 128 x 512
// x 512 8.7 and 8.6.  (A QKV of 64 rows of 512 pays for its rows' bits: 10.4 us, 9.1 in splits.)
constexpr int kTileRowK = 512;

constexpr int kTileGroupChunk = 2048;  // longest k range of a grouped reduction's workgroup

// Launches a grouped product: GROUP_M with the SwiGLU epilogues (forward: layout-N operands; backward:
// layout-T B, at most 64 neurons) or GROUP_K with the plain store (chunked: gk_chunk <=
// kTileGroupChunk, gk_first, gk_part set).  a_bytes / b_bytes set.
int gemm_tile_group_launch(const GemmArgs& p, int epi_kind, hipStream_t stream, int vec);

// Bytes the partials of a split product of this shape take, in the layouts that take most (the
// estimate gives at most two chip's worth of tiles: 128 MiB, 181 for activation rows above their
// bucket's power of two).
size_t gemm_tile_split_bytes(int M, int N, int K);

// Launches p (MODE_DENSE, operands in plain layouts with a_bytes / b_bytes set) on the tile the
// estimate picks.  EPI_STORE with a workspace of gemm_tile_split_bytes may split the reduction (the
// count is the shape's; with a workspace too small for it there is no split): *splits > 1 then says
// how many fp32 [M, N] partials the launch leaves in ws for the caller to sum in order.
int gemm_tile_launch(const GemmArgs& p, int epi_kind, hipStream_t stream, int vec, void* ws, size_t ws_bytes,
                     int* splits);

}  // namespace rte
