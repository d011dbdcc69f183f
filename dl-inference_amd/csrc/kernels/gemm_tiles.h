#pragma once

// Workgroup size and tile order shared by the MFMA GEMMs (mfma_gemm.hip, mfma_gemm_f32.hip).
#include "common.h"

namespace dk {

constexpr int kGemmThreads = 256;

// ---- tile order ----------------------------------------------------------------------------------
// Workgroups are handed to the 8 XCDs round robin by linear id, so XCD x gets the x-th contiguous
// range of tiles of a grouped order (kGroupRows row blocks per group, row blocks fastest): the
// tiles one XCD runs at once share A row blocks and B column blocks in its L2. (gridDim.x, y) =
// (column tiles, row tiles); each blockIdx.z slice (a K split) is mapped the same way. At
// 8192 x 896 x 4864 (down_proj over a 4 x 2048 prompt) this took the bf16 GEMM from 110 to
// 79 us; with the plain order, the 7 column tiles of a row block ran on 7 XCDs, each fetching
// the row block from memory.
constexpr int kGroupRows = 8;

__device__ __forceinline__ void groupedTile(int BM, int BN, int64_t& r0, int64_t& c0) {
  const uint64_t nn = gridDim.x, nm = gridDim.y, T = nn * nm;
  const uint64_t L = blockIdx.x + nn * blockIdx.y;
  const uint64_t x = L % 8, l = L / 8;
  const uint64_t g = x * (T / 8) + (x < T % 8 ? x : T % 8) + l;  // a bijection of [0, T)
  const uint64_t per = kGroupRows * nn, grp = g / per, first = grp * kGroupRows;
  const uint64_t gs = nm - first < kGroupRows ? nm - first : kGroupRows;
  const uint64_t in = g - grp * per;
  r0 = static_cast<int64_t>(first + in % gs) * BM;
  c0 = static_cast<int64_t>(in / gs) * BN;
}

}  // namespace dk
