// nm_spmm_mc.h — launch arguments shared by the matrix-core SpMM kernels
// (nm_spmm_mc.hip: up to 128 rows per launch; nm_spmm_rows.hip: any number).
#pragma once

#include "nm_gemv_kernel.h"

namespace nm_hip {

// Several products of the same activations in one grid (sibling Linears:
// q/k/v, gate/up): product i owns workgroups first[i] .. first[i + 1] - 1,
// with its own weights, gathered activations, outputs, partials and
// arrival counters, the same tile width, batch and split count.
constexpr int kMcMaxGroup = NM_MC_MAX_GROUP;
struct McGroupArgs {
  SpmmArgs p[kMcMaxGroup];
  int first[kMcMaxGroup];
  int n;
};

// nm_spmm_rows: tiles of kRowsTile or kRowsTallTile rows x kRowsTile outputs,
// fp32 partials of a split's tile.
constexpr int kRowsTile = 128, kRowsTallTile = 256;

void launch_rows_product(int dtype, const McGroupArgs& g, int bm, int mt, int blocks, hipStream_t st);

}  // namespace nm_hip
