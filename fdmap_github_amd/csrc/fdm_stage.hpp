// fdm_stage.hpp -- host launchers of the stage kernels (bulk_interior,
// bulk_interior3, bulk_interior_batch).  Their many variants are compiled in
// parts (fdm_stage.hip, one object per part); this header declares one
// launcher per (precision, operator, medium, dissipation, tile shape).
#pragma once

#include "fdm_bulk.hpp"

namespace fdm {

// interior tile shapes (columns x rows) selectable with FDM_TILE
constexpr int kTileShape[3][2] = {{64, 4}, {64, 8}, {128, 4}};

// From this many workgroups on (of 256 threads: six rounds of those that four
// waves per SIMD hold) the FP32 variants for a medium or dissipation run four
// waves instead of three: a longer launch gains more from the tiles' waves than
// it loses by what the points ahead of them spill.  ms a step at three and at
// four: 2 x 401x201 (730 workgroups) 0.066 and 0.070 with dissipation, 0.063 and
// 0.070 in a medium, 2 x 1201x601 (5913) 0.190 and 0.195, 0.177 and 0.178; 2 x
// 1301x651 (7015) 0.208 and 0.198, 0.200 and 0.194, 2 x 2201x1101 0.640 and
// 0.580 (0.590 in three launches a stage), 0.640 and 0.608.
constexpr unsigned kManyWgs = 6 * 1024;

struct StageLaunch {
  hipStream_t stream;
  dim3 grid, block;
  const int4* tiles;
  int shape;
  int full;  // FULL of the kernels
  bool nt_store, ji_calc, mcomp;
  bool many;  // more than kManyWgs workgroups
};

// plane strain: FULL = 1 (manufactured solutions, plasticity), 2 (plasticity)
// or lean, these with non-temporal or normal stores; in FP64 with or without Ji formed in the kernel (ji_calc)
// and FP32-delta metrics (mcomp)
template <typename T, int OP, bool HET, bool DISS, int SHAPE>
void stage2(const StageLaunch& L, const BulkArgs<T>& a, const EdgeArgs<T>& e);

// antiplane shear
template <typename T, int OP, bool HET, bool DISS>
void stage3(const StageLaunch& L, const BulkArgs<T>& a, const EdgeArgs<T>& e);

// an ensemble's stage, for the members with tile shape L.shape; without
// workgroups ahead the tiles alone
template <typename T>
void stage_batch(const StageLaunch& L, const BulkArgs<T>* bt, const EdgeArgs<T>* et, const int2* ahead, int nahead,
                 int swz);

}  // namespace fdm
