// fdm_stage.hpp -- host launchers of the stage kernels (bulk_interior,
// bulk_interior3, bulk_interior_batch).  Their many variants are compiled in
// parts (fdm_stage.hip, one object per part); this header declares one
// launcher per (precision, operator, medium, dissipation, tile shape).
#pragma once

#include "fdm_bulk.hpp"

namespace fdm {

// interior tile shapes (columns x rows) selectable with FDM_TILE
constexpr int kTileShape[3][2] = {{64, 4}, {64, 8}, {128, 4}};

struct StageLaunch {
  hipStream_t stream;
  dim3 grid, block;
  const int4* tiles;
  int shape;
  int full;  // FULL of the kernels
  bool nt_store, ji_calc, mcomp;
};

// plane strain: FULL = 1 (manufactured solutions, plasticity), 2 (plasticity)
// or lean, these with non-temporal or normal stores; in FP64 with or without Ji formed in the kernel (ji_calc)
// and FP32-delta metrics (mcomp)
template <typename T, int OP, bool HET, bool DISS, int SHAPE>
void stage2(const StageLaunch& L, const BulkArgs<T>& a, const EdgeArgs<T>& e);

// antiplane shear
template <typename T, int OP, bool HET, bool DISS>
void stage3(const StageLaunch& L, const BulkArgs<T>& a, const EdgeArgs<T>& e);

// an ensemble's stage, for the members with tile shape L.shape
template <typename T>
void stage_batch(const StageLaunch& L, const BulkArgs<T>* bt, const EdgeArgs<T>* et, const int2* ahead, int nahead,
                 int swz);

}  // namespace fdm
