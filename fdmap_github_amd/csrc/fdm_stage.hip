// fdm_stage.hip -- the stage kernels' variants, compiled in FDM_PARTS parts
// (-DFDM_PART=1..) so that they build in parallel.
#include "fdm_stage.hpp"

#include <type_traits>

namespace fdm {

namespace {

template <typename T, int TX, int TY, int OP, bool HET, bool DISS, bool JI, bool MC>
void stage2_v(const StageLaunch& L, const BulkArgs<T>& a, const EdgeArgs<T>& e) {
  if constexpr (std::is_same<T, float>::value && (HET || DISS)) {
    if (!L.full && L.many) {
      if (L.nt_store)
        hipLaunchKernelGGL((bulk_interior<T, TX, TY, 0, true, HET, DISS, OP, JI, MC, true>), L.grid, L.block, 0,
                           L.stream, a, e, L.tiles);
      else
        hipLaunchKernelGGL((bulk_interior<T, TX, TY, 0, false, HET, DISS, OP, JI, MC, true>), L.grid, L.block, 0,
                           L.stream, a, e, L.tiles);
      return;
    }
  }
  if (L.full == 1)
    hipLaunchKernelGGL((bulk_interior<T, TX, TY, 1, false, HET, DISS, OP, JI, MC>), L.grid, L.block, 0, L.stream, a, e,
                       L.tiles);
  else if (L.full && L.nt_store)
    hipLaunchKernelGGL((bulk_interior<T, TX, TY, 2, true, HET, DISS, OP, JI, MC>), L.grid, L.block, 0, L.stream, a, e,
                       L.tiles);
  else if (L.full)
    hipLaunchKernelGGL((bulk_interior<T, TX, TY, 2, false, HET, DISS, OP, JI, MC>), L.grid, L.block, 0, L.stream, a, e,
                       L.tiles);
  else if (L.nt_store)
    hipLaunchKernelGGL((bulk_interior<T, TX, TY, 0, true, HET, DISS, OP, JI, MC>), L.grid, L.block, 0, L.stream, a, e,
                       L.tiles);
  else
    hipLaunchKernelGGL((bulk_interior<T, TX, TY, 0, false, HET, DISS, OP, JI, MC>), L.grid, L.block, 0, L.stream, a, e,
                       L.tiles);
}

}  // namespace

template <typename T, int OP, bool HET, bool DISS, int SHAPE>
void stage2(const StageLaunch& L, const BulkArgs<T>& a, const EdgeArgs<T>& e) {
  constexpr int TX = kTileShape[SHAPE][0], TY = kTileShape[SHAPE][1];
  if constexpr (std::is_same<T, double>::value) {
    // the FP32-delta variants exist for the 64-column tiles
    if constexpr (TX == 64) {
      if (L.mcomp) {
        if (L.ji_calc) stage2_v<T, TX, TY, OP, HET, DISS, true, true>(L, a, e);
        else stage2_v<T, TX, TY, OP, HET, DISS, false, true>(L, a, e);
        return;
      }
    }
    if (L.ji_calc) {
      stage2_v<T, TX, TY, OP, HET, DISS, true, false>(L, a, e);
      return;
    }
  }
  stage2_v<T, TX, TY, OP, HET, DISS, false, false>(L, a, e);
}

namespace {

template <typename T, int OP, bool HET, bool DISS, bool JI, bool MC>
void stage3_v(const StageLaunch& L, const BulkArgs<T>& a, const EdgeArgs<T>& e) {
  if (L.nt_store)
    hipLaunchKernelGGL((bulk_interior3<T, 64, 4, true, OP, HET, DISS, JI, MC>), L.grid, L.block, 0, L.stream, a, e,
                       L.tiles);
  else
    hipLaunchKernelGGL((bulk_interior3<T, 64, 4, false, OP, HET, DISS, JI, MC>), L.grid, L.block, 0, L.stream, a, e,
                       L.tiles);
}

}  // namespace

template <typename T, int OP, bool HET, bool DISS>
void stage3(const StageLaunch& L, const BulkArgs<T>& a, const EdgeArgs<T>& e) {
  if constexpr (std::is_same<T, double>::value) {
    if (L.mcomp && L.ji_calc) {
      stage3_v<T, OP, HET, DISS, true, true>(L, a, e);
      return;
    }
    if (L.ji_calc) {
      stage3_v<T, OP, HET, DISS, true, false>(L, a, e);
      return;
    }
  }
  stage3_v<T, OP, HET, DISS, false, false>(L, a, e);
}

namespace {

template <typename T, int TX, int TY, bool AHEAD>
void batch_v(const StageLaunch& L, const BulkArgs<T>* bt, const EdgeArgs<T>* et, const int2* ahead, int nahead,
             int swz) {
  if (L.full == 1)
    hipLaunchKernelGGL((bulk_interior_batch<T, TX, TY, 1, false, AHEAD>), L.grid, L.block, 0, L.stream, bt, et, ahead,
                       nahead, L.tiles, swz);
  else if (L.full && L.nt_store)
    hipLaunchKernelGGL((bulk_interior_batch<T, TX, TY, 2, true, AHEAD>), L.grid, L.block, 0, L.stream, bt, et, ahead,
                       nahead, L.tiles, swz);
  else if (L.full)
    hipLaunchKernelGGL((bulk_interior_batch<T, TX, TY, 2, false, AHEAD>), L.grid, L.block, 0, L.stream, bt, et, ahead,
                       nahead, L.tiles, swz);
  else if (L.nt_store)
    hipLaunchKernelGGL((bulk_interior_batch<T, TX, TY, 0, true, AHEAD>), L.grid, L.block, 0, L.stream, bt, et, ahead,
                       nahead, L.tiles, swz);
  else
    hipLaunchKernelGGL((bulk_interior_batch<T, TX, TY, 0, false, AHEAD>), L.grid, L.block, 0, L.stream, bt, et, ahead,
                       nahead, L.tiles, swz);
}

template <typename T, bool AHEAD>
void batch_s(const StageLaunch& L, const BulkArgs<T>* bt, const EdgeArgs<T>* et, const int2* ahead, int nahead,
             int swz) {
  if (L.shape == 0) batch_v<T, 64, 4, AHEAD>(L, bt, et, ahead, nahead, swz);
  else if (L.shape == 1) batch_v<T, 64, 8, AHEAD>(L, bt, et, ahead, nahead, swz);
  else batch_v<T, 128, 4, AHEAD>(L, bt, et, ahead, nahead, swz);
}

}  // namespace

template <typename T>
void stage_batch(const StageLaunch& L, const BulkArgs<T>* bt, const EdgeArgs<T>* et, const int2* ahead, int nahead,
                 int swz) {
  if (nahead) batch_s<T, true>(L, bt, et, ahead, nahead, swz);
  else batch_s<T, false>(L, bt, et, ahead, nahead, swz);
}

#define STAGE2(T, OP, HET, DISS, SHAPE) \
  template void stage2<T, OP, HET, DISS, SHAPE>(const StageLaunch&, const BulkArgs<T>&, const EdgeArgs<T>&);
#define STAGE3(T, OP, HET, DISS) \
  template void stage3<T, OP, HET, DISS>(const StageLaunch&, const BulkArgs<T>&, const EdgeArgs<T>&);
#define BATCH(T)                                                                                              \
  template void stage_batch<T>(const StageLaunch&, const BulkArgs<T>*, const EdgeArgs<T>*, const int2*, int, int);

#if FDM_PART == 1
STAGE2(double, 4, false, false, 0)
#elif FDM_PART == 2
STAGE2(double, 4, false, false, 1)
STAGE2(double, 4, false, false, 2)
#elif FDM_PART == 3
STAGE2(double, 4, true, false, 0)
#elif FDM_PART == 4
STAGE2(double, 4, false, true, 0)
#elif FDM_PART == 5
STAGE2(double, 4, true, true, 0)
#elif FDM_PART == 6
STAGE2(double, 2, false, false, 0)
STAGE2(double, 2, true, false, 0)
#elif FDM_PART == 7
STAGE2(double, 6, false, false, 0)
#elif FDM_PART == 8
STAGE2(double, 6, false, false, 1)
#elif FDM_PART == 9
STAGE2(double, 6, true, false, 0)
#elif FDM_PART == 10
STAGE2(float, 4, false, false, 0)
STAGE2(float, 4, false, false, 1)
STAGE2(float, 4, false, false, 2)
STAGE2(float, 4, true, false, 0)
#elif FDM_PART == 11
STAGE2(float, 4, false, true, 0)
STAGE2(float, 4, true, true, 0)
STAGE2(float, 2, false, false, 0)
STAGE2(float, 2, true, false, 0)
#elif FDM_PART == 12
STAGE2(float, 6, false, false, 0)
STAGE2(float, 6, false, false, 1)
STAGE2(float, 6, true, false, 0)
#elif FDM_PART == 13
STAGE3(double, 4, false, false)
STAGE3(double, 4, true, false)
STAGE3(double, 4, false, true)
STAGE3(double, 4, true, true)
STAGE3(double, 2, false, false)
STAGE3(double, 2, true, false)
STAGE3(double, 6, false, false)
STAGE3(double, 6, true, false)
#elif FDM_PART == 14
STAGE3(float, 4, false, false)
STAGE3(float, 4, true, false)
STAGE3(float, 4, false, true)
STAGE3(float, 4, true, true)
STAGE3(float, 2, false, false)
STAGE3(float, 2, true, false)
STAGE3(float, 6, false, false)
STAGE3(float, 6, true, false)
#elif FDM_PART == 15
BATCH(double)
#elif FDM_PART == 16
BATCH(float)
#else
#error "FDM_PART must be 1 to 16"
#endif

}  // namespace fdm
