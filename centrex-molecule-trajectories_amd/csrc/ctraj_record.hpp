// ctraj_record.hpp -- z-grid samples in two kernels (record.hip).
#pragma once

#include "ctraj_internal.hpp"

namespace ctraj {

constexpr int64_t ZGRID_SLICE_MOL = 40960;  // molecules of a slice, molecule-major

// What record_zgrid leaves: its workspace (given back once the caller has launched the rest) and the list of
// slots it left to the one-kernel form, [0] their count.  ws null: no memory, nothing launched.
struct ZGridPlan {
  void *ws = nullptr;
  const uint32_t *odd = nullptr;
};

// Launch the two kernels for a beamline with exactly one lens, in RK4 steps under a spline force.
int record_zgrid(ctraj_ctx *c, const ctraj_record &RC, int lens_e, bool circ_only, const KBeam &B, const KTab &kt,
                 size_t lds, ZGridPlan &plan);

}  // namespace ctraj
