// ctraj_record.hpp -- z-grid samples by kernels for the rows and for the samples (record.hip).
#pragma once

#include "ctraj_internal.hpp"

namespace ctraj {

// molecules of a slice, molecule-major and field-major, and the lens rows kept for them: 512 MiB, and at most so many
// for each (padded, field-major, to the longest of 64)
constexpr int64_t ZGRID_SLICE_MOL = 40960, ZGRID_SLICE_FIELD = 32768;
constexpr int64_t ZGRID_ROWS = ((int64_t)512 << 20) / 32, ZGRID_ROWS_EACH = 1024;

// What record_zgrid leaves: its workspace (given back once the caller has launched the rest) and the list of
// slots it left to the one-kernel form, [0] their count, or ZGRID_ALL: all of them, in their own order (through the
// list, whose order is the wavefronts', the field-major form took 7 % longer).  ws null: no memory, nothing launched.
constexpr uint32_t ZGRID_ALL = 0xffffffffu;

struct ZGridPlan {
  void *ws = nullptr;
  const uint32_t *odd = nullptr;
};

// The lens rows of a molecule, on the average, for which those kernels are the faster form.
struct ZGridSteps {
  double lo = 0.0, hi = 1e300;
};

// Launch those kernels for a beamline with exactly one lens, in RK4 steps under a spline force.
int record_zgrid(ctraj_ctx *c, const ctraj_record &RC, int lens_e, bool circ_only, const KBeam &B, const KTab &kt,
                 size_t lds, const ZGridSteps &steps, ZGridPlan &plan);

}  // namespace ctraj
