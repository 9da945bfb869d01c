// Parts of the drop-in calls that other drop-in calls issue on the library
// stream without waiting (api_fft.hip).
#pragma once

#include "../../include/mitos_hip.h"
#include "api_util.h"

namespace mitos {

// box -> fbox as fft_r2c_dg, then the Poisson kernel on fbox when asked
int dg_r2c_issue(struct distributed_grid* dg, bool poisson);
// fbox -> box as fft_c2r_dg
int dg_c2r_issue(struct distributed_grid* dg);
// w = dg->fbox * kernel, w with rows of whs
int apply_padded_issue(cx<double>* w, long whs, const struct distributed_grid* dg,
                       const KSpec& ks);

}  // namespace mitos
