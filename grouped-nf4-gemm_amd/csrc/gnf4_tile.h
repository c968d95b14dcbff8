// gnf4_tile.h -- launches of the tile kernels (gnf4_tile.hip).
#pragma once

#include "gnf4_device.h"

namespace gnf4 {

// 256-row forward tiles on a grid of eight XCD ranges of per_x workgroups.
// The tile table is tt's (n > 0) or p's device arrays.
int launch_tile_fwd(int fmt, const FwdArgs& p, const PwTiles& tt, int64_t per_x,
                    hipStream_t stream);

// Dgrad tiles of at most kDgradWideRows rows x 512 columns (p.a the gradient rows,
// N % 64 == 0 and K % 64 == 0), the same grid.
constexpr int kDgradWideRows = 160;
int launch_tile_dgrad(int fmt, const FwdArgs& p, uint16_t* out, const PwTiles& tt, int64_t per_x,
                      hipStream_t stream);

}  // namespace gnf4
