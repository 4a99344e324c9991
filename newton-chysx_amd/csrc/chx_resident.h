// Host entry of the resident PCG kernel (chx_resident.hip).
#pragma once

#include "chx_internal.h"
#include "chysx_hip.h"

namespace chx {

// Workgroups of the resident kernel that run at once on the current device.
int resident_grid_limit();
// Workgroups and groups of a single instance's launch: one workgroup per
// part; above 32 a whole number per group, so that a group's parts, which
// are neighbours, share an XCD.
inline int single_grid(int parts, int limit, int* groups) {
    const int even = (parts + 7) / 8 * 8;
    *groups = parts > 32 && even <= limit ? 8 : 1;
    return *groups == 8 ? even : parts;
}
// One solve of a batch whose instances all carry a plan (res_grid > 0).
void launch_resident(const chx_cloth_batch& B, int finalize, hipStream_t stream);

}  // namespace chx
