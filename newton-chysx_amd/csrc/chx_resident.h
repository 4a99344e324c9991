// Host entry of the resident PCG kernel (chx_resident.hip).
#pragma once

#include "chx_internal.h"
#include "chysx_hip.h"

namespace chx {

// Workgroups of the resident kernel that run at once on the current device.
int resident_grid_limit();
// One solve of a batch whose instances all carry a plan (res_grid > 0).
void launch_resident(const chx_cloth_batch& B, int finalize, hipStream_t stream);

}  // namespace chx
