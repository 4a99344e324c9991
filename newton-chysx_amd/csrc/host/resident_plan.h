// Plan of the resident PCG (csrc/chx_resident.hip): how one cloth's block
// rows are dealt to workgroups that keep their part of the matrix in
// registers for the whole solve.  Integer work on the host, from the BSR
// pattern alone.
#pragma once

#include <cstdint>
#include <vector>

#include "topology.h"

namespace chysx {
namespace engine {

// Canonical order of the rows: compact patches of the mesh, so that the
// rows of a part (CHX_RES_LEAF-row leaves, consecutive in this order) have
// few neighbours outside it.  order[k] = row at position k.
std::vector<int> resident_order(const topology::Pattern& p);

// The parts of `part_rows` consecutive positions each.  blob is the device
// image (layout: include/chysx_hip.h, chx_instance::res_plan); empty when
// the pattern does not fit the kernel's limits (a row with more than
// CHX_RES_HELD upper or lower blocks, a part with more than
// CHX_RES_HALO_MAX halo rows or CHX_RES_GHOST_MAX ghost blocks).
// block_slots: value slot of CSR block k (-1 - partner's slot: lower).
struct ResidentPlan {
    int part_rows = 0;
    int parts = 0;
    int exports = 0;  // rows that some other part reads
    std::vector<std::uint32_t> blob;
};
ResidentPlan resident_plan(const topology::Pattern& p, const std::vector<int>& block_slots,
                           const std::vector<int>& order, int part_rows);

}  // namespace engine
}  // namespace chysx
