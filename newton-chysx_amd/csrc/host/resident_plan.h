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
// image (layout: include/chysx_hip.h, CHX_RES_*); empty when the pattern does
// not fit the form's limits (blocks of a row, halo rows and ghost blocks of
// a part).  block_slots: value slot of CSR block k (-1 - partner's: lower).
struct ResidentPlan {
    int part_rows = 0;
    int parts = 0;
    int exports = 0;  // rows that some other part reads
    std::vector<std::uint32_t> blob;
};
// Sheet form: the upper blocks of a row are held by the row.  `capacity`:
// rows of the largest part (CHX_RES_PART_MAX; half sheets CHX_RES_GEN_PART).
ResidentPlan resident_plan(const topology::Pattern& p, const std::vector<int>& block_slots,
                           const std::vector<int>& order, int part_rows, int capacity);
// General form: any numbering, wider rows, smaller parts.
ResidentPlan resident_plan_general(const topology::Pattern& p, const std::vector<int>& block_slots,
                                   const std::vector<int>& order, int part_rows);
// Rows form of a caller's matrix (any pattern, symmetric or not).
ResidentPlan resident_plan_rows(const topology::Pattern& p, const std::vector<int>& order, int part_rows);
// Rows per part of the resident solve of matrices with `rows` block rows
// each and at most `largest` a part: the smallest size (from 256) whose parts
// all run at once on 256 workgroups, else the largest; 0 when one matrix
// alone has more parts than that.  What fits one part is one part: it needs
// no exchange.
int resident_part_rows(const std::vector<int>& rows, int largest);
// Forms and part sizes for cloths that are solved together, the best first;
// the first that every cloth's pattern fits is taken.
struct ResidentChoice {
    int form, part_rows;
};
std::vector<ResidentChoice> resident_choices(const std::vector<int>& rows, bool bf16);
}  // namespace engine
}  // namespace chysx
