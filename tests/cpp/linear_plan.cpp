// The batched linear kernel's host-side rules, for tests/test_linear_plan.py (no GPU).
#include "../../inference-agent_amd/csrc/linear_tile.h"

extern "C" uint32_t plan_share0(uint32_t i, uint32_t n, uint32_t parts) {
    return ingot::tile_share0(i, n, parts);
}

#include "../../inference-agent_amd/csrc/linear_shape.h"

// The shape chosen for a call: ntb, k groups, splits.
extern "C" void plan_shape(uint32_t type, uint32_t n_in, uint32_t n_out, uint32_t n_tok, uint32_t requested,
                           uint64_t workspace_bytes, uint32_t* out) {
    const ingot::TileShape s = ingot::linear_shape(type, n_in, n_out, n_tok, requested, workspace_bytes);
    out[0] = s.ntb;
    out[1] = s.kg;
    out[2] = s.splits;
}
