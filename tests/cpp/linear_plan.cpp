// The batched linear kernel's host-side rules, for tests/test_linear_plan.py and
// tests/test_gpu_linear_shapes.py (built with g++, no GPU).
#include "../../inference-agent_amd/csrc/linear_shape.h"

extern "C" uint32_t plan_share0(uint32_t i, uint32_t n, uint32_t parts) { return ingot::tile_share0(i, n, parts); }

static void put(const ingot::TileShape& s, uint32_t* out) {
    out[0] = s.ntb;
    out[1] = s.kg;
    out[2] = s.splits;
}

// The shape chosen for ingot_linear: token blocks, k groups, splits.
extern "C" void plan_shape(uint32_t type, uint32_t n_in, uint32_t n_out, uint32_t n_tok, uint32_t requested,
                           uint64_t workspace_bytes, uint32_t* out) {
    put(ingot::linear_shape(type, n_in, n_out, n_tok, requested, workspace_bytes), out);
}

// The shape of a gate/up pair of n_out rows each.
extern "C" void plan_pair(uint32_t type, uint32_t n_in, uint32_t n_out, uint32_t n_tok, uint32_t* out) {
    put(ingot::unsplit_shape(type, n_in, 2 * n_out, n_tok, ingot::unsplit_k_groups(type, n_in, n_out, n_tok)), out);
}

// Do the token tiles of an ingot_linear call of that shape start apart?
extern "C" bool plan_spread(uint32_t kg, uint64_t weight_bytes, uint64_t x_bytes) {
    return ingot::tile_spread(ingot::TileShape{1, kg, 1}, weight_bytes, x_bytes);
}
