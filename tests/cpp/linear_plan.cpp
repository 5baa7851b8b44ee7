// The batched linear kernel's host-side rules, for tests/test_linear_plan.py (no GPU).
#include "../../inference-agent_amd/csrc/linear_tile.h"

extern "C" uint32_t plan_block0(uint32_t tt, uint32_t nb, uint32_t tiles_m) {
    return ingot::tile_block0(tt, nb, tiles_m);
}
