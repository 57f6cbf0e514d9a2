// step_fenced_rows.hip -- the stepping kernel instantiated for the fenced exchange mode, with rows kept in LDS.
#define FEMHIP_TEAM_BLOCK 512  // kTeamBlock
#include "step_kernel.h"

namespace femhip {
const void* step_kernel_fenced_rows(int k, int fp32, int kr) { return pick_for_mode<kFenced, true>(k, fp32, kr); }
}  // namespace femhip
