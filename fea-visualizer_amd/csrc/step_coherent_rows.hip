// step_coherent_rows.hip -- the stepping kernel instantiated for the coherent exchange mode, with rows kept in LDS.
#define FEMHIP_TEAM_BLOCK 512  // kTeamBlock
#include "step_kernel.h"

namespace femhip {
const void* step_kernel_coherent_rows(int k, int fp32, int kr) { return pick_for_mode<kCoherent, true>(k, fp32, kr); }
}  // namespace femhip
