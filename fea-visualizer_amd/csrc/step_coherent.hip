// step_coherent.hip -- the stepping kernel instantiated for the coherent exchange mode.
#define FEMHIP_TEAM_BLOCK 512  // kTeamBlock
#include "step_kernel.h"

namespace femhip {
const void* step_kernel_coherent(int k, int fp32, int kr) { return pick_for_mode<kCoherent, false>(k, fp32, kr); }
}  // namespace femhip
