// step_plain_rows.hip -- the stepping kernel instantiated for one-workgroup teams, with rows kept in LDS.
#include "step_kernel.h"

namespace femhip {
const void* step_kernel_plain_rows(int k, int fp32, int kr) { return pick_for_mode<kPlain, true>(k, fp32, kr); }
}  // namespace femhip
