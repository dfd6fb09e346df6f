// q4_rows_kernel on blocks of 16 tiles.
#include "q4_rows_device.h"

namespace mi355q {

hipError_t q4_rows_launch_16(mi355q_context *ctx, int mf, bool pair, uint32_t groups, const GemmGroup &group)
{
    return launch_rows_of<8, 2>(ctx, mf, pair, groups, group);
}

}  // namespace mi355q
