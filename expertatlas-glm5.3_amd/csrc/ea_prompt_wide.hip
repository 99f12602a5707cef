// The prompt pass's item lists for layers that hold experts above width 10 (three trellis words a lane a tile, larger
// staging regions): the kernels of ea_prompt_items.hpp built for widths 2..16. 777 rows, experts at 5, 6 and 8 bits: 428 us,
// against 2,380 with a kernel that read each tile's words straight into registers (one load a lane a word, bound by the
// address units) for items of up to 112 pairs, one list after the other.
#include <hip/hip_runtime.h>

#include "ea_prompt_items.hpp"

namespace ea {

int list_pass_wide(hipStream_t q, const ListPass& a, int big, uint32_t cb) {
    return cb == 1 ? list_pass<1, 16>(q, a, big) : cb == 2 ? list_pass<2, 16>(q, a, big) : list_pass<0, 16>(q, a, big);
}

}  // namespace ea
