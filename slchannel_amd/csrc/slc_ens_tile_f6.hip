// slc_ens_tile_f6.hip -- batched SL tile kernels, float field storage, order 6.
#include "slc_ens_tile.h"

namespace slc {

void run_ens_tile_f6(const EnsMember* mem, const EnsTiles& t, int pass, int shape,
                     hipStream_t s) {
    launch_tile_pass<float, 6>(mem, t, pass, shape, s);
}

}  // namespace slc
