// slc_ens_tile_f4.hip -- batched SL tile kernels, float field storage, order 4.
#include "slc_ens_tile.h"

namespace slc {

void run_ens_tile_f4(const EnsMember* mem, const EnsTiles& t, int pass, int shape,
                     hipStream_t s) {
    launch_tile_pass<float, 4>(mem, t, pass, shape, s);
}

}  // namespace slc
