// slc_ens_tile_d4.hip -- batched SL tile kernels, double field storage, order 4.
#include "slc_ens_tile.h"

namespace slc {

void run_ens_tile_d4(const EnsMember* mem, const EnsTiles& t, int pass, int shape,
                     hipStream_t s) {
    launch_tile_pass<double, 4>(mem, t, pass, shape, s);
}

}  // namespace slc
