// The e2m1 instantiations of the kernel in mx_ring_kernels.hpp.
#include "mx_ring_kernels.hpp"

namespace dt {

int launch_ring_e2m1(const RingArgs& p, bool ragged, int tile_m, int tile_n, int splits) {
  if (tile_m == 64) return tile_n == 64 ? ring::launch_tile<2, 2, true>(p, ragged, splits) : ring::launch_tile<2, 4, true>(p, ragged, splits);
  return tile_n == 64 ? ring::launch_tile<4, 2, true>(p, ragged, splits) : ring::launch_tile<4, 4, true>(p, ragged, splits);
}

}  // namespace dt
