#include "direct_launch.hpp"

namespace tal {

// tile shapes in the order of direct_tiles
bool direct_launch_c8(int tile, const DirectVariant &v, const DirectArgs &a, unsigned batch, hipStream_t s) {
  using namespace direct;
  switch (tile) {
    case 0:
    case 1: return run_tile<double, 2, Tile<64, 64, 16, 2, 4, 1, 4>, 1>(v, a, batch, s);
    case 2: return run_tile<double, 2, Tile<64, 32, 8, 4, 1, 2, 2>, 1>(v, a, batch, s);
    case 3: return run_tile<double, 2, Tile<32, 32, 8, 2, 2, 2, 2>, 1>(v, a, batch, s);
    default: return false;
  }
}

}  // namespace tal
