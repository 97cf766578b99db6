#include "direct_launch.hpp"

namespace tal {

// tile shapes in the order of direct_tiles
bool direct_launch_c4(int tile, const DirectVariant &v, const DirectArgs &a, unsigned batch, hipStream_t s) {
  using namespace direct;
  switch (tile) {
    case 0:
    case 1: return run_tile<float, 2, Tile<64, 64, 16, 2, 2, 1, 2>, 2>(v, a, batch, s);
    case 2: return run_tile<float, 2, Tile<64, 32, 16, 4, 1, 2, 2>, 2>(v, a, batch, s);
    case 3: return run_tile<float, 2, Tile<32, 32, 16, 2, 2, 2, 2>, 2>(v, a, batch, s);
    default: return false;
  }
}

}  // namespace tal
