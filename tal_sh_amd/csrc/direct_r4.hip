#include "direct_launch.hpp"

namespace tal {

// tile shapes in the order of direct_tiles
bool direct_launch_r4(int tile, const DirectVariant &v, const DirectArgs &a, unsigned batch, hipStream_t s) {
  using namespace direct;
  switch (tile) {
    case 0: return run_tile<float, 1, Tile<128, 128, 16, 2, 4, 2, 4>, 4>(v, a, batch, s);
    case 1: return run_tile<float, 1, Tile<64, 64, 32, 2, 4, 3, 2>, 4>(v, a, batch, s);
    case 2: return run_tile<float, 1, Tile<64, 32, 32, 4, 1, 2, 2>, 4>(v, a, batch, s);
    case 3: return run_tile<float, 1, Tile<32, 32, 32, 2, 2, 2, 2>, 4>(v, a, batch, s);
    default: return false;
  }
}

}  // namespace tal
