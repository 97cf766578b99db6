"""The direct contraction kernels at the edges of every tile shape: partial tiles, partial K steps, 16-byte and element
loads, every layout of the operands, contracted indices in one run, walked run by run and by table. test_direct_walk.py
checks that the shapes take the tiles they are listed under. Whole numbers: sums are exact."""
import pytest

from test_direct_walk import LAYOUTS, RUN_LAYOUTS, TILE_RUNS, TILES
from test_gpu_direct_walk import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dk,tile", [(dk, t) for dk in TILES for t in TILES[dk]])
def test_tiles(talsh_gpu, dk, tile):
    for size in TILES[dk][tile]:
        for pattern in LAYOUTS:
            check(talsh_gpu, dk, pattern, dict(zip("abk", size)))


@pytest.mark.parametrize("dk,tile", [(dk, t) for dk in TILE_RUNS for t in TILE_RUNS[dk]])
def test_tile_runs(talsh_gpu, dk, tile):
    for size in TILE_RUNS[dk][tile]:
        for pattern in RUN_LAYOUTS:
            check(talsh_gpu, dk, pattern, dict(zip("abij", size)))


@pytest.mark.parametrize("dk", TILES)
def test_conjugation(talsh_gpu, dk):
    for tile in TILES[dk]:
        a, b, k = TILES[dk][tile][0]
        check(talsh_gpu, dk, "D(a,b)+=L+(k,a)*R(b,k)", dict(a=a, b=b, k=k))
