"""The launch grid of the MSM pair kernels (csrc/tile_grid.hpp), compiled for the host."""
import ctypes
import os
import subprocess

import pytest

from musc_hip import build

THREADS, XCDS = 256, 8
SOURCE = '''#include "tile_grid.hpp"
extern "C" int grid_of(long long tiles, int threads, int multiple, unsigned* out) {
  musc::msm::TileGrid g = {0, 0};
  const bool ok = musc::msm::tile_grid(tiles, threads, multiple, &g);
  out[0] = g.x;
  out[1] = g.z;
  return ok;
}
'''


@pytest.fixture(scope='module')
def grid_of(tmp_path_factory):
    d = tmp_path_factory.mktemp('tile_grid')
    (d / 'g.cpp').write_text(SOURCE)
    subprocess.run(['g++', '-std=c++17', '-O1', '-shared', '-fPIC', '-I', build.CSRC, str(d / 'g.cpp'), '-o',
                    str(d / 'g.so')], check=True)
    fn = ctypes.CDLL(str(d / 'g.so')).grid_of
    fn.argtypes = [ctypes.c_longlong, ctypes.c_int, ctypes.c_int, ctypes.c_void_p]

    def call(tiles, threads=THREADS):
        out = (ctypes.c_uint * 2)()
        return (out[0], out[1]) if fn(tiles, threads, XCDS, out) else None
    return call


def _tiles(rows, tile):
    t = -(-rows // tile)
    return t * (t + 1) // 2


LIMIT = (2 ** 32 - 1) // THREADS // XCDS * XCDS   # workgroups of 256 threads in one dimension


@pytest.mark.parametrize('tiles', [1, 7, 8, 9, 528, 6000, LIMIT - 1, LIMIT, LIMIT + 1, 2 * LIMIT, 2 * LIMIT + 1,
                                   _tiles(3000 * 125, 64), _tiles(4096 * 127, 64), _tiles(4096 * 182, 128),
                                   _tiles(4096 * 363, 256), 2 ** 31 - 16, 2 ** 31 - 8])
def test_every_tile_has_a_workgroup_and_no_dimension_passes_the_launch_limit(grid_of, tiles):
    x, z = grid_of(tiles)
    assert x % XCDS == 0 and x * THREADS < 2 ** 32 and z <= 65535
    assert tiles <= x * z < tiles + z * XCDS
    assert z == 1 or tiles > LIMIT


def test_grids_past_two_to_the_31_are_refused(grid_of):
    assert grid_of(2 ** 31 - 8) is not None
    assert grid_of(2 ** 31 - 7) is None and grid_of(2 ** 45) is None


def test_the_kernels_take_their_grid_from_it():
    for name in ('msm_pair.hip', 'msm_split.hip'):
        src = open(os.path.join(build.CSRC, name)).read()
        assert 'tile_grid(ntiles, THREADS, kXcds, &grid)' in src and 'tile_number()' in src
        assert 'dim3(grid.x, pools.count, grid.z)' in src and f'THREADS = {THREADS};' in src
