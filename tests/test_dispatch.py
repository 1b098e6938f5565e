"""The rules by which the default variants choose kernels and launch shapes (cudadma_amd/csrc/dispatch.hpp), evaluated on the host for the
256 compute units of an MI355X."""
import ctypes
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CUS = 256
BLOCKS, ROW_MAJOR = 0, -1

_SHIM = r"""
#include "dispatch.hpp"
extern "C" int tile_walk(int m, int n, int k, int rows, int cols, int per_cu, int cus) { return dispatch::tile_walk(m, n, k, rows, cols, per_cu, cus); }
extern "C" int gemm_form(int m, int n, int k, int cus) { return (int)dispatch::gemm_form(m, n, k, cus); }
extern "C" int copy_form(unsigned long long bytes) { return (int)dispatch::copy_form(bytes); }
extern "C" int rowsum_workgroups(unsigned long long table, unsigned long long n_idx) { return dispatch::rowsum_workgroups(table, n_idx); }
// every tile once?
extern "C" int visits_once(int tiles_m, int tiles_n, int walk, int* seen)
{
  for (int b = 0; b < tiles_m * tiles_n; ++b) {
    int i = -1, j = -1;
    dispatch::tile_of_workgroup(b, tiles_m, tiles_n, walk, i, j);
    if (i < 0 || i >= tiles_m || j < 0 || j >= tiles_n || seen[i * tiles_n + j]++) return 0;
  }
  return 1;
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("clang++") or shutil.which("hipcc")
    if cxx is None:
        pytest.skip("no C++ compiler")
    at = tmp_path_factory.mktemp("dispatch")
    (at / "shim.cpp").write_text(_SHIM)
    subprocess.run([cxx, "-std=c++17", "-O2", "-Wall", "-Wextra", "-Werror", "-shared", "-fPIC", "-I", os.path.join(ROOT, "cudadma_amd", "csrc"),
                    str(at / "shim.cpp"), "-o", str(at / "shim.so")], check=True)
    return ctypes.CDLL(str(at / "shim.so"))


def test_every_tile_has_one_workgroup(rules):
    """All walks that the rule can choose, over grids of one tile to several rounds."""
    for tiles_m in (1, 2, 3, 4, 5, 8, 11, 12, 16, 29, 60, 64):
        for tiles_n in (1, 2, 5, 8, 17, 24, 34, 66, 128):
            for walk in range(ROW_MAJOR, 9):
                if walk == BLOCKS and (tiles_m % 4 or tiles_n % 2):
                    continue
                assert rules.visits_once(tiles_m, tiles_n, walk, (ctypes.c_int * (tiles_m * tiles_n))()), (tiles_m, tiles_n, walk)


# m, n, k, tile, workgroups of a compute unit: grids that divide into 4 x 2, on both sides of every line
@pytest.mark.parametrize("shape, tile, per_cu, walk", [
    # columns of their own
    ((1024, 6144, 2048), 128, 2, ROW_MAJOR), ((512, 8192, 1024), 128, 1, ROW_MAJOR), ((1536, 8192, 2048), 128, 2, ROW_MAJOR),
    ((1024, 5120, 1024), 128, 2, BLOCKS), ((1024, 5120, 4096), 128, 2, BLOCKS), ((1536, 8192, 1024), 128, 2, BLOCKS), ((1024, 6144, 384), 128, 2, BLOCKS),
    # one band of four rows
    ((512, 16384, 512), 128, 2, 4), ((512, 8448, 2048), 128, 2, 4), ((1024, 9728, 1024), 256, 1, 4), ((512, 16384, 256), 128, 2, BLOCKS),
    # one band of eight, and of seven with one row left over
    ((1024, 6912, 512), 128, 2, BLOCKS), ((1024, 7936, 4096), 128, 2, BLOCKS), ((2048, 13312, 1024), 256, 1, BLOCKS), ((1024, 11776, 2048), 128, 2, 8),
    ((1024, 11776, 512), 128, 2, BLOCKS), ((1024, 5632, 2048), 128, 2, BLOCKS),
    # several bands: dividing the rows evenly, and with a half left over
    ((2048, 8960, 2048), 128, 2, 8), ((2048, 8960, 1024), 128, 2, BLOCKS), ((1536, 7424, 2048), 128, 2, BLOCKS), ((1536, 11008, 1536), 128, 2, 8),
    ((1536, 9984, 512), 128, 2, BLOCKS), ((8192, 8192, 1024), 256, 1, BLOCKS),
    # tiles below 128 x 128
    ((128, 2048, 768), 32, 2, ROW_MAJOR), ((256, 2176, 512), 64, 2, 4), ((3840, 256, 2048), 64, 2, 6), ((5376, 256, 2048), 64, 2, 7),
    ((512, 2304, 2048), 64, 2, BLOCKS), ((1024, 1024, 1024), 64, 1, BLOCKS),
    # columns of their own in grids with fewer rows than a band may have
    ((256, 7680, 512), 64, 2, ROW_MAJOR), ((256, 5120, 2432), 64, 2, ROW_MAJOR), ((128, 9728, 512), 64, 2, ROW_MAJOR), ((256, 7552, 768), 64, 2, 4),
    ((640, 11264, 7040), 128, 2, 5)])
def test_walk_of_grids_in_blocks_or_narrow(rules, shape, tile, per_cu, walk):
    got = rules.tile_walk(*shape, tile, tile, per_cu, CUS)
    # a band is no higher than the grid
    assert (got if got <= 0 else min(got, shape[0] // tile)) == walk


LONG_ROWS, DEALT_32, DEALT_32_64, DEALT_64, DEALT_64_TWO, TILE_128_FAR, TILE_128, TILE_256 = range(8)


@pytest.mark.parametrize("shape, form", [
    ((512, 512, 512), DEALT_32), ((640, 512, 8192), DEALT_32_64), ((1024, 1024, 128), DEALT_64), ((128, 8192, 128), DEALT_64),
    ((1152, 1024, 384), TILE_128), ((1152, 1024, 512), DEALT_64_TWO), ((256, 8192, 3008), DEALT_64_TWO), ((256, 8192, 3072), TILE_128_FAR),
    # two rows of 64 x 64 tiles
    ((128, 10368, 896), DEALT_64_TWO), ((128, 10368, 1024), TILE_128_FAR), ((128, 10240, 2048), DEALT_64_TWO), ((128, 16384, 2048), TILE_128_FAR),
    ((128, 8320, 384), TILE_128), ((2176, 1024, 640), TILE_128), ((2176, 1024, 768), TILE_128_FAR), ((2048, 2048, 1920), TILE_128_FAR),
    ((2048, 2176, 1920), TILE_128), ((4096, 4096, 4096), TILE_256), ((1408, 2176, 1920), TILE_128_FAR), ((128, 128, 71_600_128), LONG_ROWS)])
def test_kernel_of_the_default_gemm(rules, shape, form):
    assert rules.gemm_form(*shape, CUS) == form


def test_kernel_of_the_default_copy(rules):
    tile, mib = 16 << 10, 1 << 20
    one_tile_four, two_tiles_streaming, two_tiles, one_tile_two = range(4)
    rules.copy_form.argtypes = [ctypes.c_ulonglong]
    for size, form in ((tile, one_tile_four), (16 * mib, one_tile_four), (16 * mib + tile, two_tiles_streaming), (44 * mib, two_tiles_streaming),
                       (44 * mib + tile, two_tiles), (48 * mib, two_tiles), (96 * mib, two_tiles), (96 * mib + tile, one_tile_two), (8 << 30, one_tile_two)):
        assert rules.copy_form(size) == form, size


def test_workgroups_of_the_default_row_sums(rules):
    mib, mi = 1 << 20, 1 << 20
    rules.rowsum_workgroups.argtypes = [ctypes.c_ulonglong] * 2
    for table, indices, workgroups in ((256 * mib, 32 * mi, 4), (4096 * mib, mi, 4), (257 * mib, mi + 32, 2), (512 * mib, 32 * mi, 2), (640 * mib, 32 * mi, 2),
                                       (768 * mib, 6 * mi, 2), (768 * mib, 8 * mi, 3), (1024 * mib, 16 * mi, 3), (1024 * mib, 4 * mi, 2),
                                       (1025 * mib, 2 * mi, 3), (8192 * mib, 32 * mi, 3)):
        assert rules.rowsum_workgroups(table, indices) == workgroups, (table, indices)
