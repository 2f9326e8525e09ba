"""Which kernel int8 rows on a re-tiled filter go to (lrtfc_fc_int8_packed_kernel, a host function):
each line of the rule at sizes on both its sides, as measured."""
import ctypes as C

import pytest

from litert_amd import capi


def _kernel(rows, depth, channels):
    return capi.load().lrtfc_fc_int8_packed_kernel(rows, depth, channels)


@pytest.mark.parametrize("rows,depth,channels", [
    (129, 4096, 14336), (200, 4096, 10240), (256, 4096, 12288), (400, 6144, 5120), (512, 8192, 6144),
    (640, 16384, 6144), (900, 4096, 3072)])
def test_small_tiles_in_many_rounds_stay_with_the_gemm(rows, depth, channels):
    assert _kernel(rows, depth, channels) == capi.INT8_KERNEL_TILES_64X128


@pytest.mark.parametrize("rows,depth,channels", [
    (77, 3008, 5003), (250, 2048, 2048), (400, 8192, 2048), (100, 16384, 512), (200, 4096, 4096),
    (160, 6144, 6144), (300, 16384, 4096)])
def test_small_tiles_in_one_or_two_rounds(rows, depth, channels):
    assert _kernel(rows, depth, channels) == capi.INT8_KERNEL_SPLIT


@pytest.mark.parametrize("rows,depth,channels,kernel", [
    (1, 2048, 2048, capi.INT8_KERNEL_GEMV), (16, 4096, 14336, capi.INT8_KERNEL_GEMV),
    (20, 8, 40, capi.INT8_KERNEL_GEMV),  # too shallow for a GEMM
    (32, 4096, 14336, capi.INT8_KERNEL_GEMV_TWO_TILES), (128, 4096, 14336, capi.INT8_KERNEL_ROWS),
    (400, 2048, 4096, capi.INT8_KERNEL_TILES_64X128), (2048, 4096, 4096, capi.INT8_KERNEL_TILES_128X256)])
def test_the_other_kernels(rows, depth, channels, kernel):
    assert _kernel(rows, depth, channels) == kernel


@pytest.mark.parametrize("rows,depth,channels", [
    (64, 1024, 16384), (33, 1037, 10243), (50, 1152, 14080), (40, 1370, 10240), (17, 128, 8200),
    (32, 100, 14336)])
def test_what_leaves_the_one_pass_kernels_runs_on_what_beat_them(rows, depth, channels):
    assert _kernel(rows, depth, channels) == capi.INT8_KERNEL_SPLIT


def test_no_row_count_falls_between_the_rules():
    """Wherever a kernel takes all rows in one pass, the launch is that kernel's or the small tiles'."""
    for rows in range(17, 129):
        for depth in (16, 128, 1000, 1024, 1200, 1376, 1500, 2048, 3000, 4096):
            for channels in (300, 2048, 8192, 10225, 12000, 14336, 16384, 20000):
                one_pass = (capi.INT8_KERNEL_GEMV_TWO_TILES if rows <= 32 else
                            capi.INT8_KERNEL_ROWS if depth >= 1024 and channels > 639 * 16 else None)
                if one_pass is not None:
                    assert _kernel(rows, depth, channels) in (one_pass, capi.INT8_KERNEL_SPLIT), \
                        (rows, depth, channels)


@pytest.mark.parametrize("rows,depth,channels,kernel", [
    (8, 8192, 256, capi.INT8_KERNEL_GEMV), (5, 6145, 4096, capi.INT8_KERNEL_GEMV),
    (8, 6144, 4096, capi.INT8_KERNEL_SPLIT),
    (9, 8192, 256, capi.INT8_KERNEL_SPLIT), (8, 8193, 256, capi.INT8_KERNEL_SPLIT),  # past 64 KB, 8192
    (16, 1024, 2048, capi.INT8_KERNEL_GEMV), (16, 1025, 2048, capi.INT8_KERNEL_SPLIT),  # 16 KB of rows
    (8, 2048, 6144, capi.INT8_KERNEL_GEMV), (8, 2049, 6144, capi.INT8_KERNEL_SPLIT),  # 192 workgroups
    (5, 3000, 6113, capi.INT8_KERNEL_SPLIT), (5, 3000, 6112, capi.INT8_KERNEL_GEMV),
    (9, 1024, 6144, capi.INT8_KERNEL_GEMV), (9, 1025, 6144, capi.INT8_KERNEL_SPLIT),
    (16, 4096, 8192, capi.INT8_KERNEL_SPLIT), (16, 4096, 8193, capi.INT8_KERNEL_GEMV),
    (4, 16384, 256, capi.INT8_KERNEL_GEMV), (5, 16384, 256, capi.INT8_KERNEL_SPLIT)])
def test_up_to_sixteen_rows(rows, depth, channels, kernel):
    assert _kernel(rows, depth, channels) == kernel


@pytest.mark.parametrize("rows,depth,channels,kernel", [
    (768, 512, 8192, capi.INT8_KERNEL_TILES_64X128), (768, 512, 8193, capi.INT8_KERNEL_TILES_128X256),  # 768 tiles
    (392, 704, 14656, capi.INT8_KERNEL_TILES_128X256), (652, 576, 9024, capi.INT8_KERNEL_TILES_128X256)])
def test_short_walks_in_up_to_three_rounds_of_64x128(rows, depth, channels, kernel):
    assert _kernel(rows, depth, channels) == kernel


@pytest.mark.parametrize("rows,depth,channels,kernel", [
    (1778, 1949, 6928, capi.INT8_KERNEL_TILES_128X256), (1600, 1434, 7948, capi.INT8_KERNEL_TILES_128X256),
    (1778, 1952, 6928, capi.INT8_KERNEL_TILES_64X128),  # whole pieces
    (1778, 1023, 6928, capi.INT8_KERNEL_TILES_64X128),  # shallow
    (1536, 1949, 8192, capi.INT8_KERNEL_TILES_64X128)])  # 768 tiles: three rounds for two
def test_ragged_rows_read_twice_in_two_rounds_for_one(rows, depth, channels, kernel):
    assert _kernel(rows, depth, channels) == kernel


S, T, A, Q, L = (capi.INT8_TILES_SPLIT, capi.INT8_TILES_64X128, capi.INT8_TILES_64X128_AHEAD,
                 capi.INT8_TILES_128X128, capi.INT8_TILES_128X256)


@pytest.mark.parametrize("rows,depth,channels,tiles,first", [
    (1, 2048, 2048, capi.INT8_TILES_NONE, 1), (77, 3008, 5003, S, 77),
    (130, 2048, 8200, T, 130), (130, 2049, 8200, A, 130),  # four steps ahead from there on ...
    (300, 2049, 6528, A, 300), (300, 2049, 6529, Q, 300),  # ... in one round of 64 x 128; 128 x 128 beyond it
    (300, 2048, 6529, Q, 300), (300, 2047, 6529, T, 300),
    (1000, 2048, 4096, L, 1000), (1000, 2049, 4096, Q, 1000), (1000, 2049, 4097, L, 1000),  # half a round
    (1100, 511, 7300, L, 1100), (1100, 512, 7300, Q, 1100), (1100, 2048, 7300, Q, 1100), (1100, 2049, 8192, L, 1024),
    (1024, 4096, 8192, L, 1024), (1025, 4096, 8192, L, 1024), (1280, 4096, 8192, L, 1024),  # 256, 288, 320 tiles
    (1281, 4096, 8192, L, 1281), (1025, 2048, 8192, Q, 1025), (640, 4096, 15616, L, 512),
    (1152, 4096, 8448, L, 1152)])  # 231 tiles in the rows of a round: too few
def test_tiles_of_the_gemm(rows, depth, channels, tiles, first):
    n = C.c_int()
    assert (capi.load().lrtfc_fc_int8_packed_tiles(rows, depth, channels, C.byref(n)), n.value) == (tiles, first)
    assert capi.load().lrtfc_fc_int8_packed_tiles(rows, depth, channels, None) == tiles
