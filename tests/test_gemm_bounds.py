"""The fp32 contraction touches nothing outside its operands: the index functions that its kernel calls, walked on the
CPU over every remainder of a tile, both parities and whole, ragged and split reductions."""
import ctypes
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def library(tmp_path_factory):
    path = str(tmp_path_factory.mktemp("gemm") / "gemm_bounds.so")
    subprocess.check_call([os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-shared", "-fPIC",
                           os.path.join(HERE, "gemm_bounds.cpp"), "-o", path])
    return ctypes.CDLL(path)


@pytest.fixture(scope="module")
def bounds(library):
    i64 = ctypes.c_int64

    def walk(kc, tile, extent, inner, ld, other_w, other_extent, k_chunk):
        outside, wrong = i64(), i64()
        library.gemm_bounds(int(kc), tile, i64(extent), i64(inner), i64(ld), other_w, i64(other_extent), i64(k_chunk),
                        ctypes.byref(outside), ctypes.byref(wrong))
        return outside.value, wrong.value
    return walk


@pytest.mark.parametrize("tile", [128, 96, 64, 32])
@pytest.mark.parametrize("kc", [False, True])
def test_every_load_lies_in_its_operand(bounds, kc, tile):
    for extent in list(range(1, tile + 1)) + list(range(2 * tile + 1, 3 * tile + 1)):
        for inner, k_chunk in ((32, 32), (64, 64), (33, 64), (95, 96), (96, 32), (100, 64), (1, 32),
                               (8, 32), (16, 32), (24, 32), (56, 64)):
            for other_w, other_extent in ((1, 5), (2, 6), (2, 5)):
                for pad in (0, 3):
                    ld = (inner if kc else extent) + pad
                    assert bounds(kc, tile, extent, inner, ld, other_w, other_extent, k_chunk) == (0, 0), \
                        (extent, inner, k_chunk, other_w, other_extent, pad)


@pytest.mark.parametrize("kc,tile,extent,inner,ld", [
    (False, 96, 160, 1024, 160),            # weights of 64 -> 160 channels, 16 basis values
    (False, 128, 100, 1024, 100), (False, 128, 224, 1024, 224),
    (False, 128, 720, 4096, 720),           # projection of 48 channels x 15, transposed
    (False, 128, 1680, 65536, 1680), (True, 128, 65536, 1680, 1680)])
def test_operands_of_convolutions(bounds, kc, tile, extent, inner, ld):
    for k_chunk in (inner, 512):
        assert bounds(kc, tile, extent, inner, ld, 2, 128, k_chunk) == (0, 0)


@pytest.mark.parametrize("tile", [128, 96, 64, 32])
@pytest.mark.parametrize("kc", [False, True])
def test_the_longest_rows_a_tile_takes(bounds, library, kc, tile):
    fits = lambda ld: library.tile_fits(tile, ctypes.c_int64(ld))
    ld = max(x for x in range((1 << 30) // tile - 64, (1 << 30) // tile + 1) if fits(x))
    assert ld >= 1 << 22 and not fits(ld + 1) and not fits(1 << 40)
    assert bounds(kc, tile, 2 * tile + 2, 100, ld, 1, 5, 64) == (0, 0)


@pytest.mark.parametrize("extent", [128, 129])
@pytest.mark.parametrize("other_w,other_extent", [(1, 5), (2, 5), (2, 6)])
def test_an_empty_reduction_has_no_steps(bounds, extent, other_w, other_extent):
    assert bounds(False, 128, extent, 0, extent, other_w, other_extent, 32) == (0, 0)


@pytest.mark.parametrize("rows", [9, 48, 64, 65, 720, 1024, 1920, 2560, 10240])
@pytest.mark.parametrize("cols", [1, 16, 128, 129, 256])
@pytest.mark.parametrize("batch", [1, 4])
def test_bf16_weight_gradient_is_split_into_one_round_of_workgroups_or_sixty_four_parts(library, rows, cols, batch):
    i64 = ctypes.c_int64
    floats = max(64 * rows * cols * batch, 1 << 20)
    tiles = -(-rows // 64) * -(-cols // 128) * batch
    for inner in (1, 63, 64, 1000, 4096, 8192, 20000, 29999, 30000, 65536, 200000):
        split = library.bf16_split(i64(rows), i64(cols), i64(inner), batch, i64(floats))
        assert 1 <= split <= max(1, inner // 64) and split * rows * cols * batch <= floats
        # four workgroups per CU at most ...
        assert split * tiles <= 1024 or split == 1 or (split == 64 and inner >= 30000)
        # ... and no fewer parts than 64 where the reduction is long
        assert inner < 30000 or split >= 64
