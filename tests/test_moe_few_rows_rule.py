"""Which layers take the few-rows kernel, and which the one for items of 288 rows (host only; without a GPU the rules assume
256 CUs). Both sides of each line of the few-rows rule are layers that were timed on both kernels."""
import pytest

import hipkittens_amd

lib = hipkittens_amd.load_library()


@pytest.mark.parametrize("H,I,E,k,T,mxfp8,ext,rows", [
    # means of 4 and 8 rows per expert
    (2880, 2880, 32, 4, 32, 0, 0, 16), (2880, 2880, 32, 4, 33, 0, 0, 32), (2880, 2880, 32, 4, 64, 0, 0, 32),
    (2880, 2880, 32, 4, 65, 0, 0, 0), (2880, 2880, 32, 4, 32, 1, 0, 16), (2880, 2880, 32, 4, 33, 1, 0, 0),
    # layers that the streaming kernel runs at full rate (3 to 7 % slower on the few-rows kernel from a mean of 4 on)
    (3072, 3072, 128, 4, 32, 0, 0, 16), (3072, 3072, 128, 4, 33, 0, 0, 0), (3072, 3072, 128, 4, 256, 0, 0, 0),
    (3072, 3072, 128, 4, 64, 0, 1, 16), (3072, 3072, 128, 4, 65, 0, 1, 0), (3072, 3072, 128, 4, 64, 1, 0, 16),
    (3072, 3072, 128, 4, 65, 1, 0, 0), (3072, 3072, 128, 4, 128, 1, 1, 16), (4096, 4096, 128, 8, 128, 0, 0, 0),
    (2048, 2048, 256, 8, 256, 0, 0, 0), (7168, 2048, 128, 8, 64, 0, 0, 0), (2880, 3392, 256, 8, 128, 0, 0, 0),
    (4928, 3840, 128, 8, 128, 0, 1, 0),
    # those that it runs a little below that: no items of 32 rows
    (2880, 2880, 128, 4, 128, 0, 0, 16), (2880, 2880, 128, 4, 129, 0, 0, 0), (2624, 2048, 256, 8, 256, 0, 0, 0),
    (1664, 4096, 256, 8, 256, 0, 0, 0), (1664, 4096, 256, 8, 256, 0, 1, 0),
    # fewer items per CU, the longer epilogues, or many K-steps walked without weights
    (4096, 4096, 64, 4, 128, 0, 0, 32), (4096, 2752, 128, 8, 64, 0, 1, 16), (2880, 2880, 128, 4, 256, 0, 1, 32), (4096, 2048, 128, 8, 64, 0, 1, 16),
    (2944, 2304, 128, 8, 64, 0, 0, 16), (3456, 2880, 128, 8, 67, 0, 1, 32), (2688, 1664, 256, 8, 160, 0, 1, 32),
    (2688, 1664, 256, 8, 160, 0, 0, 0), (2112, 3776, 128, 8, 128, 0, 0, 32), (1984, 1216, 256, 8, 256, 0, 1, 32)])
def test_mxfp4(H, I, E, k, T, mxfp8, ext, rows):
    assert lib.hk_moe_mxfp4_few_rows(T, H, I, E, k, mxfp8, ext) == rows


@pytest.mark.parametrize("H,I,E,k,T,rows", [
    (7168, 2048, 256, 8, 64, 16), (7168, 2048, 256, 8, 65, 0),       # two rows per expert
    (7168, 2048, 1, 1, 191, 16), (7168, 2048, 1, 1, 192, 0),         # 3/4 of an item of the gate+up GEMM per CU
    (1024, 512, 1, 1, 192, 16), (1024, 512, 1, 1, 193, 0),           # twelve times an expert's weights
    (128, 128, 64, 64, 512, 0), (256, 896, 2, 1, 384, 16), (256, 896, 2, 1, 385, 0)])
def test_fp8blk(H, I, E, k, T, rows):
    assert lib.hk_moe_fp8blk_few_rows(T, H, I, E, k) == rows


@pytest.mark.parametrize("H,I,E,k,T,mxfp8,ext,rows", [
    (2880, 2880, 128, 4, 16384, 0, 1, 288), (2880, 2880, 128, 4, 12800, 0, 1, 288), (2880, 2880, 128, 4, 12799, 0, 1, 192),
    (2880, 2880, 128, 4, 16384, 1, 0, 144), (2880, 2880, 128, 4, 1000, 1, 0, 128), (2880, 2880, 128, 4, 4, 0, 1, 16),
    (512, 2880, 128, 4, 16384, 0, 0, 192), (544, 2880, 128, 4, 16384, 0, 0, 288),     # three K-steps
    (2880, 512, 128, 4, 16384, 0, 0, 192)])
def test_mxfp4_item_rows(H, I, E, k, T, mxfp8, ext, rows):
    assert lib.hk_moe_mxfp4_item_rows(T, H, I, E, k, mxfp8, ext) == rows


@pytest.mark.parametrize("H,I,E,k,T,rows", [
    (7168, 2048, 256, 8, 8192, 288), (7168, 2048, 256, 8, 64, 16), (7168, 2048, 256, 8, 2048, 144),
    # whole rows of mean + two standard deviations: 144 and 145, 160 and 161, 288 and 289 (there two items of either length)
    (7168, 2048, 256, 8, 3930, 144), (7168, 2048, 256, 8, 3931, 160), (7168, 2048, 256, 8, 4401, 160),
    (7168, 2048, 256, 8, 4402, 288), (7168, 2048, 256, 8, 8222, 288), (7168, 2048, 256, 8, 8223, 160),
    (256, 2048, 256, 8, 8192, 144), (384, 2048, 256, 8, 8192, 288), (7168, 256, 256, 8, 8192, 144),   # three K-steps
    (7168, 2048, 1, 1, 1400, 160), (7168, 2048, 1, 1, 3000, 288)])   # one round either way; two rounds and one
def test_fp8blk_item_rows(H, I, E, k, T, rows):
    assert lib.hk_moe_fp8blk_item_rows(T, H, I, E, k) == rows


def test_refused_shapes():
    assert lib.hk_moe_mxfp4_few_rows(0, 2880, 2880, 128, 4, 0, 0) == -2
    assert lib.hk_moe_mxfp4_few_rows(4, 2880, 2880, 4, 8, 0, 0) == -2
    assert lib.hk_moe_fp8blk_few_rows(4, 100, 128, 4, 2) == -2
    assert lib.hk_moe_mxfp4_item_rows(4, 2880, 2880, 4, 8, 0, 0) == -2 and lib.hk_moe_fp8blk_item_rows(4, 100, 128, 4, 2) == -2
