"""Which products of 25 to 64 rows go to the vendor library, against times measured on MI355X (microseconds over distinct weights, own kernels and library) at sizes
inside, beside and far from where the rule's lines lie: rows of 4 KB or a multiple apart and others, rows that are no whole number of 256 bytes, sums of 768 to
7,168, outputs below, in and above one round of the library's tiles."""
import ctypes

import pytest

from levanter_amd.kernels import build
from levanter_amd.kernels.library import HipKernels

MEASURED = [  # rows, outputs, inputs, own kernels, library
    (32, 14480, 4608, 28.3, 26.1), (64, 14480, 4608, 33.8, 29.5), (32, 14896, 4544, 28.3, 36.8), (64, 14896, 4544, 33.4, 41.9), (48, 11552, 4608, 25.8, 26.6),
    (32, 12288, 4096, 21.2, 22.8), (64, 12288, 4096, 25.2, 25.0), (25, 13312, 5120, 30.9, 27.4), (48, 16384, 4096, 28.5, 32.5), (48, 16400, 4096, 37.6, 38.2),
    (64, 16384, 5120, 40.0, 35.4), (64, 14336, 7168, 48.2, 42.5), (64, 18432, 6144, 62.8, 60.1), (48, 15360, 6144, 40.2, 44.7), (64, 22528, 4096, 51.9, 44.7),
    (32, 24576, 6144, 56.9, 67.1), (64, 32768, 4096, 55.4, 60.5), (32, 25504, 4736, 56.6, 44.9), (32, 24000, 1024, 12.6, 31.3), (64, 24000, 768, 16.0, 13.6),
    (32, 50257, 768, 21.2, 19.8), (64, 50257, 1600, 40.6, 34.6), (48, 32000, 2048, 29.0, 35.6), (64, 50257, 2048, 54.9, 49.4), (32, 65536, 1024, 31.2, 29.9),
    (25, 100352, 1600, 67.0, 178.2), (48, 128256, 2048, 110.2, 128.6), (64, 100000, 768, 47.6, 62.4), (40, 32064, 768, 15.4, 28.9), (48, 40960, 1600, 33.8, 29.7),
    (40, 10416, 1984, 13.7, 20.0), (32, 32000, 1600, 23.8, 34.8), (40, 8048, 2304, 11.3, 14.8), (50, 28176, 512, 13.2, 25.8),
]


@pytest.mark.parametrize("M,N,K,own,library", MEASURED)
def test_the_choice_is_the_faster_one(M, N, K, own, library):
    taken = library if HipKernels.use_library(M, N, K, 0) else own
    assert taken <= 1.03 * min(own, library)


def test_below_25_rows_and_for_other_activations_never():
    for _, N, K, _, _ in MEASURED:
        assert not HipKernels.use_library(24, N, K, 0)
        assert not any(HipKernels.use_library(64, N, K, act) for act in range(8) if act not in HipKernels.LIBRARY_ACTIVATIONS)


def test_sums_that_the_librarys_single_chain_would_make_less_exact_stay_ours():
    for N, K in ((50257, 4096), (27648, 5120), (12000, 1280), (65024, 2560)):
        assert not any(HipKernels.use_library(M, N, K, 0) for M in range(1, 65))


# experts, width, inner width, rows an expert, microseconds of the up and the down product with tiles of 16 and of 128 rows
EXPERTS = [(8, 2048, 4096, 12, 61.9, 87.5), (16, 2048, 2048, 14, 65.9, 74.5), (16, 1024, 1024, 16, 23.3, 27.2), (32, 2048, 1024, 13, 63.8, 66.5), (33, 2048, 2048, 16, 150.2, 183.5),
           (32, 4096, 2048, 14, 232.9, 254.6), (64, 1024, 512, 13, 30.5, 34.1), (64, 2048, 2048, 14, 268.1, 256.2), (64, 2048, 1024, 15, 136.6, 127.5), (64, 2048, 2048, 16, 298.5, 253.2),
           (128, 1024, 768, 12, 95.1, 95.2), (128, 2048, 1024, 13, 253.8, 245.4), (128, 2048, 1024, 16, 305.1, 243.5), (256, 1024, 512, 14, 141.1, 129.3), (256, 1024, 512, 12, 125.8, 127.9)]


@pytest.mark.parametrize("experts,width,inner,rows,few,many", EXPERTS)
def test_the_tiles_of_the_experts_products_are_the_faster_ones(experts, width, inner, rows, few, many):
    taken = {16: few, 128: many}[HipKernels.moe_tile_rows(rows * experts, experts)]
    assert taken <= 1.05 * min(few, many)


# rows, outputs, inputs; for each of the library's kernels the order in which it adds up (0: the first kernel's bits, and so on) and its microseconds
STOPWATCH = (1088, 4096, 16384, (0, 0, 0, 1, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 4, 3),
             (201.1, 204.9, 213.5, 320.8, 313.0, 329.9, 180.4, 309.8, 200.0, 290.2, 319.9, 191.0, 187.3, 184.2, 315.0, 254.4))


@pytest.fixture(scope="module")
def keeps(core):
    library = ctypes.CDLL(build.ensure_built("gemm_library"))

    def kept(bits, us):
        n = len(bits)
        return library.lev_linear_library_keeps((ctypes.c_ulonglong * n)(*bits), (ctypes.c_float * n)(*us), n)

    return kept


def test_the_order_of_the_librarys_sums_does_not_hang_on_a_stopwatch(keeps):
    """Times that are off by up to 2 %, as those of two processes are: always a kernel with the same bits. Of these the fastest."""
    import random

    *_, bits, us = STOPWATCH
    rng = random.Random(1)
    noisy = [[t * rng.uniform(0.98, 1.02) for t in us] for _ in range(500)]
    assert {bits[min(range(len(us)), key=t.__getitem__)] for t in noisy} == {3, 10}  # what the fastest alone gives
    assert {bits[keeps(bits, t)] for t in noisy} == {3}
    assert keeps(bits, us) == 6


@pytest.mark.parametrize("bits,us,kept", [
    ((0, 1, 2), (216.0, 216.5, 205.8), 2),                          # nobody shares an order: the fastest
    ((0, 1, 2), (206.0, 216.5, 205.8), 0),                          # within the stopwatch's error: the heuristic's earlier one
    ((0, 0, 1, 1, 1), (99.0, 104.0, 103.0, 99.5, 99.9), 3),         # the one that more kernels have
    ((0, 0, 1, 1, 1), (97.0, 104.0, 103.0, 99.5, 99.9), 0),         # unless it is behind
    ((0, 1, 1, 2), (90.0, 104.0, 103.0, 80.0), 2),                  # one kernel's own order is left out
    ((0, 0, 0), (100.0, 99.9, 99.8), 2), ((0, 0), (-1.0, 7.0), 1),  # one order: the fastest that ran
    ((0, 0, 1), (-1.0, 7.0, 9.0), 1), ((5,), (3.0,), 0), ((0, 1), (-1.0, -1.0), -1),
])
def test_which_of_the_librarys_kernels_is_kept(keeps, bits, us, kept):
    assert keeps(bits, us) == kept


# the 32-bit products, over weights that no cache holds
TILES = [  # rows, outputs, inputs, microseconds of the tiles in the order of the kernels' two lists
    (100, 5120, 6400, (203.6, 171.7, 172.8, 180.6, 143.5, 150.0, 112.8, 119.1, 129.8, 129.3, 137.8, 165.4)),
    (203, 3072, 6400, (223.6, 199.9, 175.6, 181.5, 143.9, 147.5, 114.1, 113.5, 125.5, 126.3, 133.5, 163.5)),
    (256, 3072, 4096, (171.0, 132.7, 133.3, 117.1, 94.4, 97.1, 76.3, 75.8, 81.8, 81.9, 84.9, 107.0)),
    (777, 768, 6400, (220.3, 171.0, 172.6, 173.5, 139.5, 139.6, 110.9, 103.7, 117.0, 122.4, 129.8, 162.1)),
    (404, 1600, 4096, (156.0, 127.5, 131.1, 113.9, 91.5, 93.6, 75.0, 70.7, 77.6, 79.3, 83.8, 106.1)),
    (512, 1200, 6400, (221.8, 171.7, 174.0, 174.7, 142.9, 140.0, 112.3, 105.7, 117.7, 122.2, 130.4, 162.5)),
    (160, 4096, 4096, (145.7, 111.9, 113.8, 117.7, 96.2, 97.3, 76.7, 75.3, 82.6, 83.7, 86.7, 106.6)),
    (33, 10240, 2048, (58.2, 57.9, 47.7, 44.9, 49.3, 51.8, 42.5, 43.0, 46.8, 47.2, 49.5, 57.9)),
    (100, 5120, 3072, (99.0, 83.5, 85.3, 89.7, 71.5, 75.0, 59.2, 59.1, 64.4, 64.5, 68.7, 81.9)),
    (1500, 400, 4096, (142.2, 109.5, 110.0, 112.8, 90.7, 90.2, 74.8, 67.5, 77.1, 78.0, 83.8, 105.2)),
    (100, 6400, 3072, (121.6, 115.0, 101.3, 93.9, 93.3, 75.5, 61.0, 67.4, 65.2, 81.0, 69.2, 82.8)),
    (777, 3072, 1024, (132.0, 105.5, 103.6, 102.4, 78.2, 62.2, 66.4, 54.6, 47.5, 53.8, 53.7, 53.5)),
    (404, 768, 3072, (56.8, 51.7, 52.4, 58.5, 46.2, 39.4, 58.3, 49.8, 55.3, 60.9, 65.0, 80.6)),
    (1024, 4096, 4096, (896.8, 680.4, 683.6, 585.4, 467.6, 360.1, 335.2, 347.4, 311.2, 311.7, 266.2, 286.0)),
    (64, 768, 768, (5.5, 6.9, 7.0, 10.5, 8.3, 11.7, 18.8, 10.5, 12.0, 13.9, 16.8, 23.1)),
    (17, 1600, 1600, (8.7, 11.1, 12.3, 19.0, 14.8, 23.1, 30.5, 28.1, 31.6, 35.0, 36.7, 44.3)),
    (203, 2304, 768, (24.8, 20.6, 20.6, 19.8, 15.6, 13.1, 19.4, 15.2, 16.6, 18.4, 19.7, 24.1)),
    (1500, 10240, 1600, (1287.5, 994.4, 999.2, 813.1, 663.3, 532.5, 482.6, 497.8, 432.4, 411.3, 390.7, 407.8)),
    (48, 400, 6400, (25.2, 36.7, 38.8, 68.5, 48.7, 76.4, 108.9, 101.5, 113.0, 124.5, 132.9, 161.6)),
    (777, 25000, 96, (134.3, 161.8, 152.5, 106.5, 86.0, 74.8, 90.6, 58.2, 50.8, 50.6, 49.0, 53.0)),
    (777, 1600, 384, (30.9, 26.3, 25.7, 20.2, 18.6, 18.3, 23.0, 13.5, 14.3, 14.7, 17.0, 14.7)),
    (777, 1024, 4096, (183.3, 149.5, 151.0, 146.5, 117.8, 90.2, 74.2, 80.1, 76.3, 105.2, 84.1, 105.9)),
    (777, 1024, 1024, (47.7, 40.3, 39.6, 41.3, 32.5, 26.5, 23.7, 22.3, 21.4, 29.5, 21.7, 29.9)),
    (777, 50257, 1024, (2115.1, 1670.5, 1652.2, 1539.1, 1188.0, 926.8, 844.0, 833.1, 747.2, 737.3, 706.9, 696.5)),
    (662, 25055, 96, (117.7, 148.5, 145.4, 99.1, 86.6, 77.5, 88.2, 59.4, 54.0, 53.3, 55.3, 58.2)),
]
SPLIT = [  # rows, outputs, inputs, microseconds on the 32-bit instruction and of the three tiles of split operands
    (92, 50257, 576, 62.7, (74.1, 76.1, 99.1)), (149, 8535, 6212, 180.2, (224.9, 205.8, 192.2)), (349, 9882, 256, 22.9, (26.7, 25.8, 36.7)), (548, 7246, 1024, 77.8, (95.2, 87.2, 101.4)),
    (1254, 3204, 4292, 297.2, (347.1, 326.6, 300.1)), (264, 8243, 680, 37.6, (40.7, 40.5, 46.2)), (1853, 2304, 1972, 144.3, (170.9, 155.5, 178.2)), (1451, 3072, 1192, 92.0, (108.7, 96.7, 119.7)),
    (1207, 3528, 2292, 168.7, (195.1, 178.2, 197.7)), (860, 6787, 308, 42.7, (51.1, 44.9, 60.8)), (1274, 1200, 6400, 182.2, (222.5, 189.5, 189.5)), (1510, 3072, 720, 58.4, (71.2, 60.6, 82.3)),
    (777, 4096, 1024, 63.8, (49.8, 53.4, 77.8)), (777, 1024, 4096, 74.3, (144.1, 105.3, 64.0)), (777, 3072, 1024, 47.1, (44.6, 49.1, 58.4)), (777, 1024, 1024, 21.8, (42.4, 29.2, 20.2)),
    (606, 3072, 768, 29.8, (34.3, 25.6, 31.9)), (2000, 11063, 1600, 563.4, (490.3, 507.7, 694.1)), (925, 2148, 3072, 103.8, (113.0, 92.9, 109.8)), (846, 3072, 900, 49.4, (43.0, 46.2, 55.8)),
    (1969, 3072, 496, 57.7, (55.8, 48.0, 76.5)), (123, 6191, 3072, 65.2, (115.4, 102.9, 54.5)), (708, 11626, 1244, 199.6, (192.8, 181.1, 231.5)), (2052, 768, 3596, 120.1, (132.2, 107.7, 117.0)),
    (103, 5451, 3072, 58.8, (114.3, 102.1, 48.8)), (1166, 2262, 3636, 177.7, (150.3, 173.6, 185.3)), (290, 768, 3096, 21.6, (112.5, 87.7, 46.2)), (298, 1024, 1768, 18.9, (67.6, 47.1, 29.0)),
    (512, 768, 3072, 35.8, (109.3, 83.8, 45.9)), (400, 768, 3072, 35.5, (109.9, 83.7, 45.6)),
]
# of one to eight rows
FEW_ROWS = [  # rows, outputs, inputs, microseconds of the few-row kernel and of the tiles
    (8, 1600, 2048, 12.4, 9.0), (5, 1200, 2048, 11.6, 8.3), (5, 1200, 3072, 12.5, 10.8), (8, 1600, 4096, 14.9, 14.8), (8, 1000, 2048, 7.3, 8.9),
    (6, 800, 1024, 5.5, 5.5), (8, 1400, 8192, 21.9, 26.4), (4, 3200, 2048, 11.1, 8.9), (4, 3200, 4096, 15.0, 14.3), (3, 2304, 2048, 9.3, 8.3),
    (4, 2800, 3072, 11.3, 11.4), (4, 1600, 256, 4.7, 3.5), (4, 1200, 256, 4.6, 3.4), (4, 1600, 1024, 5.5, 5.7), (3, 1000, 512, 3.9, 4.1), (4, 64, 256, 3.4, 2.9),
    (4, 800, 768, 4.0, 4.7), (2, 3200, 1024, 6.5, 5.8), (2, 2304, 256, 4.0, 3.4), (2, 2304, 768, 5.3, 5.2), (2, 2800, 1600, 6.8, 7.2), (2, 1200, 256, 3.6, 3.4),
    (2, 1600, 512, 3.8, 4.1), (2, 600, 128, 2.9, 2.7), (2, 6400, 4096, 21.3, 26.6), (1, 6400, 256, 5.4, 4.4), (1, 6400, 1024, 7.9, 9.1), (1, 2304, 64, 2.9, 2.7),
    (1, 2304, 256, 3.4, 3.4), (1, 4096, 384, 4.7, 4.5), (1, 800, 64, 2.5, 2.5), (1, 12800, 2048, 19.7, 25.7), (1, 16, 16384, 4.8, 36.6), (7, 200, 16384, 17.5, 46.2),
]


@pytest.fixture(scope="module")
def core():
    return ctypes.CDLL(build.ensure_built("core"), mode=ctypes.RTLD_GLOBAL)


@pytest.mark.parametrize("M,N,K,us", TILES)
def test_the_tile_of_a_32_bit_product_is_among_the_fastest(core, M, N, K, us):
    """Within 8 % of the fastest that is no less exact than a split of K in four: 32 x 64 and 32 x 96 tiles (places 8, 9) from 128 inputs on, larger ones from 256."""
    allowed = [t for i, t in enumerate(us) if i < 8 or K >= 256 or (K >= 128 and i < 10)]
    assert us[core.lev_linear_f32_choice(M, N, K)] <= 1.08 * min(allowed)


@pytest.mark.parametrize("M,N,K,whole,split", SPLIT)
def test_operands_are_split_only_where_that_is_faster(core, M, N, K, whole, split):
    tile = core.lev_linear_f32_split(M, N, K)
    taken = split[tile] if tile >= 0 else whole
    assert taken <= 1.02 * whole and taken <= 1.12 * min(whole, *split)


@pytest.mark.parametrize("M,N,K,few,tiles", FEW_ROWS)
def test_few_rows_of_a_32_bit_product_take_the_faster_kernel(core, M, N, K, few, tiles):
    assert (few if core.lev_linear_f32_choice(M, N, K) < 0 else tiles) <= 1.07 * min(few, tiles)
