"""Which products of 25 to 64 rows go to the vendor library, against times measured on MI355X (microseconds over distinct weights, own kernels and library) at sizes
inside, beside and far from where the rule's lines lie: rows of 4 KB or a multiple apart and others, rows that are no whole number of 256 bytes, sums of 768 to
7,168, outputs below, in and above one round of the library's tiles."""
import pytest

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
