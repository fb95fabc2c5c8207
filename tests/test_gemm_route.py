"""How launches of binary16 products are cut into tiles: frhip_gemm_route, a function of the sizes alone.  The expected
cuts are the faster ones of what was measured on an MI355X (256 compute units); the figures are microseconds."""
import ctypes as C
import importlib

import pytest

fr = importlib.import_module("faster-rwkv_amd")


def route(T, K, *N):
    """-> launches, [(rows of a tile, widest tile in blocks of 32 columns, rounds)] per product"""
    out = (C.c_int * (3 * len(N)))()
    launches = fr.lib().frhip_gemm_route(T, K, len(N), (C.c_int * len(N))(*N), 256, out)
    assert launches > 0, launches
    return launches, [tuple(out[3 * i:3 * i + 3]) for i in range(len(N))]


@pytest.mark.parametrize("T,K,N", [(300, 2048, 6144),   # 19.2 against 22.7 as 128 x 96
                                   (129, 2048, 10240),  # 19.0 against 21.6
                                   (129, 2560, 8960)])  # 24.8 against 26.3
def test_one_round_of_64_row_tiles_is_kept_where_it_is_cheaper(T, K, N):
    assert route(T, K, N) == (1, [(64, 4, 1)])


@pytest.mark.parametrize("T,K,N,rows", [(3000, 2048, 8192, 256),   # 105.5 against 119 as three rounds of 128 rows
                                        (1500, 4096, 14336, 256),  # 176 against 209
                                        (640, 2048, 65536, 128),   # 200 against 217
                                        (768, 2048, 8192, 128),    # 32 against 37
                                        (512, 768, 6144, 128)])    # 128 x 96
def test_tile_height(T, K, N, rows):
    assert route(T, K, N)[1][0][0] == rows


def test_an_extra_launch_costs_the_same_whatever_k():
    """2048 and 8192 columns one by one save part of a round, which grows with K; the launch they cost does not."""
    assert [route(3074, k, 2048, 8192)[0] for k in (512, 1024, 2048, 4096)] == [1, 1, 2, 2]


def test_refused_sizes():
    lib, n, out = fr.lib(), (C.c_int * 1)(64), (C.c_int * 3)()
    for args in ((0, 64, 1), (4, 96, 1), (4, 64, 0), (4, 64, 5)):
        assert lib.frhip_gemm_route(*args, n, 256, out) == -2
    assert lib.frhip_gemm_route(4, 64, 1, None, 256, out) == -1
