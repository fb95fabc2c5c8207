"""How launches of binary16 products go out in tiles: frhip_gemm_route, a function of the sizes alone, for 256 compute units.  The
figures are microseconds, measured on an MI355X."""
import ctypes as C
import importlib

import pytest

fr = importlib.import_module("faster-rwkv_amd")


def route(T, K, *N):
    """-> launches, [(rows of a tile, widest tile in blocks of 32 columns, rounds, loader wave)] per product"""
    out = (C.c_int * (4 * len(N)))()
    launches = fr.lib().frhip_gemm_route(T, K, len(N), (C.c_int * len(N))(*N), 256, out)
    assert launches > 0, launches
    return launches, [tuple(out[4 * i:4 * i + 4]) for i in range(len(N))]


@pytest.mark.parametrize("T,K,N", [(300, 2048, 6144), (129, 2048, 10240), (129, 2560, 8960)])
def test_one_round_of_64_row_tiles_is_kept_where_it_is_cheaper(T, K, N):
    assert route(T, K, N) == (1, [(64, 4, 1, 1)])


@pytest.mark.parametrize("T,K,N,rows", [(2048, 2048, 8192, 256), (4096, 2048, 8192, 256),
                                        (3000, 2048, 8192, 128),   # 113 against 115
                                        (1500, 4096, 14336, 128),  # 185 against 187
                                        (640, 2048, 65536, 128),   # 189 against 217
                                        (768, 2048, 8192, 128),    # 35 against 37
                                        (512, 768, 6144, 128)])    # 128 x 96
def test_tile_height(T, K, N, rows):
    assert route(T, K, N)[1][0][0] == rows


def test_what_goes_out_is_what_is_told():
    """The launch takes the tiles with four loading waves exactly where frhip_gemm_ring_tile says so, with those tiles."""
    ring = 0
    for T in (4, 65, 300, 513, 777, 1024, 1472, 1793, 3000, 4099, 16400):
        for K in (64, 320, 2048, 8192):
            for N in ((64,), (1111,), (2048,), (50277,), (768, 10752), (2048, 8192), (2560, 2560, 2560, 2560)):
                launches, told = route(T, K, *N)
                for i in range(1 if launches == 1 else len(N)):
                    n = N if launches == 1 else N[i:i + 1]
                    out = (C.c_int * 4)()
                    assert fr.lib().frhip_gemm_ring_tile(T, K, len(n), (C.c_int * len(n))(*n), 1, 256, out) == 0
                    ring += out[3]
                    if out[3]:
                        assert told[i] == (out[0], out[1], out[2], 1)
                    else:
                        assert told[i][0] == 256
    assert ring > 100


@pytest.mark.parametrize("T,K,N,loader", [(512, 5120, 20480, 1),    # 101 against 115 without the loader wave
                                          (1024, 5120, 20480, 1),   # 200 against 219
                                          (2048, 20480, 5120, 1),   # 375 against 423
                                          (768, 2560, 11520, 1),    # 51 against 59
                                          (1793, 5120, 5120, 0),    # 119 with it against 101: rows past the end
                                          (1025, 320, 10000, 0),
                                          (2048, 2048, 5110, 0),    # columns past the end
                                          (2048, 2048, 8192, 0)])   # wider than its stages allow
def test_loader_wave_of_256_row_tiles(T, K, N, loader):
    rows, blocks, _, got = route(T, K, N)[1][0]
    assert (rows, got) == (256, loader) and (blocks <= 5 or not loader)


@pytest.mark.parametrize("T", [8192, 8193, 16000, 100000])
def test_no_limit_on_rounds(T):
    """The logits of every position of a long text: planned tiles, however many rounds they take."""
    rows, blocks, rounds, _ = route(T, 2048, 65536)[1][0]
    assert (rows, blocks) == (256, 8) and -(-T // 256) * 256 <= rounds * 256 < -(-T // 256) * 256 + 512


def test_many_products_of_few_columns():
    """More strips than compute units: a round holds a part of a strip."""
    assert route(300000, 64, 96, 96, 96, 96)[1][0][0] in (0, 128, 256)
    assert route(300000, 64, 32) == (1, [(64, 1, 19, 1)])


def test_rows_too_long_for_32_bit_offsets_go_out_on_fixed_tiles():
    """The lane offsets of planned tiles reach 255 rows and 128 bytes beyond a tile's first: 2 K 256 must stay below 2^32."""
    k = (1 << 32) // 512 - 64
    assert k % 64 == 0 and route(2048, k, 8192)[1][0] == (256, 8, 1, 0)
    for more in (64, 128, 1 << 20):
        assert route(2048, k + more, 8192) == (1, [(0, 0, 0, 0)])


def test_an_extra_launch_costs_the_same_whatever_k():
    """2048 and 8192 columns one by one save part of a round, which grows with K; the launch they cost does not."""
    assert [route(1793, k, 2048, 8192)[0] for k in (512, 1024, 2048, 4096)] == [1, 1, 2, 2]


def test_refused_sizes():
    lib, n, out = fr.lib(), (C.c_int * 1)(64), (C.c_int * 4)()
    for args in ((0, 64, 1), (4, 96, 1), (4, 64, 0), (4, 64, 5)):
        assert lib.frhip_gemm_route(*args, n, 256, out) == -2
    assert lib.frhip_gemm_route(4, 64, 1, None, 256, out) == -1
