"""Which form a launch of the seq operators takes on 256 compute units: frhip_seq_gemm_form, a function of the sizes alone."""
import ctypes as C
import importlib

import pytest

fr = importlib.import_module("faster-rwkv_amd")

TILES, FEW, SPLIT, ONE_BY_ONE = range(4)
V4, VALUE = 1, 2


def form(T, K, *N, which=0):
    out = (C.c_int * 2)()
    f = fr.lib().frhip_seq_gemm_form(T, K, len(N), (C.c_int * len(N))(*N), which, 256, out)
    assert f >= 0, fr.lib().frhip_error_string()
    return f, out[0], out[1]


@pytest.mark.parametrize("T,K,N", [(4, 256, (256,) * 4), (64, 256, (256, 1024)), (65, 320, (320,) * 3), (300, 448, (448,) * 4), (100, 384, (384, 1344))])
def test_a_group_without_two_slices_stays_one_launch(T, K, N):
    """K of four to seven steps of 64: a slice has at least four, so that neither the group nor its members are split."""
    assert form(T, K, *N) == (TILES, 0, 0)
    assert all(form(T, K, n) == (TILES, 0, 0) for n in N)


def test_groups_that_are_split_as_a_whole_or_product_by_product():
    assert form(40, 2560, *(2560,) * 4) == (SPLIT, 3, 0)
    assert form(13, 2560, 2560, 8960) == (SPLIT, 2, 0)
    assert form(130, 2048, 2048, 8192)[0] == ONE_BY_ONE and form(130, 2048, 2048)[0] == SPLIT
    assert form(361, 2048, 2048)[0] == TILES  # no scratch
    assert form(512, 8960, 2560, which=VALUE) == (SPLIT, 3, 0)


@pytest.mark.parametrize("T,c,f,rk,v", [(16, 2048, 8192, (SPLIT, 3, 0), (SPLIT, 16, 0)), (130, 2048, 8192, (ONE_BY_ONE, 0, 0), (SPLIT, 5, 0)),
                                        (200, 2560, 8960, (TILES, 0, 0), (SPLIT, 3, 0)), (300, 2048, 8192, (TILES, 0, 0), (SPLIT, 3, 0)),
                                        (64, 512, 1792, (SPLIT, 2, 0), (SPLIT, 7, 0)), (33, 768, 3072, (SPLIT, 3, 0), (SPLIT, 12, 0)),
                                        (13, 576, 1856, (SPLIT, 2, 0), (SPLIT, 7, 0)), (13, 2560, 8960, (SPLIT, 2, 0), (SPLIT, 12, 0)),
                                        (64, 512, 2048, (SPLIT, 2, 0), (SPLIT, 8, 0)), (65, 768, 3072, (SPLIT, 3, 0), (SPLIT, 12, 0))])
def test_what_the_operator_tests_of_ffn_seq_run(T, c, f, rk, v):
    assert form(T, c, c, f) == rk and form(T, f, c, which=VALUE) == v


@pytest.mark.parametrize("T,c", [(64, 512), (24, 2048), (37, 768), (150, 2048), (66, 2560), (500, 512)])
def test_what_the_operator_tests_of_att_seq_v4_run(T, c):
    assert form(T, c, c, c, c, which=V4)[0] == form(T, c, c, which=V4)[0] == FEW


@pytest.mark.parametrize("T,c,f,rk,v", [(1, 512, 1024, FEW, FEW), (13, 2560, 8960, FEW, FEW), (16, 2048, 8192, FEW, FEW), (65, 768, 3072, FEW, FEW),
                                        (200, 768, 3072, FEW, FEW), (130, 2048, 8192, FEW, SPLIT), (300, 2048, 8192, TILES, SPLIT),
                                        (40, 2816, 11264, SPLIT, SPLIT), (17, 5120, 20480, ONE_BY_ONE, SPLIT)])
def test_forms_of_rwkv4_ffn(T, c, f, rk, v):
    assert form(T, c, c, f, which=V4)[0] == rk and form(T, f, c, which=V4 + VALUE)[0] == v


def test_the_expected_times_decide_up_to_512_rows():
    for T, c, f in ((361, 768, 3072), (512, 768, 3072), (400, 1280, 5120)):
        assert form(T, c, c, which=V4)[0] == form(T, f, c, which=V4 + VALUE)[0] == FEW
    assert form(500, 512, *(512,) * 3, which=V4)[0] == form(512, 2048, 2048, which=V4)[0] == FEW
    assert form(512, 4096, 4096, which=V4)[0] == form(513, 768, 768, which=V4)[0] == TILES


@pytest.mark.parametrize("T", [4, 16, 64, 65, 128, 360, 361])
def test_rwkv5_sums_are_never_those_of_the_kernel_for_a_few_rows(T):
    for c, f in ((256, 896), (1024, 3584), (2560, 8960), (4096, 14336)):
        for which, K, N in ((0, c, (c,) * 4), (0, c, (c,) * 3), (0, c, (c,)), (0, c, (c, f)), (VALUE, f, (c,))):
            assert form(T, K, *N, which=which)[0] != FEW
        assert form(T, c, c, which=V4)[0] == FEW


def test_arguments():
    out = (C.c_int * 2)()
    f = fr.lib().frhip_seq_gemm_form
    one = (C.c_int * 1)(64)
    assert f(4, 64, 1, None, 0, 256, out) == -1 and f(4, 64, 1, one, 0, 256, None) == -1
    assert f(0, 64, 1, one, 0, 256, out) == f(4, 96, 1, one, 0, 256, out) == f(4, 64, 5, one, 0, 256, out) == -2
