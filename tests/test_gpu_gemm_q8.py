"""Products of uint8 weights whose codes are dequantised on their way into LDS: the bits of the binary16 image, at every tile,
with remainders in rows, columns and K-steps, whole and in slices of K."""
import ctypes as C

import numpy as np
import pytest

from hipref import DevBuf, L, dev, fr


EXPANDED, TILES, ONE_BY_ONE, FEW = range(4)
V4, VALUE = 1, 2


def tile(T, K, *N, slices=1):
    out = (C.c_int * 3)()
    fr.check(L().frhip_gemm_q8_tile(T, K, len(N), (C.c_int * len(N))(*N), slices, 256, out))
    return tuple(out)


def few(T, K, N):
    out = (C.c_int * 2)()
    fr.check(L().frhip_gemm_few_tile(T, K, 1, (C.c_int * 1)(N), 256, out))
    return out[0] != 0


def way(T, K, *N, which=0):
    """frhip_seq_codes_way -> way, (rows of a tile, its widest in blocks of 32 columns, slices of K)"""
    out = (C.c_int * 3)()
    w = L().frhip_seq_codes_way(T, K, len(N), (C.c_int * len(N))(*N), which, 256, out)
    assert w >= 0, fr.lib().frhip_error_string()
    return w, tuple(out)


# one to sixteen K-steps (the producers hold four), and not the kernel for a few rows
CASES = [((64, 2, 1), 513, 64, 64), ((64, 3, 1), 520, 128, 80), ((64, 2, 1), 577, 192, 1600), ((64, 3, 1), 513, 256, 2672),
         ((128, 2, 1), 641, 320, 2608), ((128, 3, 1), 700, 384, 3600), ((128, 4, 1), 641, 448, 5232), ((128, 5, 1), 700, 128, 6416),
         ((128, 6, 1), 769, 320, 6384), ((128, 6, 2), 1025, 192, 10016), ((64, 4, 1), 385, 64, 3536), ((64, 5, 1), 129, 192, 12400),
         ((64, 8, 1), 129, 1024, 20560)]
# RWKV-5's ffn (rows, width, ffn width): what its r,k and its value product do with the codes
FFN = [((TILES, (64, 4, 1)), (TILES, (64, 2, 33)), 129, 64, 8512), ((TILES, (64, 5, 1)), (TILES, (64, 3, 42)), 129, 192, 12352),
       ((TILES, (64, 7, 1)), (EXPANDED, (0, 0, 0)), 257, 2240, 8960), ((TILES, (64, 8, 1)), (TILES, (64, 4, 10)), 129, 1024, 19648),
       ((TILES, (128, 4, 1)), (EXPANDED, (0, 0, 0)), 1024, 768, 3072), ((EXPANDED, (0, 0, 0)), (EXPANDED, (0, 0, 0)), 1030, 2048, 7168)]


def test_cases_reach_their_tiles():
    assert [tile(T, K, N) for _, T, K, N in CASES] == [t for t, *_ in CASES]
    assert not any(few(T, K, N) for _, T, K, N in CASES)
    assert tile(13, 2560, 2560, slices=10)[0] == 64 and tile(300, 2560, 2560, 8960) == (128, 5, 1)
    assert [(way(T, c, c, f), way(T, f, c, which=VALUE)) for _, _, T, c, f in FFN] == [v[:2] for v in FFN]


def test_every_tile_that_launches_of_the_operators_take_is_among_the_cases():
    """Rows of tiles and widths over models of 256 to 5120 channels; a wave's part of a tile follows from the two."""
    taken = set()

    def go(T, K, *N, which):
        w, out = way(T, K, *N, which=which)
        if w == ONE_BY_ONE:
            for n in N:
                go(T, K, n, which=which & V4)
        elif w == TILES:
            taken.add(out[:2])

    for T in [4, 13, 40, 64, 65, 100, 129, 150, 193, 257, 300, 361, 513, 641, 777, 1024, 1536, 4099]:
        for c in range(256, 5184, 64):
            for f in (4 * c, 7 * c // 128 * 64):
                for v4 in (V4, 0):
                    go(T, c, c, f, which=v4)
                    go(T, f, c, which=v4 + VALUE)
                    go(T, c, *(c,) * (3 if v4 else 4), which=v4)
                    go(T, c, c, which=v4)
    assert taken == {t[:2] for t, *_ in CASES} | {rk[1][:2] for rk, *_ in FFN if rk[0] == TILES}


@pytest.mark.parametrize("T,K,N", [(64, 64, (16,)), (64, 64, (32,)), (100, 128, (2048, 24))])  # one block of columns; not a multiple of 16
def test_what_is_not_of_this_form(T, K, N):
    assert tile(T, K, *N) == (0, 0, 0)


def coded(g, K, N):
    """codes over the whole range, scales of every size that occurs, some of them zero -> (weight, its binary16 image)"""
    h = lambda a: np.asarray(a, np.float32).astype(np.float16)
    q = g.integers(0, 256, (N, K), dtype=np.uint8)
    rx, ry = h(g.uniform(0.01, 0.3, N)), h(g.uniform(0.2, 1, K))
    rx[::7], ry[::5], rx[0] = 6e-8, 0, 0
    bufs = [dev(a) for a in (q, h(g.standard_normal(N) * 0.1), rx, h(g.standard_normal(K) * 0.01), ry)]
    w = fr.Weight(*[b.ptr for b in bufs], K, N, fr.U8)
    img = DevBuf.empty((N, K), np.float16)
    fr.check(L().frhip_dequant_u8(C.byref(w), img.ptr, None))
    return w, fr.Weight(img.ptr, None, None, None, None, K, N, fr.F16), bufs + [img]


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=lambda c: "%dx%d-%d-%d-%d" % (c[0][:2] + c[1:]))
def test_every_tile_gives_the_bits_of_the_image(case):
    _, T, K, N = case
    g = np.random.default_rng([T, K, N])
    x = dev(g.standard_normal((T, K)).astype(np.float16))
    w, image, keep = coded(g, K, N)
    got = []
    for v in (w, image):
        y = DevBuf.empty((T + 1, N), np.float32)
        y.upload(np.full((T + 1, N), 7.5, np.float32))
        fr.check(L().frhip_gemm(x.ptr, C.byref(v), y.ptr, T, fr.F32, None))
        got.append(y.numpy())
        assert (got[-1][T] == 7.5).all()
    assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32))
    xs, ws = x.numpy().astype(np.float64), keep[-1].numpy().astype(np.float64)
    assert (np.abs(got[0][:T] - xs @ ws.T) <= 2 * K * 2.0 ** -24 * (np.abs(xs) @ np.abs(ws).T) + 1e-30).all()


@pytest.mark.gpu
@pytest.mark.parametrize("act", [2, 3, 4])
def test_activations(act):
    g = np.random.default_rng(act)
    x = dev(g.standard_normal((530, 192)).astype(np.float16))
    w, image, keep = coded(g, 192, 1616)
    got = []
    for v in (w, image):
        y = DevBuf.empty((530, 1616), np.float16)
        fr.check(L().frhip_gemm_act(x.ptr, C.byref(v), y.ptr, 530, act, None))
        got.append(y.numpy())
    assert np.array_equal(got[0].view(np.uint16), got[1].view(np.uint16))


@pytest.mark.gpu
@pytest.mark.parametrize("T", [4, 17, 64, 65, 128, 129, 200, 300, 361, 513])
@pytest.mark.parametrize("C_,F_", [(320, 1088), (576, 2000 // 64 * 64), (1024, 3584)])
def test_ffn_in_slices_and_whole(T, C_, F_):
    """RWKV-5's operator, whose products keep the slices of the binary16 launches: a group, its members one by one, split or whole."""
    _ffn_gives_the_bits_of_the_images(T, C_, F_)


@pytest.mark.gpu
@pytest.mark.parametrize("T,C_,F_", [v[2:] for v in FFN])
def test_groups_on_wide_tiles_and_expanded_codes(T, C_, F_):
    """Two products on one launch of the wide tiles of 64 rows; codes expanded ahead of one product or of all."""
    _ffn_gives_the_bits_of_the_images(T, C_, F_)


def _ffn_gives_the_bits_of_the_images(T, C_, F_):
    g = np.random.default_rng([T, C_])
    h = lambda a: np.asarray(a, np.float32).astype(np.float16)
    vecs = [dev(a) for a in (h(g.standard_normal((T, C_)) * 2), h(g.standard_normal(C_)), h(1 + 0.1 * g.standard_normal(C_)),
                             h(0.1 * g.standard_normal(C_)), h(g.uniform(0, 1, C_)), h(g.uniform(0, 1, C_)))]
    pairs = [coded(g, *s) for s in ((C_, F_), (F_, C_), (C_, C_))]
    ws = DevBuf(L().frhip_seq_workspace_bytes(T, C_, F_))
    got = []
    for which in (0, 1):
        x_out, xx = DevBuf.empty((T, C_), np.float16), DevBuf.empty(C_, np.float16)
        fr.check(L().frhip_ffn_seq(T, C_, F_, *[b.ptr for b in vecs], *[C.byref(p[which]) for p in pairs], x_out.ptr, xx.ptr, 0, ws.ptr, None))
        got.append(x_out.numpy().view(np.uint16))
    assert np.array_equal(*got)
