"""Binary16 products with four loading waves: every tile, with remainders in rows, columns and K-steps, whole and in slices of K."""
import ctypes as C

import numpy as np
import pytest

from hipref import DevBuf, L, dev, fr, make_weight


def tile(T, K, *N, slices=1):
    out = (C.c_int * 4)()
    fr.check(L().frhip_gemm_ring_tile(T, K, len(N), (C.c_int * len(N))(*N), slices, 256, out))
    return tuple(out)


def few(T, K, N):
    out = (C.c_int * 2)()
    fr.check(L().frhip_gemm_few_tile(T, K, 1, (C.c_int * 1)(N), 256, out))
    return out[0] != 0


# one to seven K-steps (the ring holds three or four), and not the kernel for a few rows
CASES = [((64, 1), 513, 64, 20), ((64, 2), 577, 128, 1085), ((64, 3), 513, 256, 2672), ((64, 4), 1000, 192, 2048), ((64, 5), 513, 320, 3792),
         ((64, 6), 529, 384, 5040), ((128, 3), 513, 128, 4624), ((128, 4), 520, 192, 5450), ((128, 5), 700, 384, 6416), ((128, 6), 641, 448, 8000),
         ((128, 7), 600, 192, 10600), ((128, 8), 513, 448, 12000), ((128, 8), 1537, 128, 9408), ((64, 7), 129, 64, 16421), ((64, 8), 129, 192, 20565),
         ((128, 2), 321, 192, 5429)]


def test_cases_reach_their_tiles():
    assert [tile(T, K, N)[:2] for _, T, K, N in CASES] == [t for t, *_ in CASES]
    assert all(tile(T, K, N)[3] for _, T, K, N in CASES) and not any(few(T, K, N) for _, T, K, N in CASES)


def test_every_tile_that_launches_of_the_operators_take_is_among_the_cases():
    """Rows of tiles and widths over models of 256 to 5120 channels; a wave's part of a tile follows from the two."""
    taken = set()

    def go(T, K, *N, which):
        out = (C.c_int * 2)()
        form = L().frhip_seq_gemm_form(T, K, len(N), (C.c_int * len(N))(*N), which, 256, out)
        if form == 3:  # one by one
            for n in N:
                go(T, K, n, which=which & 1)
        elif form != 1:  # not the kernel for a few rows
            t = tile(T, K, *N, slices=out[0] if form == 2 else 1)
            if form == 2 or t[3]:
                taken.add(t[:2])

    for T in [4, 13, 40, 64, 65, 100, 129, 150, 193, 257, 300, 361, 513, 641, 777, 1024, 1536, 4099]:
        for c in range(256, 5184, 64):
            for f in (4 * c, 7 * c // 128 * 64):
                for v4 in (1, 0):
                    go(T, c, c, f, which=v4)
                    go(T, f, c, which=v4 + 2)
                    go(T, c, *(c,) * (3 if v4 else 4), which=v4)
                    go(T, c, c, which=v4)
    assert taken == {t for t, *_ in CASES}


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=lambda c: "%dx%d-%d-%d-%d" % (c[0] + c[1:]))
def test_every_tile_against_float64(case):
    """fp32 sums of exact products in any order: |error| <= K 2^-24 sum |x w|, twice that for the unit's own rounding of its inner
    sums; binary16 outputs are the fp32 ones rounded; a row with an infinity leaves the others alone; nothing past the end is written."""
    _, T, K, N = case
    g = np.random.default_rng([T, K, N])
    x, w = g.standard_normal((T, K)).astype(np.float16), (g.standard_normal((K, N)) * 0.3).astype(np.float16)
    pw, _ = make_weight(w, False)
    xd = dev(x)

    def run(dt):
        y = DevBuf.empty((T * N + 16,), dt)
        y.upload(np.full(T * N + 16, 7.5, dt))
        fr.check(L().frhip_gemm(xd.ptr, pw.ref, y.ptr, T, fr.F32 if dt is np.float32 else fr.F16, None))
        got = y.numpy()
        assert (got[T * N:] == 7.5).all()
        return got[:T * N].reshape(T, N)

    y = run(np.float32)
    x64, w64 = x.astype(np.float64), w.astype(np.float64)
    assert (np.abs(y - x64 @ w64) <= 2 * K * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64)) + 1e-30).all()
    assert np.array_equal(run(np.float16), y.astype(np.float16))
    x[T - 1, K // 2] = np.inf
    xd = dev(x)
    inf = run(np.float32)
    assert np.array_equal(inf[:T - 1].view(np.uint32), y[:T - 1].view(np.uint32)) and not np.isfinite(inf[T - 1]).any()


@pytest.mark.gpu
@pytest.mark.parametrize("T", [4, 33, 64, 65, 129, 200, 360, 361])
@pytest.mark.parametrize("C_,F_", [(320, 1088), (576, 4160), (1024, 3584)])
def test_rwkv5_ffn_in_slices_and_whole(T, C_, F_):
    """Every row of a prompt is that of a longer prompt whose products are cut otherwise, within the rounding of the fp32 sums."""
    g = np.random.default_rng([T, C_])
    h = lambda a: np.asarray(a, np.float32).astype(np.float16)
    n = 520
    x = h(g.standard_normal((n, C_)) * 2)
    vecs = [dev(a) for a in (h(g.standard_normal(C_)), h(1 + 0.1 * g.standard_normal(C_)), h(0.1 * g.standard_normal(C_)),
                             h(g.uniform(0, 1, C_)), h(g.uniform(0, 1, C_)))]
    ws = [make_weight(h(g.standard_normal(s) * 0.02), False)[0] for s in ((C_, F_), (F_, C_), (C_, C_))]
    got = []
    for t in (T, n):
        xd, x_out, xx = dev(x[:t]), DevBuf.empty((t, C_), np.float16), DevBuf.empty(C_, np.float16)
        space = DevBuf(L().frhip_seq_workspace_bytes(t, C_, F_))
        fr.check(L().frhip_ffn_seq(t, C_, F_, xd.ptr, *[v.ptr for v in vecs], *[w.ref for w in ws], x_out.ptr, xx.ptr, 0, space.ptr, None))
        got.append(x_out.numpy()[:T].astype(np.float64))
    # one spacing of binary16 at most, and where sums of another order round the other way (relu^2 of a rounded key passes it on)
    scale = np.maximum(np.abs(got[1]), np.sqrt((got[1] ** 2).mean()))
    assert (np.abs(got[0] - got[1]) <= 3 * 2.0 ** -10 * scale).all()
