"""Products of a few rows in one launch (K split over the waves of a workgroup): every tile that is built, at sizes with a
remainder in rows, columns and K-steps, against float64."""
import ctypes as C

import numpy as np
import pytest

import pyoracle as po
from hipref import DevBuf, L, assert_close_f16, dev, fr, make_weight


def tile(T, K, *N):
    out = (C.c_int * 2)()
    fr.check(L().frhip_gemm_few_tile(T, K, len(N), (C.c_int * len(N))(*N), 256, out))
    return tuple(out)


CASES = [((1, 1), 1, 64, 32), ((1, 1), 13, 576, 1856), ((1, 2), 1, 64, 4112), ((1, 3), 1, 64, 8208), ((1, 4), 1, 64, 12336),
         ((2, 1), 17, 64, 2064), ((2, 2), 17, 64, 6160), ((2, 3), 17, 64, 8256), ((2, 4), 65, 192, 4192), ((3, 1), 33, 64, 2752),
         ((3, 2), 33, 64, 5456), ((3, 3), 300, 192, 1648), ((3, 4), 129, 448, 4128), ((3, 5), 161, 704, 4112), ((4, 2), 300, 128, 1232),
         ((4, 3), 110, 384, 4144), ((4, 4), 161, 704, 4368), ((5, 2), 150, 256, 3280), ((5, 3), 150, 576, 4144), ((5, 4), 200, 960, 4160),
         ((5, 5), 300, 1600, 4128), ((6, 4), 270, 2048, 4112)]


def test_cases_reach_every_tile():
    assert [tile(T, K, N) for _, T, K, N in CASES] == [t for t, *_ in CASES]
    assert len({t for t, *_ in CASES}) == 21


@pytest.mark.parametrize("T,K,N", [(256, 5120, (5120, 20480)),  # 91 us on planned tiles, 143 in one launch of this form
                                   (513, 64, (64,)), (13, 2048, (2048, 2040))])  # too many rows; not a multiple of 16 columns
def test_other_forms_keep_what_is_theirs(T, K, N):
    assert tile(T, K, *N) == (0, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=lambda c: "%dx%d-%d-%d-%d" % (c[0] + c[1:]))
def test_every_tile_against_float64(case):
    """fp32 sums of exact products in any order: |error| <= K 2^-24 sum |x w|, twice that for the unit's own rounding of its
    inner sums.  A uint8 weight gives the bits of its binary16 image; a row with an infinity leaves the others alone."""
    _, T, K, N = case
    g = np.random.default_rng(100000 * T + K + N)
    x = g.standard_normal((T, K)).astype(np.float16)
    coded, wref = make_weight((g.standard_normal((K, N)) * 0.02).astype(np.float16), True)
    img = DevBuf.empty((N, K), np.float16)
    fr.check(L().frhip_dequant_u8(coded.ref, img.ptr, None))
    image = fr.Weight(img.ptr, None, None, None, None, K, N, fr.F16)
    w = img.numpy().T.astype(np.float64)
    ref, size = x.astype(np.float64) @ w, np.abs(x).astype(np.float64) @ np.abs(w)
    xd, y = dev(x), DevBuf.empty((T, N), np.float32)
    fr.check(L().frhip_gemm(xd.ptr, C.byref(image), y.ptr, T, fr.F32, None))
    plain = y.numpy()
    assert (np.abs(plain - ref) <= 2 * K * 2.0 ** -24 * size + 1e-30).all()
    fr.check(L().frhip_gemm(xd.ptr, coded.ref, y.ptr, T, fr.F32, None))
    assert np.array_equal(y.numpy().view(np.uint32), plain.view(np.uint32))
    x[0, K // 2] = np.inf
    xd = dev(x)
    fr.check(L().frhip_gemm(xd.ptr, coded.ref, y.ptr, T, fr.F32, None))
    got = y.numpy()
    assert np.array_equal(got[1:].view(np.uint32), plain[1:].view(np.uint32)) and not np.isfinite(got[0]).any()


@pytest.mark.gpu
@pytest.mark.parametrize("T,K,N", [(5, 128, 96), (40, 320, 3008), (77, 448, 6160)])
def test_activations_of_few_rows(T, K, N):
    """sigmoid, relu^2 and silu are those of the stored binary16 product, bit for bit (the formulas in float64)."""
    assert tile(T, K, N) != (0, 0)
    g = np.random.default_rng(T)
    x, w = g.standard_normal((T, K)).astype(np.float16), g.standard_normal((K, N)).astype(np.float16)
    pw, _ = make_weight((w * 0.3).astype(np.float16), False)
    xd, y = dev(x), DevBuf.empty((T, N), np.float16)
    fr.check(L().frhip_gemm(xd.ptr, pw.ref, y.ptr, T, fr.F16, None))
    p = y.numpy()
    e = np.exp(-p.astype(np.float64))
    with np.errstate(over="ignore"):
        h = np.exp(-p.astype(np.float32)).astype(np.float16)
        want = {2: (1 / (1 + e)).astype(np.float32).astype(np.float16),
                3: np.where(p > 0, p * p, np.float16(0)).astype(np.float16),
                4: (p.astype(np.float32) / (np.float16(1) + h).astype(np.float32)).astype(np.float16)}
    for act, ref in want.items():
        fr.check(L().frhip_gemm_act(xd.ptr, pw.ref, y.ptr, T, act, None))
        got = y.numpy()
        if act == 4:  # numpy's expf and the device's may round the binary16 exponential the other way at a tie
            d = np.abs(got.view(np.int16).astype(int) - ref.view(np.int16).astype(int))
            assert d.max() <= 2 and (d != 0).mean() < 1e-3
        else:
            assert np.array_equal(got, ref)


def form(T, K, *N, value=False):
    """-> (form, blocks of 16 rows, blocks of 16 columns) of a launch of frhip_ffn_seq_v4"""
    out = (C.c_int * 2)()
    return L().frhip_seq_gemm_form(T, K, len(N), (C.c_int * len(N))(*N), 1 + 2 * value, 256, out), out[0], out[1]


@pytest.mark.gpu
@pytest.mark.parametrize("quant", [False, True])
@pytest.mark.parametrize("T,C_,F_,rk,v", [(1, 512, 1024, (1, 1, 1), (1, 1, 1)), (13, 576, 1856, (1, 1, 1), (1, 1, 1)),
                                          (16, 2048, 8192, (1, 1, 3), (1, 1, 1)),    # 2048 and 8192 are no multiples of 48
                                          (65, 768, 3072, (1, 3, 2), (1, 1, 1)), (200, 768, 3072, (1, 5, 3), (1, 3, 1)),
                                          (129, 512, 1792, (1, 3, 2), (1, 2, 1)),
                                          (361, 768, 3072, (0, 0, 0), (1, 3, 2)), (512, 576, 1856, (0, 0, 0), (1, 3, 2))])  # the group on tiles
def test_ffn_of_few_rows(T, C_, F_, rk, v, quant):
    """Groups (sigmoid and relu^2) and ffn's last epilogue, with rows past the end and tiles past a product's columns.
    Bounds as for frhip_ffn_seq; halved outputs are the halves of the others, uint8 codes give the bits of their binary16 image."""
    assert form(T, C_, C_, F_) == rk and form(T, F_, C_, value=True) == v
    g = np.random.default_rng([T, C_])
    h = lambda a: np.asarray(a, np.float32).astype(np.float16)
    vecs = [h(g.standard_normal((T, C_)) * 2), h(g.standard_normal(C_)), h(1 + 0.1 * g.standard_normal(C_)), h(0.1 * g.standard_normal(C_)),
            h(g.uniform(0, 1, C_)), h(g.uniform(0, 1, C_))]
    (kw, kref), (vw, vref), (rw, rref) = (make_weight(h(g.standard_normal(s) * 0.02), quant) for s in ((C_, F_), (F_, C_), (C_, C_)))
    want, xx = po.ffn_f16(*vecs, kref, vref, rref)
    bufs, ws = [dev(a) for a in vecs], DevBuf(L().frhip_seq_workspace_bytes(T, C_, F_))

    def run(weights, div2=0):
        x_out, xx_out = DevBuf.empty((T + 1, C_), np.float16), DevBuf.empty(C_, np.float16)
        x_out.upload(np.full((T + 1, C_), 7.5, np.float16))
        fr.check(L().frhip_ffn_seq_v4(T, C_, F_, *[b.ptr for b in bufs], *weights, x_out.ptr, xx_out.ptr, div2, ws.ptr, None))
        assert (x_out.numpy()[T] == 7.5).all()
        assert_close_f16(xx_out.numpy(), xx, max_ulp=1, what="xx_last")
        return x_out.numpy()[:T]

    refs = [w.ref for w in (kw, vw, rw)]
    got = run(refs)
    assert_close_f16(got, want.reshape(got.shape), max_ulp=3, max_frac=0.2, what="x_out", floor_rms=1.0)
    assert np.array_equal(run(refs, 1), got / np.float16(2))
    if quant:
        images = []
        for w in (kw, vw, rw):
            img = DevBuf.empty((w.N, w.K), np.float16)
            fr.check(L().frhip_dequant_u8(w.ref, img.ptr, None))
            images.append((img, fr.Weight(img.ptr, None, None, None, None, w.K, w.N, fr.F16)))
        assert np.array_equal(run([C.byref(w) for _, w in images]).view(np.uint16), got.view(np.uint16))
