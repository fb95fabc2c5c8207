"""GPU parity tests of the seq-mode (prompt) operators against the oracle."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import pyoracle as po
from hipref import DevBuf, L, assert_close_f16, dev, fr, make_weight

_alive = []


def keep(a):
    b = dev(a)
    _alive.append(b)
    if len(_alive) > 96:
        fr.check(L().frhip_device_sync())
        del _alive[:48]
    return b


rng = np.random.default_rng(777)


@pytest.fixture(autouse=True)
def _rng_per_test(request):
    """Every test draws from a generator seeded by its own name, so its data do not depend on which
    other tests ran before it (or on cases added to them)."""
    import zlib
    global rng
    rng = np.random.default_rng([777, zlib.crc32(request.node.name.encode())])


def _routes(T, K, *N):
    """frhip_gemm_route on 256 compute units -> launches, [(rows of a tile, widest tile in blocks of 32 columns, rounds, loading waves)]"""
    out = (C.c_int * (4 * len(N)))()
    launches = L().frhip_gemm_route(T, K, len(N), (C.c_int * len(N))(*N), 256, out)
    return launches, [tuple(out[4 * i:4 * i + 4]) for i in range(len(N))]


def h(x):
    return np.asarray(x, np.float32).astype(np.float16)


@pytest.mark.parametrize("T,K,N", [(1024, 2048, 2048), (512, 2560, 8960), (100, 8192, 2048), (1, 64, 128), (130, 128, 200), (7, 1792, 512),
                                   # wide enough for the variable-width tiles: ragged N (last block partial), ragged T
                                   (1024, 256, 7000), (900, 128, 6144),
                                   # one round of 256-row tiles beats two of 128-row tiles: with a loader wave (whole tiles) and without
                                   (1024, 128, 10240), (1000, 128, 10000)])
@pytest.mark.parametrize("quant", [False, True])
def test_gemm_against_oracle(T, K, N, quant):
    x = h(rng.standard_normal((T, K)))
    w = h(rng.standard_normal((K, N)) * 0.02)
    pw, wref = make_weight(w, quant)
    ref = po.gemm_f16(x, wref, "f32")
    y32, y16 = DevBuf.empty((T, N), np.float32), DevBuf.empty((T, N), np.float16)
    fr.check(L().frhip_gemm(keep(x).ptr, pw.ref, y32.ptr, T, fr.F32, None))
    fr.check(L().frhip_gemm(keep(x).ptr, pw.ref, y16.ptr, T, fr.F16, None))
    got = y32.numpy()
    tol = 3e-6 * np.sqrt(K) * np.abs(ref).max() + 1e-5
    assert np.abs(got - ref).max() <= tol, np.abs(got - ref).max()
    assert_close_f16(y16.numpy(), ref.astype(np.float16), max_ulp=1, what="gemm f16 out")
    # an asymmetric probe: row t = e_k picks out row k of the weight exactly (catches a swapped
    # operand or a wrong fragment layout that a random comparison could only show as noise)
    if T >= 4:
        e = np.zeros((T, K), np.float16)
        ks = [0, 1, K // 2 + 3, K - 1]
        for t, k in enumerate(ks):
            e[t, k] = 1
        fr.check(L().frhip_gemm(keep(e).ptr, pw.ref, y32.ptr, T, fr.F32, None))
        out = y32.numpy()
        for t, k in enumerate(ks):
            assert np.array_equal(out[t], wref[k].astype(np.float32)), (t, k)
        assert not out[len(ks):].any()


@pytest.mark.parametrize("T,K,N", [(2048, 64, 8192),    # 256 x 256 tiles, two stages, a single K-step
                                   (2048, 128, 6100),   # 256 x 192, two K-steps, ragged columns
                                   (4099, 192, 2048),   # 256 x 160 / 128; the last strip has three rows
                                   (1024, 192, 10240),  # 256 x 160, whole tiles: the loader wave's form, three stages
                                   (1025, 320, 10000),  # one row in the last strip, ragged columns
                                   (512, 192, 6144),    # 128 x 96: the narrowest planned tile
                                   (3000, 128, 10240)]) # more than four rounds' worth of 128 x 128 tiles
def test_gemm_planned_tiles_against_oracle(T, K, N):
    """Tile heights, widths, stage counts and edges of the planned binary16 launches.  Both sides add K exact products
    in fp32, in another order: K 2^-24 of the sum of the magnitudes at most, which 3e-6 sqrt(K) max|y| covers here."""
    x = h(rng.standard_normal((T, K)))
    w = h(rng.standard_normal((K, N)) * 0.02)
    pw, wref = make_weight(w, False)
    ref = po.gemm_f16(x, wref, "f32")
    y = DevBuf.empty((T, N), np.float32)
    fr.check(L().frhip_gemm(keep(x).ptr, pw.ref, y.ptr, T, fr.F32, None))
    assert np.abs(y.numpy() - ref).max() <= 3e-6 * np.sqrt(K) * np.abs(ref).max() + 1e-5


@pytest.mark.parametrize("T,N,shift", [(300, 16384, 0), (257, 16376, 0), (300, 16377, 0), (385, 16384, 4), (513, 16377, 0), (769, 16348, 0),
                                       (1000, 16384, 2)])
def test_tiles_over_the_edge_give_the_bits_of_whole_ones(T, N, shift):
    """Rows and columns that end inside a tile of 128 or 256 rows, outputs at any address (`shift` bytes past a multiple of 16),
    against the same outputs of a product of whole tiles; nothing is written beside them."""
    K, M, W = 192, 1024, 16384
    x, w = h(rng.standard_normal((M, K))), h(rng.standard_normal((K, W)) * 0.3)
    xd, whole, part = keep(x), make_weight(w, False)[0], make_weight(np.ascontiguousarray(w[:, :N]), False)[0]
    tile = (C.c_int * 2)()
    fr.check(L().frhip_gemm_few_tile(T, K, 1, (C.c_int * 1)(N), 256, tile))
    assert _routes(T, K, N)[1][0][0] in (128, 256) and tuple(tile) == (0, 0)

    def run(pw, T, N, shift, dt, act):
        lead = shift // dt().itemsize
        y = keep(np.full(lead + T * N + 16, 7.5, dt))
        if act:
            fr.check(L().frhip_gemm_act(xd.ptr, pw.ref, y.ptr + shift, T, act, None))
        else:
            fr.check(L().frhip_gemm(xd.ptr, pw.ref, y.ptr + shift, T, fr.F32 if dt is np.float32 else fr.F16, None))
        got = y.numpy()
        assert (got[:lead] == 7.5).all() and (got[lead + T * N:] == 7.5).all()
        return got[lead:lead + T * N].reshape(T, N)

    for dt, act in ((np.float32, 0), (np.float16, 0), (np.float16, 2), (np.float16, 3), (np.float16, 4)):
        want = np.ascontiguousarray(run(whole, M, W, 0, dt, act)[:T, :N])
        assert np.array_equal(np.ascontiguousarray(run(part, T, N, shift - shift % dt().itemsize, dt, act)).view(np.uint8), want.view(np.uint8))


def test_gemm_sigmoid_and_silu_epilogues_every_binary16_bit_exact():
    """Every finite binary16 value goes through the product's sigmoid epilogue (identity weight, so the
    accumulator is the input exactly) and must come out as the oracle's double-evaluated sigmoid (and its silu), bit for bit;
    once on 64-row tiles (T = 1024, N = 64) and once on the variable-width tiles (N = 8192, columns repeat)."""
    bits = np.arange(65536, dtype=np.uint16)
    x = bits.view(np.float16).copy()
    x[~np.isfinite(x)] = 0
    x[bits == 0x8000] = 0  # the accumulator of 0 + (-0)(1) is +0: -0 cannot reach the epilogue this way
    a = x.reshape(1024, 64)
    want = po.sigmoid_f16(a)
    want_silu = po.silu_f16(a)
    for N in (64, 8192):
        w = np.zeros((64, N), np.float16)
        w[np.arange(N) % 64, np.arange(N)] = 1
        pw = fr.PackedWeight(w_kn=w)
        y = DevBuf.empty((1024, N), np.float16)
        for act, ref in ((2, want), (4, want_silu)):  # FRHIP_ACT_SIGMOID, FRHIP_ACT_SILU
            fr.check(L().frhip_gemm_act(keep(a).ptr, pw.ref, y.ptr, 1024, act, None))
            got = y.numpy()
            for c0 in range(0, N, 64):
                assert np.array_equal(got[:, c0:c0 + 64].view(np.uint16), ref.view(np.uint16)), (act, c0)


def test_gemm_act_relu2_and_silu_match_the_oracle():
    x = h(rng.standard_normal((256, 128)))
    w = h(rng.standard_normal((128, 192)) * 0.1)
    pw = fr.PackedWeight(w_kn=w)
    lin = po.gemm_f16(x, w, "f16")
    y = DevBuf.empty((256, 192), np.float16)
    fr.check(L().frhip_gemm_act(keep(x).ptr, pw.ref, y.ptr, 256, 3, None))
    t = lin.astype(np.float16)
    assert_close_f16(y.numpy(), np.where(t > 0, t * t, np.float16(0)).astype(np.float16), max_ulp=4, max_frac=0.05, what="relu2")  # one spacing of t is two of t*t
    assert L().frhip_gemm_act(keep(x).ptr, pw.ref, y.ptr, 256, 7, None) == -1


@pytest.mark.parametrize("act", [2, 4])  # FRHIP_ACT_SIGMOID, FRHIP_ACT_SILU
def test_rows_past_the_end_do_not_slow_an_epilogue(act):
    """777 and 1024 rows are the same four strips of 256-row tiles, the last one with 9 or 256 rows.  The elements that
    are not stored, copies of the last row, may not be worked off one by one (that took half as long again and more)."""
    assert _routes(777, 2048, 10240)[1][0][:3] == _routes(1024, 2048, 10240)[1][0][:3] == (256, 5, 1)
    x, pw = keep(h(rng.standard_normal((1024, 2048)))), fr.PackedWeight(w_kn=h(rng.standard_normal((2048, 10240)) * 0.02))
    y = DevBuf.empty((1024, 10240), np.float16)
    events = [C.c_void_p() for _ in range(2)]
    for e in events:
        fr.check(L().frhip_event_create(C.byref(e)))
    best = {777: 1e9, 1024: 1e9}
    for _ in range(12):
        for T in best:
            ms = C.c_float()
            fr.check(L().frhip_event_record(events[0], None))
            for _ in range(4):
                fr.check(L().frhip_gemm_act(x.ptr, pw.ref, y.ptr, T, act, None))
            fr.check(L().frhip_event_record(events[1], None))
            fr.check(L().frhip_event_sync(events[1]))
            fr.check(L().frhip_event_elapsed_ms(*events, C.byref(ms)))
            best[T] = min(best[T], ms.value)
    for e in events:
        fr.check(L().frhip_event_destroy(e))
    assert best[777] <= 1.2 * best[1024], best


@pytest.mark.parametrize("T,K,N,most", [(384, 768, 50277, 1.25), (777, 768, 50277, 1.25),  # tiles of 128 rows; of 256, the last ones over the edge
                                        (1024, 192, 16377, 1.6)])
def test_rows_at_any_address_do_not_slow_an_epilogue(T, K, N, most):
    """50277 outputs a row (the vocabulary of the 169M model) begin at any even address; 50280 at multiples of 16 bytes.  The bounds are between
    what was measured: 1.0 times as long, 1.2 to 1.27 the small one; 1.40, 1.46 and 1.95 where such rows went out one element a lane and instruction."""
    more = -(-N // 8) * 8
    x, w = keep(h(rng.standard_normal((T, K)))), h(rng.standard_normal((K, more)) * 0.02)
    pw = {n: fr.PackedWeight(w_kn=np.ascontiguousarray(w[:, :n])) for n in (N, more)}
    y = DevBuf.empty((T, more), np.float16)
    events = [C.c_void_p() for _ in range(2)]
    for e in events:
        fr.check(L().frhip_event_create(C.byref(e)))
    best = {N: 1e9, more: 1e9}
    for _ in range(12):
        for n in best:
            ms = C.c_float()
            fr.check(L().frhip_event_record(events[0], None))
            for _ in range(4):
                fr.check(L().frhip_gemm(x.ptr, pw[n].ref, y.ptr, T, fr.F16, None))
            fr.check(L().frhip_event_record(events[1], None))
            fr.check(L().frhip_event_sync(events[1]))
            fr.check(L().frhip_event_elapsed_ms(*events, C.byref(ms)))
            best[n] = min(best[n], ms.value)
    for e in events:
        fr.check(L().frhip_event_destroy(e))
    print(best)
    assert best[N] <= most * best[more], best


def test_gemm_rejects_bad_shapes():
    w = fr.PackedWeight(w_kn=h(rng.standard_normal((96, 64))))
    y = DevBuf.empty((4, 64), np.float32)
    assert L().frhip_gemm(keep(h(np.zeros((4, 96)))).ptr, w.ref, y.ptr, 4, fr.F32, None) == -2  # K % 64
    assert L().frhip_gemm(None, w.ref, y.ptr, 4, fr.F32, None) == -1


def _common(C_):
    return (h(1 + 0.1 * rng.standard_normal(C_)), h(0.1 * rng.standard_normal(C_)))


# (1024, 2048, 8192): r and k as one round of 256-row tiles, the value product split over K in two slices;
# (300, 2048, 8192): the value product in four slices over ragged row tiles; (512, 2560, 8960): three slices of 47, 47 and 46 K-steps
# (16, 2048, 8192), (130, 2048, 8192), (200, 2560, 8960): short prompts at full width -- products split over K across the idle compute
# units: r,k grouped in one split launch (16 rows), product by product because the group is too wide (130 rows) or on planned
# tiles (200 rows), the value product in 16, five and three slices (test_seq_gemm_form.py holds these to it)
@pytest.mark.parametrize("T,C_,F_", [(64, 512, 1792), (300, 2048, 8192), (1024, 2048, 8192), (512, 2560, 8960), (1, 512, 1024), (33, 768, 3072), (3000, 512, 1792),
                                     (16, 2048, 8192), (130, 2048, 8192), (200, 2560, 8960)])
@pytest.mark.parametrize("quant", [False, True])
def test_ffn_seq(T, C_, F_, quant):
    g = np.random.default_rng(5000 + T) if T >= 512 else rng  # the full-size cases draw from a stream of their own
    x, sx = h(g.standard_normal((T, C_)) * 2), h(g.standard_normal(C_))
    ln_w, ln_b = h(1 + 0.1 * g.standard_normal(C_)), h(0.1 * g.standard_normal(C_))
    mk, mr = h(g.uniform(0, 1, C_)), h(g.uniform(0, 1, C_))
    kw, kref = make_weight(h(g.standard_normal((C_, F_)) * 0.02), quant)
    vw, vref = make_weight(h(g.standard_normal((F_, C_)) * 0.02), quant)
    rw, rref = make_weight(h(g.standard_normal((C_, C_)) * 0.02), quant)
    ref_x, ref_xx = po.ffn_f16(x, sx, ln_w, ln_b, mk, mr, kref, vref, rref)
    x_out, xx_out = DevBuf.empty((T, C_), np.float16), DevBuf.empty(C_, np.float16)
    ws = DevBuf(L().frhip_seq_workspace_bytes(T, C_, F_))
    fr.check(L().frhip_ffn_seq(T, C_, F_, keep(x).ptr, keep(sx).ptr, keep(ln_w).ptr, keep(ln_b).ptr, keep(mk).ptr,
                               keep(mr).ptr, kw.ref, vw.ref, rw.ref, x_out.ptr, xx_out.ptr, 0, ws.ptr, None))
    assert_close_f16(xx_out.numpy(), ref_xx, max_ulp=1, what="xx_last")
    assert_close_f16(x_out.numpy(), ref_x, max_ulp=3, max_frac=0.2, what="x_out", floor_rms=1.0)


@pytest.mark.parametrize("T,C_,F_,rk,v", [
    # every product on 256-row tiles whose last strip has 16 rows: sigmoid, relu^2 and the output's epilogue, predicated
    (16400, 320, 256, (1, [(256, 8, 1, 0)] * 2), (256, 4, 1, 0)),
    (2049, 1024, 4096, (1, [(256, 6, 1, 0)] * 2), None),  # ... one row in the last strip, 16 K-steps
    (1472, 768, 10752, (2, [(64, 3, 1, 1), (256, 8, 1, 0)]), None),  # r and k one by one, on tiles of different heights
    (8448, 640, 1280, (1, [(256, 4, 2, 1)] * 2), (256, 3, 1, 1))])  # whole tiles: the loader wave's form, grouped and alone
def test_ffn_seq_on_planned_tiles(T, C_, F_, rk, v):
    """The fused epilogues on 256-row tiles, with rows past the end and without, in groups and one by one.  Bounds as in
    test_ffn_seq."""
    assert _routes(T, C_, C_, F_) == rk
    assert v is None or _routes(T, F_, C_)[1] == [v]
    test_ffn_seq(T, C_, F_, False)


@pytest.mark.parametrize("T,C_,F_", [(4, 512, 1792), (64, 512, 2048), (65, 768, 3072), (128, 2048, 8192), (129, 512, 1792)])
def test_ffn_seq_uint8_dequantised_in_the_product(T, C_, F_):
    """uint8 weights of RWKV-5's operator, up to 129 rows: in slices of K and whole, a group on one launch and its members one by one.
    Bounds as in test_ffn_seq."""
    test_ffn_seq(T, C_, F_, True)


# (576, 1856): ragged tiles; (2560, 8960): r,k of 13 rows in two slices of 20 K-steps, the value product in twelve of 11 or 12
@pytest.mark.parametrize("T", [4, 13, 63, 64, 65, 129])
@pytest.mark.parametrize("C_,F_", [(576, 1856), (2560, 8960)])
def test_ffn_seq_uint8_gives_the_bits_of_its_binary16_image(T, C_, F_):
    """A uint8 weight, whose codes these products dequantise on their way into LDS, and its dequantised image as a binary16 weight: the
    same slices of K, so the same bits.  (Codes expanded ahead of the product: test_gpu_gemm_q8.py.)"""
    x, sx = h(rng.standard_normal((T, C_)) * 2), h(rng.standard_normal(C_))
    vecs = [keep(a) for a in (x, sx, *_common(C_), h(rng.uniform(0, 1, C_)), h(rng.uniform(0, 1, C_)))]
    coded = [make_weight(h(rng.standard_normal(s) * 0.02), True)[0] for s in ((C_, F_), (F_, C_), (C_, C_))]
    images = []
    for w in coded:
        img = DevBuf.empty((w.N, w.K), np.float16)
        _alive.append(img)
        fr.check(L().frhip_dequant_u8(w.ref, img.ptr, None))
        images.append(fr.Weight(img.ptr, None, None, None, None, w.K, w.N, fr.F16))
    outs = []
    for kw, vw, rw in ([w.ref for w in coded], [C.byref(w) for w in images]):
        x_out, xx_out, ws = DevBuf.empty((T, C_), np.float16), DevBuf.empty(C_, np.float16), DevBuf(L().frhip_seq_workspace_bytes(T, C_, F_))
        fr.check(L().frhip_ffn_seq(T, C_, F_, *[a.ptr for a in vecs], kw, vw, rw, x_out.ptr, xx_out.ptr, 0, ws.ptr, None))
        outs.append(x_out.numpy())
    assert np.array_equal(outs[0].view(np.uint16), outs[1].view(np.uint16))


# Of the value product: slices of K, the tile of the whole binary16 product, and that of the codes (0: expanded ahead of it)
@pytest.mark.parametrize("T,C_,F_,slices,tile,coded", [
    (13, 512, 1792, 7, None, 64), (129, 576, 1856, 7, None, 64),     # the reduction launch
    (700, 1024, 256, 0, (64, 2), 64), (777, 3072, 128, 0, (128, 3), 128),  # the last strip over the edge
    (16400, 320, 256, 0, (256, 4), 0), (8448, 640, 1280, 0, (256, 3), 0)])  # tiles of 256 rows, over the edge and whole
@pytest.mark.parametrize("quant", [False, True])
def test_ffn_seq_rows_at_any_address(T, C_, F_, slices, tile, coded, quant):
    """The residual epilogue reads x and writes x_out wherever they begin (2 and 6 bytes past a multiple of 16): the bits of aligned ones."""
    out = (C.c_int * 3)()
    assert L().frhip_seq_gemm_form(T, F_, 1, (C.c_int * 1)(C_), 2, 256, out) == (2 if slices else 0) and out[0] == slices
    assert slices or _routes(T, F_, C_)[1][0][:2] == tile
    assert L().frhip_seq_codes_way(T, F_, 1, (C.c_int * 1)(C_), 2, 256, out) == (1 if coded else 0) and out[0] == coded
    g = np.random.default_rng([T, C_])
    x = h(g.standard_normal((T, C_)) * 2)
    vecs = [keep(v) for v in (h(g.standard_normal(C_)), h(1 + 0.1 * g.standard_normal(C_)), h(0.1 * g.standard_normal(C_)), h(g.uniform(0, 1, C_)), h(g.uniform(0, 1, C_)))]
    kw, vw, rw = [make_weight(h(g.standard_normal(s) * 0.02), quant)[0] for s in ((C_, F_), (F_, C_), (C_, C_))]
    outs = []
    for at_x, at_out in ((0, 0), (1, 3)):  # elements
        xs = keep(np.concatenate([np.zeros(at_x, np.float16), x.reshape(-1)]))
        out, xx, ws = DevBuf.empty(T * C_ + 8, np.float16), DevBuf.empty(C_, np.float16), DevBuf(L().frhip_seq_workspace_bytes(T, C_, F_))
        fr.check(L().frhip_ffn_seq(T, C_, F_, xs.ptr + 2 * at_x, *[v.ptr for v in vecs], kw.ref, vw.ref, rw.ref, out.ptr + 2 * at_out, xx.ptr, 0, ws.ptr, None))
        outs.append((out.numpy()[at_out:at_out + T * C_].view(np.uint16), xx.numpy().view(np.uint16)))
    assert all(np.array_equal(a, b) for a, b in zip(*outs))


@pytest.mark.parametrize("T", [4, 13, 64, 65])
def test_ffn_seq_uint8_scales_at_any_address(T):
    """Row scales and codes that do not start at a multiple of 16 bytes are taken, with the same bits."""
    C_, F_ = 512, 1792
    x, sx = h(rng.standard_normal((T, C_)) * 2), h(rng.standard_normal(C_))
    vecs = [keep(v) for v in (x, sx, h(1 + 0.1 * rng.standard_normal(C_)), h(0.1 * rng.standard_normal(C_)), h(rng.uniform(0, 1, C_)), h(rng.uniform(0, 1, C_)))]
    weights = [make_weight(h(rng.standard_normal(s) * 0.02), True)[0] for s in ((C_, F_), (F_, C_), (C_, C_))]
    moved = []
    for w in weights:
        q, mx, rx, my, ry = w.parts
        ptrs = [keep(np.concatenate([np.zeros(b, np.uint8), np.ascontiguousarray(v).reshape(-1).view(np.uint8)])).ptr + b
                for v, b in ((q.T, 4), (mx, 2), (rx, 2), (my, 2), (ry, 2))]
        moved.append(fr.Weight(*ptrs, w.K, w.N, fr.U8))
    outs = []
    for kw, vw, rw in ([w.ref for w in weights], [C.byref(m) for m in moved]):
        x_out, xx_out, ws = DevBuf.empty((T, C_), np.float16), DevBuf.empty(C_, np.float16), DevBuf(L().frhip_seq_workspace_bytes(T, C_, F_))
        fr.check(L().frhip_ffn_seq(T, C_, F_, *[v.ptr for v in vecs], kw, vw, rw, x_out.ptr, xx_out.ptr, 0, ws.ptr, None))
        outs.append(x_out.numpy())
    assert np.array_equal(outs[0].view(np.uint16), outs[1].view(np.uint16))


@pytest.mark.parametrize("T,C_", [(3, 2048), (1, 2112), (5, 2304), (2, 2560), (7, 4032)])  # a thread per group, one to five waves beside the first four
def test_layernorm_of_rows_with_more_groups_than_sums(T, C_):
    test_ffn_seq(T, C_, 128, False)
    test_att_seq_v4(T, C_, False, True)
    test_att_seq_v5_2(T, C_, C_ // 64, False)


@pytest.mark.parametrize("T,C_", [(9, 4096), (5, 4160), (9, 5120), (1, 6144), (3, 6208)])  # 16-byte groups; one element at a time (three times); general form
def test_ffn_seq_wide_rows(T, C_):
    """The layernorm and mix of wide rows, at the edges of the register forms.  Bounds as in test_ffn_seq."""
    test_ffn_seq(T, C_, 128, False)


def _ln_rows(x, g, b, strided):
    """LN of the rows of x in fp32 with the sums taken thread by thread (256 threads: elements t, t + 256, ..., or groups
    of 8 consecutive ones), then over the lanes of a wave (pairs, fours, eights, rows of 16, the four rows in turn), then
    over the four waves."""
    f = np.float32
    rows, C_ = x.shape
    if strided:
        own = np.zeros((rows, -(-C_ // 256) * 256), f)
        own[:, :C_] = x
        valid = (np.arange(own.shape[1]) < C_).reshape(-1, 256)
        own = own.reshape(rows, -1, 256).transpose(1, 0, 2)
    else:
        n = -(-C_ // 2048) * 2048
        own, valid = np.zeros((rows, n), f), np.arange(n) < C_
        own[:, :C_] = x
        own = own.reshape(rows, -1, 256, 8).transpose(1, 3, 0, 2).reshape(-1, rows, 256)
        valid = valid.reshape(-1, 256, 8).transpose(0, 2, 1).reshape(-1, 256)

    def total(v):
        s = np.zeros((rows, 256), f)
        for e, ok in zip(v, valid):
            s = np.where(ok, s + e, s)
        for _ in range(4):
            s = s[:, 0::2] + s[:, 1::2]
        s = s.reshape(rows, 4, 4)
        w = ((s[:, :, 0] + s[:, :, 1]) + s[:, :, 2]) + s[:, :, 3]
        return ((w[:, 0] + w[:, 1]) + w[:, 2]) + w[:, 3]

    mean = total(own) / f(C_)
    d = own - mean[None, :, None]
    var = np.maximum(total(d * d) / f(C_), f(0))
    inv = f(1) / np.sqrt(var + f(1e-5))
    d = x.astype(f) - mean[:, None]
    n = (d * inv[:, None]).astype(np.float16)
    if strided:  # the last element of a thread with an odd count is rounded once, from the exact product
        at = np.arange(C_)
        last = (at + 256 >= C_) & (at // 256 % 2 == 0)
        n[:, last] = (d[:, last].astype(np.float64) * inv[:, None]).astype(np.float16)
    return n * g + b


@pytest.mark.parametrize("C_", [4160, 4608, 4736, 5120, 5952, 6144, 6208, 6656])
def test_layernorm_of_wide_rows_sums_in_one_order(C_):
    """The new shift state is LN of the last row, bit for bit, with thread t summing elements t, t + 256, ... whichever
    form of the kernel a width takes (6208, 6656: the general one; 4160 to 6208 but for 4608, 5120 and 6144: some threads have an odd
    count of elements); vectors that start at an odd binary16 address are taken as they are.  (The inputs
    tell that order from groups of 8 consecutive elements.)"""
    rows = 96
    x, g, b = h(rng.standard_normal((rows, C_)) * 2 + 1), h(1 + 0.1 * rng.standard_normal(C_)), h(0.1 * rng.standard_normal(C_))
    want = _ln_rows(x, g, b, True)
    assert (want.view(np.uint16) != _ln_rows(x, g, b, False).view(np.uint16)).any(axis=1).sum() >= 3
    odd = [keep(np.concatenate([h([7]), v])) for v in (h(rng.standard_normal(C_)), g, b, h(rng.uniform(0, 1, C_)), h(rng.uniform(0, 1, C_)))]
    kw, vw, rw = (make_weight(h(rng.standard_normal(s) * 0.02), False)[0] for s in ((C_, 64), (64, C_), (C_, C_)))
    x_dev, x_out, xx_out = keep(x), DevBuf.empty((8, C_), np.float16), DevBuf.empty(C_ + 1, np.float16)
    ws = DevBuf(L().frhip_seq_workspace_bytes(8, C_, 64))
    for last in range(rows):
        T = min(last + 1, 1 + last % 8)
        fr.check(L().frhip_ffn_seq(T, C_, 64, x_dev.ptr + 2 * C_ * (last + 1 - T), *[v.ptr + 2 for v in odd], kw.ref, vw.ref,
                                   rw.ref, x_out.ptr, xx_out.ptr + 2, 0, ws.ptr, None))
        assert np.array_equal(xx_out.numpy()[1:].view(np.uint16), want[last].view(np.uint16)), last


@pytest.mark.parametrize("T,C_,F_", [(64, 512, 1792), (1024, 2048, 8192), (1, 512, 1024), (200, 768, 3072)])
@pytest.mark.parametrize("quant", [False, True])
def test_ffn_seq_with_the_halving_folded_in(T, C_, F_, quant):
    """post_div2 = 1: the rows leave halved in binary16 after the residual, the bits of scalar_div_(x_out, 2) on
    the result without it (model_forward_seq.cpp:163-165 halves the rows after every sixth layer); in the
    launch split over K the halving sits in the reduction pass."""
    g = np.random.default_rng(7000 + T)
    x, sx = h(g.standard_normal((T, C_)) * 2), h(g.standard_normal(C_))
    ln_w, ln_b = h(1 + 0.1 * g.standard_normal(C_)), h(0.1 * g.standard_normal(C_))
    mk, mr = h(g.uniform(0, 1, C_)), h(g.uniform(0, 1, C_))
    kw, _ = make_weight(h(g.standard_normal((C_, F_)) * 0.02), quant)
    vw, _ = make_weight(h(g.standard_normal((F_, C_)) * 0.02), quant)
    rw, _ = make_weight(h(g.standard_normal((C_, C_)) * 0.02), quant)
    ws = DevBuf(L().frhip_seq_workspace_bytes(T, C_, F_))
    outs = []
    for div2 in (0, 1):
        x_out, xx_out = DevBuf.empty((T, C_), np.float16), DevBuf.empty(C_, np.float16)
        fr.check(L().frhip_ffn_seq(T, C_, F_, keep(x).ptr, keep(sx).ptr, keep(ln_w).ptr, keep(ln_b).ptr, keep(mk).ptr,
                                   keep(mr).ptr, kw.ref, vw.ref, rw.ref, x_out.ptr, xx_out.ptr, div2, ws.ptr, None))
        outs.append((x_out.numpy(), xx_out.numpy()))
    assert np.array_equal(outs[1][0], outs[0][0] / np.float16(2))
    assert np.array_equal(outs[1][1], outs[0][1])  # the shift state is LN(x) of the last row: not halved


def _state_v4(C_, fresh):
    if fresh:
        return np.zeros(C_, np.float32), np.zeros(C_, np.float32), np.full(C_, -1e30, np.float32)
    return (rng.standard_normal(C_).astype(np.float32), rng.uniform(0.5, 3, C_).astype(np.float32),
            rng.standard_normal(C_).astype(np.float32))


@pytest.mark.parametrize("T,C_", [(64, 512), (1024, 2048), (1, 512), (37, 768), (3000, 512), (24, 2048), (150, 2048), (500, 512)])  # 3000: a long, ragged prompt (two blocks); 24, 150: short prompts at full width; 500: products of many rows and few columns
@pytest.mark.parametrize("quant", [False, True])
@pytest.mark.parametrize("fresh", [True, False])
def test_att_seq_v4(T, C_, quant, fresh):
    x, sx = h(rng.standard_normal((T, C_)) * 2), h(rng.standard_normal(C_))
    aa, bb, pp = _state_v4(C_, fresh)
    ln_w, ln_b = _common(C_)
    mixes = [h(rng.uniform(0, 1, C_)) for _ in range(3)]
    td = (-np.exp(rng.uniform(-5, 1, C_))).astype(np.float32)
    tf = rng.uniform(-1, 1, C_).astype(np.float32)
    ws_, refs = [], []
    for _ in range(4):
        w, r = make_weight(h(rng.standard_normal((C_, C_)) * 0.02), quant)
        ws_.append(w)
        refs.append(r)
    ref = po.att_seq_v4_f16(x, sx, aa, bb, pp, ln_w, ln_b, *mixes, td, tf, *refs)
    x_out, xx_out = DevBuf.empty((T, C_), np.float16), DevBuf.empty(C_, np.float16)
    ao, bo, po_ = (DevBuf.empty(C_, np.float32) for _ in range(3))
    ws = DevBuf(L().frhip_seq_workspace_bytes(T, C_, 4 * C_))
    fr.check(L().frhip_att_seq_v4(T, C_, keep(x).ptr, keep(sx).ptr, keep(aa).ptr, keep(bb).ptr, keep(pp).ptr,
                                  keep(ln_w).ptr, keep(ln_b).ptr, *[keep(m).ptr for m in mixes], keep(td).ptr,
                                  keep(tf).ptr, *[w.ref for w in ws_], x_out.ptr, xx_out.ptr, ao.ptr, bo.ptr, po_.ptr,
                                  ws.ptr, None))
    assert_close_f16(xx_out.numpy(), ref[1], max_ulp=1, what="xx_last")
    assert_close_f16(x_out.numpy(), ref[0], max_ulp=3, max_frac=0.1, what="x_out")
    # the carried state: same value, possibly another exponent offset pp -> compare aa*e^pp etc.
    for got, want in ((ao, ref[2]), (bo, ref[3])):
        g = got.numpy().astype(np.float64) * np.exp(po_.numpy().astype(np.float64) - ref[4].astype(np.float64))
        assert np.allclose(g, want, rtol=2e-3, atol=2e-3 * np.abs(want).max())
    assert np.abs(po_.numpy() - ref[4]).max() < 30  # offsets stay in a sane range


@pytest.mark.parametrize("T,C_", [(2, 512), (3, 512), (32, 512), (33, 512),  # one wave's chunks of 2 steps; of 4
                                  (513, 320), (1025, 192),                  # 5 of 8 and 9 of 16 registers of a chunk in use
                                  (2049, 128), (4097, 64),                  # two and three blocks, the last one ragged
                                  (66, 2560), (17, 5120)])                  # 10 and 20 channels a workgroup, partial waves
def test_att_seq_v4_scan_cuts(T, C_):
    """The scan's cuts of time with 8 channels a workgroup, one to three blocks, and of one block with 10 and 20; blocks of
    wider models: the test below.  Bounds as in test_att_seq_v4."""
    test_att_seq_v4(T, C_, False, False)


@pytest.mark.parametrize("T,C_,cut", [(1900, 2112, (9, 235, 2, 106, 9)),    # two blocks; three channels past the end in the last workgroup
                                      (1100, 2304, (9, 256, 1, 110, 10)),   # ten registers of a chunk in use
                                      (1700, 2560, (10, 256, 2, 95, 9)),
                                      (1250, 3584, (14, 256, 2, 70, 9)),    # a partial wave
                                      (900, 5120, (20, 256, 2, 50, 9)),
                                      (1280, 4736, (19, 250, 2, 50, 13)),   # 13 of 14 registers; 14 channels past the end
                                      (560, 8256, (17, 486, 1, 56, 10))])   # two workgroups a compute unit
def test_att_seq_v4_in_one_pass_and_in_parts(T, C_, cut):
    """Blocks of time one after another with more than 8 channels a workgroup, and channels past the end: a prompt in one
    pass against the same prompt in parts of at most 256 rows (one block each, held against the oracle above), the state
    carried between them.  The fp32 sums are in another order, the products' as well, so that a binary16 rounding may go
    the other way: of the output product o, by one spacing of o, and of x + o, by one of x + o; a third for an o at the edge
    of its binade.  The inputs of o may have gone the other way too: 1 % of up to 8256 elements by 2^-12 or so, times weights
    of 0.02, is 4e-5 rms, which the spacing at a quarter of the outputs' rms (2.4e-4 to 4.9e-4) covers six times over.
    States as in test_att_seq_v4.  What lies past the last channel's state stays as it was."""
    out = (C.c_int * 5)()
    fr.check(L().frhip_wkv4_cut(T, C_, 256, out))
    assert tuple(out) == cut
    x, sx = h(rng.standard_normal((T, C_)) * 2), h(rng.standard_normal(C_))
    state = _state_v4(C_, False)
    consts = [keep(a).ptr for a in (*_common(C_), *[h(rng.uniform(0, 1, C_)) for _ in range(3)],
                                    (-np.exp(rng.uniform(-5, 1, C_))).astype(np.float32), rng.uniform(-1, 1, C_).astype(np.float32))]
    w = h(rng.standard_normal((C_, C_)) * 0.02)
    ws_ = [make_weight(np.ascontiguousarray(np.roll(w, 17 * i)), False)[0] for i in range(4)]
    ws, x_dev = DevBuf(L().frhip_seq_workspace_bytes(T, C_, 64)), keep(x)
    results = []
    for step in (T, 256):
        x_out, xx = DevBuf.empty((T, C_), np.float16), [keep(sx), DevBuf.empty(C_, np.float16)]
        st = [dev(np.concatenate([s, [7.5]]).astype(np.float32)) for s in state]
        for lo in range(0, T, step):
            fr.check(L().frhip_att_seq_v4(min(step, T - lo), C_, x_dev.ptr + 2 * C_ * lo, xx[0].ptr, *[s.ptr for s in st], *consts,
                                          *[v.ref for v in ws_], x_out.ptr + 2 * C_ * lo, xx[1].ptr, *[s.ptr for s in st], ws.ptr, None))
            xx = [xx[1], DevBuf.empty(C_, np.float16)]
        results.append((x_out.numpy(), *[s.numpy() for s in st]))
    (one, a1, b1, p1), (parts, a2, b2, p2) = results
    assert a1[C_] == b1[C_] == p1[C_] == 7.5
    one, parts = one.astype(np.float32), parts.astype(np.float32)
    spacing = np.exp2(np.floor(np.log2(np.maximum(np.abs(parts - x), np.maximum(np.abs(parts), parts.std() / 4)))) - 10)
    assert (np.abs(one - parts) <= 3 * spacing).all() and (one != parts).mean() < 0.1
    scale = np.exp((p1 - p2)[:C_].astype(np.float64))
    for got, want in ((a1, a2), (b1, b2)):
        want = want[:C_].astype(np.float64)
        assert np.allclose(got[:C_] * scale, want, rtol=2e-3, atol=2e-3 * np.abs(want).max())


@pytest.mark.parametrize("T,C_,kvr,o", [(16400, 320, (256, 5, 2, 0), (256, 4, 1, 0)),  # predicated epilogues: 16 rows in the last strip
                                        (5632, 320, (256, 4, 1, 1), (128, 2, 1, 1))])  # whole tiles: the loader wave's form
def test_att_seq_v4_on_planned_tiles(T, C_, kvr, o):
    """k, v, r grouped and the residual's epilogue on 256-row tiles.  Bounds as in test_att_seq_v4."""
    assert _routes(T, C_, C_, C_, C_) == (1, [kvr] * 3) and _routes(T, C_, C_) == (1, [o])
    test_att_seq_v4(T, C_, False, False)


@pytest.mark.parametrize("T,C_", [(1024, 2048), (700, 512), (5000, 256)])  # 5000: three blocks of time
def test_att_seq_v4_state_updated_in_place_equals_separate_outputs(T, C_):
    """The header allows aa_out / bb_out / pp_out to be the buffers of aa / bb / pp (as frhip_att_one_v4 does).
    A channel's workgroup reads the state before it writes it, and no other touches it.  Bit for bit the same as with
    separate outputs."""
    x, sx = h(rng.standard_normal((T, C_)) * 2), h(rng.standard_normal(C_))
    aa, bb, pp = _state_v4(C_, False)
    ln_w, ln_b = _common(C_)
    mixes = [h(rng.uniform(0, 1, C_)) for _ in range(3)]
    td = (-np.exp(rng.uniform(-5, 1, C_))).astype(np.float32)
    tf = rng.uniform(-1, 1, C_).astype(np.float32)
    pairs = [make_weight(h(rng.standard_normal((C_, C_)) * 0.02), False) for _ in range(4)]
    ws_, refs = [p[0] for p in pairs], [p[1] for p in pairs]
    ws = DevBuf(L().frhip_seq_workspace_bytes(T, C_, 4 * C_))
    dx, dsx = keep(x), keep(sx)
    consts = [keep(a).ptr for a in (ln_w, ln_b, *mixes, td, tf)]
    results = []
    for in_place in (False, True):
        st = [dev(aa), dev(bb), dev(pp)]
        outs = st if in_place else [DevBuf.empty(C_, np.float32) for _ in range(3)]
        x_out, xx_out = DevBuf.empty((T, C_), np.float16), DevBuf.empty(C_, np.float16)
        fr.check(L().frhip_att_seq_v4(T, C_, dx.ptr, dsx.ptr, st[0].ptr, st[1].ptr, st[2].ptr, *consts,
                                      *[w.ref for w in ws_], x_out.ptr, xx_out.ptr, outs[0].ptr, outs[1].ptr, outs[2].ptr,
                                      ws.ptr, None))
        results.append([x_out.numpy(), xx_out.numpy()] + [o.numpy() for o in outs])
    for sep, inp in zip(*results):
        assert np.array_equal(sep, inp)
    if T == 5000:  # the long prompt against the oracle as well
        ref = po.att_seq_v4_f16(x, sx, aa, bb, pp, ln_w, ln_b, *mixes, td, tf, *refs)
        assert_close_f16(results[0][0], ref[0], max_ulp=3, max_frac=0.1, what="x_out, T = 5000")


@pytest.mark.parametrize("T,C_,H_", [(48, 512, 8), (512, 2560, 40), (1, 512, 8), (77, 512, 8), (3000, 512, 8), (40, 2560, 40)])  # (40, 2560, 40): k,v,r,g of a short prompt in one split launch
@pytest.mark.parametrize("quant", [False, True])
def test_att_seq_v5_2(T, C_, H_, quant):
    S_ = C_ // H_
    x, sx = h(rng.standard_normal((T, C_)) * 2), h(rng.standard_normal(C_))
    s = rng.standard_normal((H_, S_, S_)).astype(np.float32)
    ln_w, ln_b = _common(C_)
    lx_w = (1 + 0.1 * rng.standard_normal(C_)).astype(np.float32)
    lx_b = (0.1 * rng.standard_normal(C_)).astype(np.float32)
    mixes = [h(rng.uniform(0, 1, C_)) for _ in range(4)]
    td = np.exp(-np.exp(rng.uniform(-6, 0, (H_, S_)))).astype(np.float32)
    tf = rng.uniform(-1, 1, (H_, S_)).astype(np.float32)
    ws_, refs = [], []
    for _ in range(5):
        w, r = make_weight(h(rng.standard_normal((C_, C_)) * 0.02), quant)
        ws_.append(w)
        refs.append(r)
    ref_x, ref_xx, ref_s = po.att_v5_2_f16(x if T > 1 else x[0], sx, s, ln_w, ln_b, lx_w, lx_b, *mixes, td, tf, *refs, H_)
    x_out, xx_out = DevBuf.empty((T, C_), np.float16), DevBuf.empty(C_, np.float16)
    s_out = DevBuf.empty((H_, S_, S_), np.float32)
    ws = DevBuf(L().frhip_seq_workspace_bytes(T, C_, 4 * C_))
    fr.check(L().frhip_att_seq_v5_2(T, C_, H_, keep(x).ptr, keep(sx).ptr, keep(s).ptr, keep(ln_w).ptr, keep(ln_b).ptr,
                                    keep(lx_w).ptr, keep(lx_b).ptr, *[keep(m).ptr for m in mixes], keep(td).ptr,
                                    keep(tf).ptr, *[w.ref for w in ws_], x_out.ptr, xx_out.ptr, s_out.ptr, ws.ptr,
                                    None))
    assert_close_f16(xx_out.numpy(), ref_xx, max_ulp=1, what="xx_last")
    assert np.allclose(s_out.numpy(), ref_s, rtol=1e-4, atol=1e-4 * np.abs(ref_s).max())
    assert_close_f16(x_out.numpy().reshape(ref_x.shape), ref_x, max_ulp=4, max_frac=0.2, what="x_out", floor_rms=1.0)


@pytest.mark.parametrize("T,C_,H_", [(48, 512, 8), (300, 2048, 32), (1, 512, 8), (77, 512, 8)])
@pytest.mark.parametrize("quant", [False, True])
def test_att_seq_v5(T, C_, H_, quant):
    """RWKV-5.0 seq attention against the oracle's matrix form (kernels/cuda/att_seq.cu:158-256)."""
    S_ = C_ // H_
    x, sx = h(rng.standard_normal((T, C_)) * 2), h(rng.standard_normal(C_))
    s = rng.standard_normal((H_, S_, S_)).astype(np.float32)
    ln_w, ln_b = _common(C_)
    lx_w = (1 + 0.1 * rng.standard_normal(C_)).astype(np.float32)
    lx_b = (0.1 * rng.standard_normal(C_)).astype(np.float32)
    mixes = [h(rng.uniform(0, 1, C_)) for _ in range(3)]
    td = np.exp(-np.exp(rng.uniform(-6, 0, H_))).astype(np.float32)
    tf = rng.uniform(-1, 1, H_).astype(np.float32)
    ws_, refs = [], []
    for _ in range(4):
        w, r = make_weight(h(rng.standard_normal((C_, C_)) * 0.02), quant)
        ws_.append(w)
        refs.append(r)
    ref_x, ref_xx, ref_s = po.att_v5_0_f16(x if T > 1 else x[0], sx, s, ln_w, ln_b, lx_w, lx_b, *mixes, td, tf, *refs, H_)
    x_out, xx_out = DevBuf.empty((T, C_), np.float16), DevBuf.empty(C_, np.float16)
    s_out = DevBuf.empty((H_, S_, S_), np.float32)
    ws = DevBuf(L().frhip_seq_workspace_bytes(T, C_, 4 * C_))
    fr.check(L().frhip_att_seq_v5(T, C_, H_, keep(x).ptr, keep(sx).ptr, keep(s).ptr, keep(ln_w).ptr, keep(ln_b).ptr,
                                  keep(lx_w).ptr, keep(lx_b).ptr, *[keep(m).ptr for m in mixes], keep(td).ptr,
                                  keep(tf).ptr, *[w.ref for w in ws_], x_out.ptr, xx_out.ptr, s_out.ptr, ws.ptr,
                                  None))
    assert_close_f16(xx_out.numpy(), ref_xx, max_ulp=1, what="xx_last")
    assert np.allclose(s_out.numpy(), ref_s, rtol=1e-4, atol=1e-4 * np.abs(ref_s).max())
    assert_close_f16(x_out.numpy().reshape(ref_x.shape), ref_x, max_ulp=4, max_frac=0.2, what="x_out", floor_rms=1.0)
