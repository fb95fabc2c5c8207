"""The order in which the seq operators of RWKV-5 models add over K: contiguous slices, at any number of rows."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import pyoracle as po
from hipref import DevBuf, L, dev, fr, make_weight

BIG = 2.0 ** 15
rng = np.random.default_rng(4)


def _rows(n, at=1.0):
    """A vector with +-2^15 at 0 and 64, and `at` at 256 and 512: against a weight of 2^15 in rows 0 and 64, the products
    are +-2^30 in the first and second K-step of 64 and small numbers in the fifth and ninth.  Slices of at least four steps
    cancel the large ones before anything else is added, and the sums are exact; with every fourth or eighth step in one
    sum, a small number is added to 2^30, whose spacing is 128, and is lost."""
    v = np.zeros(n, np.float16)
    v[[0, 64]] = BIG, -BIG
    v[[256, 512]] = at
    return v


def _weight(K, N, a, b):
    w = np.zeros((K, N), np.float16)
    w[[0, 64]] = BIG
    w[256], w[512] = a, b
    return w, w[256].astype(np.float64), w[512].astype(np.float64)


def _h(x):
    return np.asarray(x, np.float64).astype(np.float16)


@pytest.mark.parametrize("T", [4, 16, 64, 65, 130, 300])
def test_ffn_seq_adds_in_slices(T):
    C_, F_ = 1024, 2048
    n, c = np.arange(F_), np.arange(C_)
    kw, k1, k2 = _weight(C_, F_, 1 + n % 3, n % 5)
    kw[256, [0, 64]], kw[512, [0, 64]] = 1, 180  # the key's rows 0 and 64: 181^2 = 2^15 in binary16
    k1[[0, 64]], k2[[0, 64]] = 1, 180
    rw, r1, r2 = _weight(C_, C_, c % 7 - 3, c % 4 - 1)
    vw, v1, v2 = _weight(F_, C_, 1 + c % 3, c % 5)
    vw[64] = -BIG
    x, xx = (rng.standard_normal((T, C_)) * 2).astype(np.float16), _rows(C_)
    key = _h((k1 + k2) ** 2).astype(np.float64)
    assert key[0] == key[64] == BIG
    value = key[256] * v1 + key[512] * v2
    want = _h(value[None, :] * po.sigmoid_f16(_h(r1 + r2)).astype(np.float64) + x.astype(np.float64))
    ones, zeros = np.ones(C_, np.float16), np.zeros(C_, np.float16)
    bufs = [dev(a) for a in (x, (rng.standard_normal(C_)).astype(np.float16), zeros, xx, ones, ones)]
    W = [make_weight(w, False)[0] for w in (kw, vw, rw)]
    x_out, xx_out, ws = DevBuf.empty((T, C_), np.float16), DevBuf.empty(C_, np.float16), DevBuf(L().frhip_seq_workspace_bytes(T, C_, F_))
    fr.check(L().frhip_ffn_seq(T, C_, F_, *[b.ptr for b in bufs], *[w.ref for w in W], x_out.ptr, xx_out.ptr, 0, ws.ptr, None))
    assert np.array_equal(xx_out.numpy(), xx)
    assert np.array_equal(x_out.numpy(), want)


@pytest.mark.parametrize("T", [4, 16, 64, 65, 130, 300])
@pytest.mark.parametrize("gate", [True, False])
def test_att_seq_v5_adds_in_slices(T, gate):
    """gate: RWKV-5.2, else 5.0.  A decay of zero leaves k v^T of the last token as the new state; a group normalisation of
    weight zero leaves its bias, times the gate, as the vector that the output weight multiplies."""
    C_, H_ = 1024, 16
    c = np.arange(C_)
    (kw, k1, k2), (vw, v1, v2), (rw, _, _) = (_weight(C_, C_, a, b) for a, b in ((1 + c % 3, c % 5), (c % 4, 1 + c % 7), (c % 2, c % 3)))
    gw, g1, g2 = _weight(C_, C_, 1 + c % 2 * (c > 64), 1 + c % 3 * (c > 64))
    ow, o1, o2 = _weight(C_, C_, 1 + c % 5, c % 3)
    x, xx = (rng.standard_normal((T, C_)) * 2).astype(np.float16), _rows(C_)
    bias = _rows(C_)
    bias[[0, 64]] = BIG / 4, -BIG / 4
    gated = bias * po.silu_f16(_h(g1 + g2)) if gate else bias
    assert gated[0] == -gated[64] and np.isfinite(gated).all() and abs(float(gated[0])) >= BIG / 4
    out = float(gated[256]) * o1 + float(gated[512]) * o2
    state = ((k1 + k2).reshape(H_, 64, 1) * (v1 + v2).reshape(H_, 1, 64)).astype(np.float32)
    ones, zeros = np.ones(C_, np.float16), np.zeros(C_, np.float16)
    per = C_ if gate else H_
    bufs = [dev(a) for a in (x, rng.standard_normal(C_).astype(np.float16), rng.standard_normal((H_, 64, 64)).astype(np.float32), zeros, xx,
                             np.zeros(C_, np.float32), bias.astype(np.float32), *[ones] * (4 if gate else 3),
                             np.zeros(per, np.float32), np.ones(per, np.float32))]
    W = [make_weight(w, False)[0] for w in (kw, vw, rw, *[gw] * gate, ow)]
    x_out, xx_out, s_out = DevBuf.empty((T, C_), np.float16), DevBuf.empty(C_, np.float16), DevBuf.empty((H_, 64, 64), np.float32)
    ws = DevBuf(L().frhip_seq_workspace_bytes(T, C_, 64))
    f = L().frhip_att_seq_v5_2 if gate else L().frhip_att_seq_v5
    fr.check(f(T, C_, H_, *[b.ptr for b in bufs], *[w.ref for w in W], x_out.ptr, xx_out.ptr, s_out.ptr, ws.ptr, None))
    assert np.array_equal(s_out.numpy(), state)
    # the products' sums are exact or, the gate's binary16 values times small numbers, rounded at most twice in fp32
    want = x.astype(np.float64) + _h(out).astype(np.float64)
    assert np.array_equal(x_out.numpy(), _h(want))


@pytest.mark.parametrize("version,H", [("5.2", 8), ("5", 8), ("4", 0)])
def test_model_pass_takes_the_operators_of_its_version(tmp_path, version, H, monkeypatch):
    """A short prompt through the fused pass and through the operators one by one leaves the same bits behind."""
    from synth import make_model
    params, emb = make_model({"4": 4, "5": 50}.get(version, 52), 3, 512, 1792, 2048, H, seed=9)
    path = str(tmp_path / "m.fr")
    fr.write_fr(path, version, 3, 512, 1792, H, params, emb)
    ids = [int(t) for t in np.random.default_rng(1).integers(0, 2048, 16)]
    after = []
    for generic in (False, True):
        m = fr.Model(path, "hip fp16")
        if generic:
            monkeypatch.setenv("FR_HIP_GENERIC", "1")
        m.run(ids)
        monkeypatch.delenv("FR_HIP_GENERIC", raising=False)
        after.append(np.array(m.run(7)))
        m.close()
    assert np.array_equal(after[0].view(np.uint32), after[1].view(np.uint32))
