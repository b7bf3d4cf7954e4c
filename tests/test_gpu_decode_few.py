"""Decode launches of few rows: the several-wave variants of the GQA MFMA
decode (8 waves per (row, kv-head) up to one item per CU, 4 up to five, one
beyond; a step's store fused into the first two) and the eight-wave VALU
launches, at the edges of those rules, against attention in 64 bits over the
rows as the cache holds them.

Tolerances: every weight and product carries an error of a few units of 2^-22
(fp16 pairs) or 2^-24 (fp32), and an output is a weighted mean of |v| < 6, so
1e-5 is ten times what they add up to."""
import numpy as np
import pytest

import ndoracle as O

pytestmark = pytest.mark.gpu

TOL = 1e-5
RNG = np.random.default_rng


def nda():
    import ndattn
    return ndattn


def attend(q, k, v, gate):
    """q [nh][qk], k / v [L][nkv][...] -> [nh][v]"""
    rep = q.shape[0] // k.shape[1]
    s = np.einsum("hd,lhd->hl", q.astype(np.float64), np.repeat(k, rep, 1)) / np.sqrt(q.shape[1])
    p = np.exp(s - s.max(-1, keepdims=True))
    out = np.einsum("hl,lhd->hd", p / p.sum(-1, keepdims=True), np.repeat(v, rep, 1))
    return out / (1 + np.exp(-gate.astype(np.float64)))


def check(nh, nkv, qk, f16, lens, seed, page=16, fused=True, vscale=None, tol=TOL, least=1.0):
    """One token of each sequence b behind lens[b] positions; nda_step, or an
    append and a decode. vscale [rows]: per-position factors of v. Errors are
    relative to a row's largest output, or to `least` where that is more."""
    N = nda()
    vd, B = 64, len(lens)
    rng = RNG(seed)
    total = int(sum(lens))
    W = max(lens) + 64
    k = rng.standard_normal((total, nkv, qk)).astype(np.float32)
    v = rng.standard_normal((total, nkv, vd)).astype(np.float32)
    if vscale is not None:
        v *= vscale(total)[:, None, None].astype(np.float32)
    ctx = N.Context(1, nh, nkv, qk, vd, W, kv_dtype=N.KV_F16 if f16 else N.KV_INT8, max_seqs=B, page_size=page)
    zero = N.DevBuf.from_array(np.zeros((total, nh, qk), np.float32))
    dk, dv, dump = N.DevBuf.from_array(k), N.DevBuf.from_array(v), N.DevBuf(total * nh * vd * 4)
    ctx.prefill(0, np.asarray(lens, np.uint32), zero, dk, dv, dump)
    for b, n in enumerate(lens):
        if n:
            ctx.advance(1, [b], int(n))
    q = rng.standard_normal((B, nh, qk)).astype(np.float32)
    kn = rng.standard_normal((B, nkv, qk)).astype(np.float32)
    vn = rng.standard_normal((B, nkv, vd)).astype(np.float32)
    if vscale is not None:
        vn *= np.float32(vscale(total)[-1])
    gate = rng.standard_normal((B, nh, vd)).astype(np.float32)
    bufs = [N.DevBuf.from_array(a) for a in (q, kn, vn, gate)]
    out = N.DevBuf(B * nh * vd * 4)
    if fused:
        ctx.step(0, B, bufs[0], bufs[1], bufs[2], out, gate=bufs[3])
    else:
        ctx.kv_append(0, B, bufs[1], bufs[2])
        ctx.decode(0, B, bufs[0], out, gate=bufs[3])
    ctx.sync()
    got = out.to_array(np.float32, (B, nh, vd))
    worst = 0.0
    for b in range(B):
        kr, vr, sk, sv = ctx.kv_read(0, b, 0, int(lens[b]) + 1)
        if f16:
            kr, vr = kr.view(np.float16), vr.view(np.float16)
        if not f16:
            for new, codes in ((kn[b], kr[-1]), (vn[b], vr[-1])):       # the stored token
                for g in range(nkv):
                    want = np.zeros(new.shape[1], np.int8)
                    O.lib().ndo_kv_quant_row(np.ascontiguousarray(new[g]), new.shape[1], want)
                    assert np.array_equal(codes[g], want)
        else:
            assert np.array_equal(kr[-1], kn[b].astype(np.float16)) and np.array_equal(vr[-1], vn[b].astype(np.float16))
        want = attend(q[b], kr.astype(np.float64) * sk[..., None], vr.astype(np.float64) * sv[..., None], gate[b])
        worst = max(worst, float(np.abs(got[b] - want).max() / max(least, np.abs(want).max())))
    ctx.close()
    print("[gpu-case] heads %d/%d qk %d %s rows %d page %d: %.3g" % (nh, nkv, qk, "f16" if f16 else "i8", B, page, worst),
          flush=True)
    assert worst <= tol


# 2 kv-heads: 256 items (8 waves), 258 and 1280 (4), 1282 (1)
@pytest.mark.parametrize("rows", [1, 3, 128, 129, 640, 641])
@pytest.mark.parametrize("fused", [True, False])
def test_mfma_waves(rows, fused):
    # fewer tiles than waves, the edges of a tile, one tile more than waves
    lens = [(0, 1, 15, 30, 31, 32, 33, 63, 64, 127, 128, 255, 256, 300)[(5 * b + rows) % 14] for b in range(rows)]
    check(12, 2, 48, False, lens, 10 + rows, fused=fused)


@pytest.mark.parametrize("nh,nkv,qk,page", [(12, 2, 48, 32), (8, 2, 64, 16), (6, 1, 64, 64), (16, 2, 64, 16)])
@pytest.mark.parametrize("rows", [5, 300])
def test_mfma_waves_shapes(nh, nkv, qk, page, rows):
    check(nh, nkv, qk, False, [(3 * b + 7) % 290 for b in range(rows)], rows, page=page)


@pytest.mark.parametrize("f", [lambda n: np.geomspace(1e-6, 1e6, n), lambda n: np.geomspace(1e6, 1e-6, n),
                               lambda n: np.where(np.arange(n) % 3, 1.0, 0.0)])
def test_mfma_v_scales(f):
    """v rows whose scales span many powers of two, either way, and zero rows:
    errors relative to the largest output, which the largest rows make."""
    check(12, 2, 48, False, [277], 3, vscale=f)


@pytest.mark.parametrize("rows", [1, 130])
def test_mfma_zero_v_before_small_v(rows):
    """A wave's first key tile with v all zero, then v of about 1e-6: the
    scales' running exponent starts at the first nonzero one (8 and 4 waves
    over 32 tiles; every fourth tile is zero)."""
    f = lambda n: np.where(np.arange(n) % 1000 // 32 % 4, 1e-6, 0.0)     # noqa: E731
    check(12, 2, 48, False, [1000] * rows, 4, vscale=f, least=0.0)


@pytest.mark.parametrize("nh,nkv,qk,f16", [(12, 2, 48, True), (8, 8, 64, True), (8, 8, 64, False), (6, 2, 36, False),
                                           (10, 2, 64, True)])
@pytest.mark.parametrize("n", [126, 127, 128, 160, 255, 256, 420])
@pytest.mark.parametrize("fused", [True, False])
def test_valu_waves(nh, nkv, qk, f16, n, fused):
    check(nh, nkv, qk, f16, [n, n, n], n, fused=fused)


# 3 rows; one item per CU and one more, two and one more: where the least
# length for eight waves changes (rep 8: 128, 256 and 512 positions)
@pytest.mark.parametrize("nh,nkv,qk,f16,rows,n", [
    (8, 2, 64, True, 3, 128), (14, 2, 64, True, 3, 128), (16, 2, 64, True, 3, 300), (21, 3, 48, False, 3, 200),
    (16, 2, 64, True, 128, 128), (16, 2, 64, True, 129, 255), (16, 2, 64, True, 129, 256), (16, 2, 64, True, 257, 511),
    (16, 2, 64, True, 257, 512), (10, 2, 36, False, 200, 170),
])
@pytest.mark.parametrize("fused", [True, False])
def test_valu_waves_by_heads(nh, nkv, qk, f16, rows, n, fused):
    check(nh, nkv, qk, f16, [n - 1] * rows, n, fused=fused)


def test_valu_chunks():
    """Long rows in chunks, int8 and fp16, where the MFMA decode does not go."""
    for f16 in (True, False):
        check(12, 2, 48, f16, [3000, 1023, 40], 5, fused=True)
