"""The few-token MFMA kernels (gemm_skinny_impl.hpp) at the edges of their
tiles: half and whole row tiles, one and several K phases and K ranges, token
blocks, the streaming form, rows whose columns end inside a chunk, unaligned
activations.  Reference: the decoded weights (bit-exact, the oracle) times the
activations in 64 bits.

Bound: a product of two operand terms is exact, and an output is a sum of at
most 160 + K / 128 roundings in a row (a chain of eight MFMAs of 32 products
each, the chunk sums, the ways' and ranges' tree), each at most 2^-24 of the
sum of the terms' magnitudes.
"""
import numpy as np
import pytest

import oracle
from vxg_amd import engine, synth
from vxg_amd.formats import bf16_bits_to_f32, f32_to_bf16_bits
from parity_util import make, run_dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    e = engine.HipEngine()
    yield e
    e.close()


# rows, cols, tokens, f32 activations
SHAPES = [
    (1, 1, 2, False), (67, 31, 3, False), (9, 130, 4, True), (33, 576, 8, False), (130, 2047, 5, False),
    (16, 2048, 2, True), (4095, 260, 8, False), (4097, 264, 4, False), (40, 2056, 16, True), (37, 4104, 4, False),
    (70, 8200, 4, False), (70, 4104, 7, False), (24, 9001, 2, True), (35, 2049, 9, False), (50, 4160, 16, False),
    (49, 1032, 17, False), (97, 2047, 33, False), (31, 6144, 64, False), (32771, 72, 4, False), (32784, 2048, 9, False),
]


@pytest.mark.parametrize("kind", ["cb4", "g64", "q8", "q4_0"])
@pytest.mark.parametrize("rows,cols,M,f32", SHAPES)
def test_skinny_edges(eng, kind, rows, cols, M, f32):
    print(f"skinny {kind} rows={rows} cols={cols} M={M} f32={f32}", flush=True)
    m = synth.make_q40(rows, cols, seed=rows + M) if kind == "q4_0" else make(kind, rows, cols, seed=rows + M)
    t = eng.upload_packed(m)
    X = np.random.default_rng(cols + M).standard_normal((M, cols)).astype(np.float32)
    xh = X if f32 else f32_to_bf16_bits(X)
    Xq = (X if f32 else bf16_bits_to_f32(xh).reshape(M, cols)).astype(np.float64)
    got = run_dev(eng, t, xh, engine.DTYPE_F32 if f32 else engine.DTYPE_BF16, M, engine.DTYPE_F32)
    W = oracle.decode_rows(m).astype(np.float64)
    want, mag = Xq @ W.T, np.abs(Xq) @ np.abs(W).T
    bound = (160 + cols / 128) * 2.0 ** -24 * mag + 1e-30
    err = np.abs(got - want)
    assert np.all(err <= bound), float((err / bound).max())
    t.free()


def _special_rows(m, M, cols, p, seed):
    """N(0, 1) rows; row 0 scaled by 2^p, rows 1 .. 4 with an Inf, a -Inf (on a
    residual's column where the matrix has some), a NaN, and Infs of both signs."""
    X = np.random.default_rng(seed).standard_normal((M, cols)).astype(np.float32)
    res = np.unique(m.outliers_packed & 0xFFFF) if hasattr(m, "outliers_packed") else np.zeros(0, int)
    at = res[res.size // 2] if res.size else cols - 1
    X[0] = np.ldexp(np.clip(X[0], -3, 3), p)
    X[1, cols // 3] = np.inf
    X[2, at] = -np.inf
    X[3, cols - 2] = np.nan
    X[min(4, M - 1), 3], X[min(4, M - 1), cols - 1] = np.inf, -np.inf
    return X


@pytest.mark.parametrize("kind,p", [("cb4", 124), ("g64", 124), ("q8", 120), ("q4_0", 124)])
@pytest.mark.parametrize("rows,cols,M,f32", [
    (70, 544, 5, False), (70, 4160, 7, False), (4200, 300, 5, False), (40, 2600, 16, False), (40, 2600, 40, False),
    (70, 2100, 5, True), (70, 2600, 12, True), (32800, 288, 12, False)])
def test_skinny_values_at_the_end_of_f32_and_nonfinite(eng, kind, p, rows, cols, M, f32):
    """Outputs that f32 holds come out even where a group's or a block's sum
    before its scale does not fit, and Inf and NaN reach the outputs that the
    reference's loops give them to: gemv_cpu's up to 8 tokens (block dots
    overflow there as in the reference, so Q8_0 and Q4_0 stay smaller),
    gemm_cpu's above."""
    print(f"skinny nonfinite {kind} rows={rows} cols={cols} M={M} f32={f32}", flush=True)
    m = synth.make_q40(rows, cols, seed=9) if kind == "q4_0" else make(kind, rows, cols, seed=9)
    t = eng.upload_packed(m)
    if M <= 8 and kind in ("q8", "q4_0"):
        p = 60
    X = _special_rows(m, M, cols, p, cols + M)
    xh = X if f32 else f32_to_bf16_bits(X)
    Xq = X if f32 else bf16_bits_to_f32(xh).reshape(M, cols)
    got = run_dev(eng, t, xh, engine.DTYPE_F32 if f32 else engine.DTYPE_BF16, M, engine.DTYPE_F32)
    t.free()
    W = oracle.decode_rows(m).astype(np.float64)
    with np.errstate(all="ignore"):
        pat = oracle.gemm(m, Xq[1:5], threads=8) if M > 8 else np.stack([oracle.gemv(m, x) for x in Xq[1:5]])
    y = got[1:5]
    assert np.array_equal(np.isnan(y), np.isnan(pat)) and np.array_equal(np.isinf(y), np.isinf(pat))
    both = np.isinf(pat)
    assert np.array_equal(np.sign(y[both]), np.sign(pat[both]))
    fin = np.r_[0, 5:M]
    Xf = Xq[fin].astype(np.float64)
    want, mag = Xf @ W.T, np.abs(Xf) @ np.abs(W).T
    assert np.abs(want).max() < 3.4e38
    err = np.abs(got[fin] - want)
    assert np.all(err <= (160 + cols / 128) * 2.0 ** -24 * mag)


@pytest.mark.parametrize("kind,p", [("cb4", 124), ("q8", 120), ("q4_0", 124)])
@pytest.mark.parametrize("cols,M", [(544, 12), (2600, 12), (544, 40)])
def test_gated_values_at_the_end_of_f32(eng, kind, p, cols, M):
    """The gated form on such activations: a gate far below zero gives zero
    times a finite up, not 0 * Inf."""
    print(f"gated end of f32 {kind} cols={cols} M={M}", flush=True)
    F = 48
    m = synth.make_q40(2 * F, cols, seed=9) if kind == "q4_0" else make(kind, 2 * F, cols, seed=9)
    t = eng.upload_packed(m)
    X = np.ldexp(np.clip(np.random.default_rng(M).standard_normal((M, cols)), -3, 3).astype(np.float32), p)
    xh = f32_to_bf16_bits(X)
    xd, yd = eng.to_device(xh), eng.alloc(M * F * 4)
    eng.ffn_glu_dev(t, xd.ptr, engine.DTYPE_BF16, M, yd.ptr, engine.DTYPE_F32, F, engine.ACT_SILU, eng.stream)
    eng.synchronize()
    got = yd.download(np.float32, (M, F))
    for b in (xd, yd, t):
        b.free()
    y = bf16_bits_to_f32(xh).reshape(M, cols).astype(np.float64) @ oracle.decode_rows(m).astype(np.float64).T
    assert np.abs(y).max() < 3.4e38 and np.abs(y).min() > 200
    g, u = y[:, :F], y[:, F:]
    assert np.array_equal(got == 0, g < 0)
    assert np.array_equal(got[g > 0], np.where(u[g > 0] > 0, np.inf, -np.inf).astype(np.float32))


@pytest.mark.parametrize("kind", ["cb4", "g64", "q8", "q4_0"])
@pytest.mark.parametrize("rows,cols,M", [(70, 544, 3), (40, 2600, 7), (40, 2100, 12)])
def test_skinny_f32_activations_near_the_small_end(eng, kind, rows, cols, M):
    """f32 activations down to the subnormals keep all their bits.  Beyond the
    file's bound an output has an absolute error of at most half of f32's
    smallest step (2^-150) per product and per sum, before a scale below 1."""
    print(f"skinny small f32 {kind} rows={rows} cols={cols} M={M}", flush=True)
    m = synth.make_q40(rows, cols, seed=4) if kind == "q4_0" else make(kind, rows, cols, seed=4)
    t = eng.upload_packed(m)
    X = np.random.default_rng(M).standard_normal((M, cols))
    X = (X * np.exp2(np.linspace(-100, -136, M))[:, None]).astype(np.float32)
    got = run_dev(eng, t, X, engine.DTYPE_F32, M, engine.DTYPE_F32)
    t.free()
    W = oracle.decode_rows(m).astype(np.float64)
    want, mag = X.astype(np.float64) @ W.T, np.abs(X).astype(np.float64) @ np.abs(W).T
    err = np.abs(got - want)
    assert np.all(err <= (160 + cols / 128) * 2.0 ** -24 * mag + 2 * cols * 2.0 ** -150)


def test_skinny_small_centroids(eng):
    """Centroids near f32's small end keep all their bits: the table times
    2^-118, against the same products times 2^-118."""
    rows, cols, M = 70, 544, 6
    m = synth.make_cb4(rows, cols, seed=4, outlier_frac=0.0)
    W = oracle.decode_rows(m).astype(np.float64)
    m.centroids[:] = np.ldexp(m.centroids, -118)
    t = eng.upload_packed(m)
    X = np.full((M, cols), np.ldexp(1.0, 100), np.float32)
    X[1:] *= np.random.default_rng(M).standard_normal((M - 1, cols)).astype(np.float32)
    X = bf16_bits_to_f32(f32_to_bf16_bits(X)).reshape(M, cols)
    got = run_dev(eng, t, f32_to_bf16_bits(X), engine.DTYPE_BF16, M, engine.DTYPE_F32)
    t.free()
    want = np.ldexp(X.astype(np.float64) @ W.T, -118)
    rel = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
    assert rel.max() <= 4 * 2.0 ** -24, rel      # the sums' own error is 0.7 .. 0.9e-7; lost centroid bits gave 2^-15


@pytest.mark.parametrize("kind", ["cb4", "g64", "q8", "q4_0"])
@pytest.mark.parametrize("rows,cols,M", [
    (40, 600, 4), (2048, 1300, 3), (2049, 2600, 4), (40, 1500, 7), (40, 5000, 6), (70, 8200, 11), (4200, 3100, 16),
    (33, 12300, 9)])
def test_skinny_f32_forms(eng, kind, rows, cols, M):
    """f32 activations: half tiles of one and of several phases up to 2048 rows,
    and K ranges of one to several thousand columns above 8 tokens, plain and
    gated (silu(g) u: |silu'| <= 1.1)."""
    print(f"skinny f32 forms {kind} rows={rows} cols={cols} M={M}", flush=True)
    rows += rows & 1
    m = synth.make_q40(rows, cols, seed=6) if kind == "q4_0" else make(kind, rows, cols, seed=6)
    t = eng.upload_packed(m)
    X = (np.random.default_rng(cols).standard_normal((M, cols)) / cols ** 0.5).astype(np.float32)
    got = run_dev(eng, t, X, engine.DTYPE_F32, M, engine.DTYPE_F32)
    F = rows // 2
    xd, yd = eng.to_device(X), eng.alloc(M * F * 4)
    eng.ffn_glu_dev(t, xd.ptr, engine.DTYPE_F32, M, yd.ptr, engine.DTYPE_F32, F, engine.ACT_SILU, eng.stream)
    eng.synchronize()
    act = yd.download(np.float32, (M, F))
    for b in (xd, yd, t):
        b.free()
    W = oracle.decode_rows(m).astype(np.float64)
    want = X.astype(np.float64) @ W.T
    bound = (160 + cols / 128) * 2.0 ** -24 * (np.abs(X) @ np.abs(W).T)
    assert np.all(np.abs(got - want) <= bound)
    g, u = want[:, :F], want[:, F:]
    s = g / (1 + np.exp(-g))
    tol = 1.1 * bound[:, :F] * np.abs(u) + np.abs(s) * bound[:, F:] + 2.0 ** -20 * np.abs(s * u) + 1e-12
    assert np.all(np.abs(act - s * u) <= tol)


@pytest.mark.parametrize("rows,cols,M", [(8192, 2050, 11), (8201, 4097, 16), (12288, 2304, 12)])
def test_g64_all_of_k_in_one_range(eng, rows, cols, M):
    """g64 from 11 tokens and 8192 rows: all of K in several phases of one
    workgroup, the last one ragged; the file's bound."""
    print(f"g64 one range rows={rows} cols={cols} M={M}", flush=True)
    m = make("g64", rows, cols, seed=2)
    t = eng.upload_packed(m)
    xh = f32_to_bf16_bits(np.random.default_rng(M).standard_normal((M, cols)).astype(np.float32))
    X = bf16_bits_to_f32(xh).reshape(M, cols).astype(np.float64)
    got = run_dev(eng, t, xh, engine.DTYPE_BF16, M, engine.DTYPE_F32)
    t.free()
    W = oracle.decode_rows(m).astype(np.float64)
    assert np.all(np.abs(got - X @ W.T) <= (160 + cols / 128) * 2.0 ** -24 * (np.abs(X) @ np.abs(W).T))


FORMS = [(70, 544, 5, False), (70, 4160, 7, False), (4200, 300, 5, False), (40, 2600, 16, False), (40, 2600, 40, False),
         (70, 2100, 5, True), (4200, 700, 3, True), (70, 2600, 12, True), (32800, 288, 12, False)]


@pytest.mark.parametrize("kind", ["cb4", "g64", "q8", "q4_0"])
@pytest.mark.parametrize("rows,cols,M,f32", FORMS + [(67, 2047, 2, False), (33, 1031, 33, False)])
def test_skinny_single_products(eng, kind, rows, cols, M, f32):
    """One activation per token is not zero, at the first and last column and
    over the chunks between: an output is one product, of operands with all
    24 bits set where they have them (cb4's centroids, f32 activations), and may
    not miss the lowest of their three terms.  At most four roundings (the
    term sums, a scale, the result); products of the terms left out are below
    2^-24 of it, twice."""
    print(f"skinny single {kind} rows={rows} cols={cols} M={M} f32={f32}", flush=True)
    m = synth.make_q40(rows, cols, seed=3) if kind == "q4_0" else make(kind, rows, cols, seed=3)
    if kind == "cb4":
        m.centroids[:] = (m.centroids.view(np.uint32) | 0xFF).view(np.float32)
    t = eng.upload_packed(m)
    X = np.zeros((M, cols), np.float32)
    at = np.linspace(0, cols - 1, M).astype(int)
    x = 1 + np.random.default_rng(cols).random(M).astype(np.float32)
    X[np.arange(M), at] = (x.view(np.uint32) | 0xFF).view(np.float32) if f32 else bf16_bits_to_f32(f32_to_bf16_bits(x))
    got = run_dev(eng, t, X if f32 else f32_to_bf16_bits(X), engine.DTYPE_F32 if f32 else engine.DTYPE_BF16, M,
                  engine.DTYPE_F32)
    t.free()
    W = oracle.decode_rows(m)[:, at].astype(np.float64).T
    xs = X[np.arange(M), at].astype(np.float64)[:, None]
    # a residual is a product of its own: its column's weight is a sum
    mag = np.abs(W * xs)
    if kind == "cb4":
        mag = mag + 0.1 * np.abs(xs) * np.isin(at, m.outliers_packed & 0xFFFF)[:, None]
    bound = 6 * 2.0 ** -24 * mag
    assert np.all(np.abs(got - W * xs) <= bound)
    # ... and the bound shows a lost third term
    if kind == "cb4" or f32:
        lost = (X.view(np.uint32) & 0xFFFFFF00).view(np.float32)[np.arange(M), at].astype(np.float64)[:, None] if f32 else \
            xs * (1 - 2.0 ** -17)
        assert np.any(np.abs(W * lost - W * xs) > bound)


def _nibbles(b):
    return np.stack([b & 15, b >> 4], -1).reshape(-1)


def _nonfinite(m, kind):
    """Inf and NaN in tables and scales of a few rows; returns the rows that
    have any.  Padded columns keep finite entries; cb4's shared table has its Inf
    at entry 0, which no other row's columns hold."""
    rows, cols = m.rows, m.cols
    if kind == "cb4":
        q = _nibbles(m.packed_words.view(np.uint8)).reshape(rows, -1)
        q[q == 0], q[q == 7] = 1, 8
        q[2, 5], q[3, cols - 1], q[6, cols // 2] = 0, 0, 7
        b = q.reshape(-1, 2)
        m.packed_words[:] = np.ascontiguousarray(b[:, 0] | b[:, 1] << 4).astype(np.uint8).view(np.uint32)
        m.centroids[0], m.centroids[7] = np.inf, np.nan
        s = m.scales_f16.reshape(rows, -1)
        s[9, 0], s[11, (cols - 1) // 128] = 0x7C00, 0x7E00
        return [2, 3, 6, 9, 11]
    if kind == "g64":
        q = _nibbles(m.idx).reshape(rows, -1)
        last = (cols - 1) // 64
        q[q == 3], q[:, cols:] = 4, 1
        q[2, 5], q[3, cols - 1], q[6, cols - 1] = 3, 3, 3
        b = q.reshape(-1, 2)
        m.idx[:] = (b[:, 0] | b[:, 1] << 4).reshape(m.idx.shape)
        L = m.lut_f16.reshape(rows, -1, 16)
        L[2, 0, 3], L[3, last, 3], L[6, last, 3], L[9, last, 3] = 0x7C00, 0xFC00, 0x7E00, 0x7C00
        return [2, 3, 6]
    if kind == "q8":
        s = m.blocks.reshape(rows, -1, 34)[:, :, :2].copy().view(np.uint16)[:, :, 0]
    else:
        s = m.scales_f16.reshape(rows, -1)
    s[2, 0], s[3, (cols - 1) // 32], s[6, (cols - 1) // 64] = 0x7C00, 0xFC00, 0x7E00
    if kind == "q8":
        m.blocks.reshape(rows, -1, 34)[:, :, :2] = np.ascontiguousarray(s)[:, :, None].view(np.uint8)
        m.blocks.reshape(rows, -1, 34)[2, 0, 2:] = 5
    else:
        m.qs_words.reshape(rows, -1, 4)[2, 0] = 0x9B9B9B9B
    return [2, 3, 6]


@pytest.mark.parametrize("kind", ["cb4", "g64", "q8", "q4_0"])
@pytest.mark.parametrize("rows,cols,M,f32", FORMS)
def test_skinny_nonfinite_tables_and_scales(eng, kind, rows, cols, M, f32):
    """Inf and NaN in codebooks, centroids and scales reach the outputs that
    the reference's loops give them to, and no others."""
    print(f"skinny nonfinite weights {kind} rows={rows} cols={cols} M={M} f32={f32}", flush=True)
    m = synth.make_q40(rows, cols, seed=12) if kind == "q4_0" else make(kind, rows, cols, seed=12)
    bad = _nonfinite(m, kind)
    t = eng.upload_packed(m)
    X = np.random.default_rng(M).standard_normal((M, cols)).astype(np.float32)
    X[0], X[1, ::3] = np.abs(X[0]) + 0.5, 0
    xh = X if f32 else f32_to_bf16_bits(X)
    Xq = X if f32 else bf16_bits_to_f32(xh).reshape(M, cols)
    got = run_dev(eng, t, xh, engine.DTYPE_F32 if f32 else engine.DTYPE_BF16, M, engine.DTYPE_F32)
    t.free()
    with np.errstate(all="ignore"):
        pat = oracle.gemm(m, Xq, threads=8) if M > 8 else np.stack([oracle.gemv(m, x, threads=8) for x in Xq])
        W = oracle.decode_rows(m).astype(np.float64)
    assert not np.isfinite(pat[0, bad]).any() and np.isinf(pat[0, bad]).any()
    assert np.array_equal(np.isnan(got), np.isnan(pat)) and np.array_equal(np.isinf(got), np.isinf(pat))
    both = np.isinf(pat)
    assert np.array_equal(np.sign(got[both]), np.sign(pat[both]))
    good = np.setdiff1d(np.arange(rows), bad)
    W, Xf = W[good], Xq.astype(np.float64)
    assert np.all(np.abs(got[:, good] - Xf @ W.T) <= (160 + cols / 128) * 2.0 ** -24 * (np.abs(Xf) @ np.abs(W).T))
