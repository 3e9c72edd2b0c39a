"""The large-tile dense kernel (gemm_dense3.hip) with f32 activations, below 96
output tiles and with the gated epilogue, at the edges of its ranges: tiles that
end inside the batch and the rows, one and several K ranges, 4- and 8-wave
workgroups, columns that end inside a K tile.  Reference: the decoded weights
(bit-exact, the oracle) times the activations in 64 bits.

Bound: an f32 operand is split as hi + lo * 2^-11 in f16 (relative error at
most 2^-22, or 2^-36 of the row's largest entry for small ones) and the lo lo
product (2^-22) is left out, twice 2^-22 if both operands are split; an output
is a sum of at most K / 8 + 8 roundings of 2^-24 of the sum of the terms'
magnitudes (an MFMA adds 16 products in two halves).
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


def bound_of(X, W, cols):
    mag = np.abs(X) @ np.abs(W).T
    tiny = np.abs(X).max(1)[:, None] * np.abs(W).sum(1)[None] + np.abs(X).sum(1)[:, None] * np.abs(W).max(1)[None]
    return (3 * 2.0 ** -22 + (cols / 8 + 8) * 2.0 ** -24) * mag + 2.0 ** -36 * tiny


# rows, cols, tokens, f32 activations
@pytest.mark.parametrize("rows,cols,M,f32", [
    (4000, 600, 129, True), (2050, 4128, 192, True), (1500, 1030, 300, True), (6144, 520, 1030, True),
    (128, 300, 257, True), (6100, 2048, 72, False), (2100, 4130, 200, False)])
@pytest.mark.parametrize("kind", ["cb4", "g64", "q8", "q4_0"])
def test_large_tile_edges(eng, kind, rows, cols, M, f32):
    print(f"large tile {kind} rows={rows} cols={cols} M={M} f32={f32}", flush=True)
    m = synth.make_q40(rows, cols, seed=rows + M) if kind == "q4_0" else make(kind, rows, cols, seed=rows + M)
    t = eng.upload_packed(m)
    X = np.random.default_rng(cols + M).standard_normal((M, cols)).astype(np.float32)
    xh = X if f32 else f32_to_bf16_bits(X)
    Xq = (X if f32 else bf16_bits_to_f32(xh).reshape(M, cols)).astype(np.float64)
    eng.set_gemm_path(engine.GEMM_PANEL)
    try:
        got = run_dev(eng, t, xh, engine.DTYPE_F32 if f32 else engine.DTYPE_BF16, M, engine.DTYPE_F32)
    finally:
        eng.set_gemm_path(engine.GEMM_AUTO)
    W = oracle.decode_rows(m).astype(np.float64)
    err, bound = np.abs(got - Xq @ W.T), bound_of(Xq, W, cols)
    assert np.all(err <= bound), float((err / bound).max())
    t.free()


@pytest.mark.parametrize("rows,cols,M", [(4000, 600, 129), (6144, 520, 1030), (2050, 4128, 192)])
@pytest.mark.parametrize("kind", ["cb4", "g64", "q8", "q4_0"])
def test_large_tile_f32_inf_rows(eng, kind, rows, cols, M):
    """f32 activations with an Inf, or Infs of both signs, beside entries of
    1e10, and a NaN: the reference's pattern of Inf and NaN outputs; the other
    rows keep the file's bound."""
    print(f"large tile f32 inf {kind} rows={rows} cols={cols} M={M}", flush=True)
    m = synth.make_q40(rows, cols, seed=8) if kind == "q4_0" else make(kind, rows, cols, seed=8)
    t = eng.upload_packed(m)
    X = np.random.default_rng(M).standard_normal((M, cols)).astype(np.float32)
    X[3] *= np.float32(1e10)
    X[3, 17], X[M - 1, cols - 5], X[7, 0], X[7, cols - 1], X[9, cols // 2] = np.inf, -np.inf, np.inf, -np.inf, np.nan
    eng.set_gemm_path(engine.GEMM_PANEL)
    try:
        got = run_dev(eng, t, X, engine.DTYPE_F32, M, engine.DTYPE_F32)
    finally:
        eng.set_gemm_path(engine.GEMM_AUTO)
    t.free()
    sel = [3, 7, 9, M - 1]
    with np.errstate(all="ignore"):
        pat = oracle.gemm(m, X[sel], threads=8)
    y = got[sel]
    assert np.array_equal(np.isnan(y), np.isnan(pat)) and np.array_equal(np.isinf(y), np.isinf(pat))
    both = np.isinf(pat)
    assert both.any() and np.array_equal(np.sign(y[both]), np.sign(pat[both]))
    fin = np.setdiff1d(np.arange(M), sel)
    Xf, W = X[fin].astype(np.float64), oracle.decode_rows(m).astype(np.float64)
    assert np.all(np.abs(got[fin] - Xf @ W.T) <= bound_of(Xf, W, cols))


# Gated [gate; up] calls in one K range: batch and outputs that end inside a
# tile, output counts that are and are not multiples of 8 pieces, 4- and 8-wave
# workgroups and 256 x 192 tiles.  Bound: an output is act(g) u with g and u
# within B of the exact sums; |act'| <= 1.13 and |act(g)| <= |g| for both
# activations; 2^-18 of the result and 2^-20 |g u| for expf, tanh and
# 1 + tanh of a negative g.  bf16 outputs are the f32 outputs' rounding.
@pytest.mark.parametrize("n_ff,cols,M", [(6144, 520, 256), (6160, 200, 257), (9216, 320, 1050), (3072, 1030, 1000),
                                         (2064, 640, 1999)])
@pytest.mark.parametrize("kind", ["cb4", "g64", "q8", "q4_0"])
def test_gated_epilogue_edges(eng, kind, n_ff, cols, M):
    print(f"gated {kind} n_ff={n_ff} cols={cols} M={M}", flush=True)
    seed = n_ff + M
    m = synth.make_q40(2 * n_ff, cols, seed=seed) if kind == "q4_0" else make(kind, 2 * n_ff, cols, seed=seed)
    t = eng.upload_packed(m)
    xh = f32_to_bf16_bits(np.random.default_rng(seed).standard_normal((M, cols)).astype(np.float32))
    xd = eng.to_device(xh)
    sel = np.unique(np.r_[0:2, 31:34, M // 2, M - 18:M])
    X = bf16_bits_to_f32(xh).reshape(M, cols)[sel].astype(np.float64)
    W = oracle.decode_rows(m).astype(np.float64)
    z, B = X @ W.T, bound_of(X, W, cols)
    g, u, Bg, Bu = z[:, :n_ff], z[:, n_ff:], B[:, :n_ff], B[:, n_ff:]
    for activation in (engine.ACT_SILU, engine.ACT_GELU_TANH):
        out = {}
        for dt, np_dt, sz in ((engine.DTYPE_F32, np.float32, 4), (engine.DTYPE_BF16, np.uint16, 2)):
            ad = eng.alloc(M * n_ff * sz)
            eng.ffn_glu_dev(t, xd.ptr, engine.DTYPE_BF16, M, ad.ptr, dt, n_ff, activation, eng.stream)
            eng.synchronize()
            out[dt] = ad.download(np_dt, (M, n_ff))
            ad.free()
        if activation == engine.ACT_SILU:
            want = g / (1 + np.exp(-g)) * u
        else:
            want = 0.5 * g * (1 + np.tanh(0.7978846 * (g + 0.044715 * g ** 3))) * u
        bound = (1.13 * (np.abs(u) + Bu) * Bg + np.abs(g) * Bu + 2.0 ** -18 * np.abs(want) +
                 2.0 ** -20 * np.abs(g * u) + 1e-30)
        err = np.abs(out[engine.DTYPE_F32][sel] - want)
        assert np.all(err <= bound), (activation, float((err / bound).max()))
        assert np.array_equal(out[engine.DTYPE_BF16].ravel(), f32_to_bf16_bits(out[engine.DTYPE_F32]).ravel())
    xd.free()
    t.free()
