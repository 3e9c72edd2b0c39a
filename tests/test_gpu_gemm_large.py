"""The large-tile dense kernel (gemm_dense3.hip) with f32 activations and below
96 output tiles, at the edges of its ranges: tiles that end inside the batch and
the rows, one and several K ranges, 4- and 8-wave workgroups, columns that end
inside a K tile.  Reference: the decoded weights (bit-exact, the oracle) times
the activations in 64 bits.

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
