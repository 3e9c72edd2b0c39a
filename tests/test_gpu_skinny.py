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
