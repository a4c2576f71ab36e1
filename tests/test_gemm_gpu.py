"""The grouped GEMM's row tiles (short: up to 64 rows, tall: up to 128) and the
dense matrices' dispatch to it, against the oracle."""
import ctypes as C

import numpy as np
import pytest

from moe_ref import Layer, cref
from quant_util import deq_i4, deq_mxfp4, magnitude, rand_i4, rand_mxfp4, rand_x, rel_err

pytestmark = pytest.mark.gpu
TOL = 1e-3


def err_bound(K):
    """|error| over the magnitude sum: 22 significant bits of an activation,
    and one f32 rounding per 32-column group of the accumulation."""
    return 2.0 ** -22 + (K / 32 + 32) * 2.0 ** -24


@pytest.mark.parametrize("fmt,lo,e8", [(4, True, None), (4, False, None), (7, True, (114, 140)), (7, False, (114, 140)),
                                       (7, True, (100, 150))])
@pytest.mark.parametrize("rows", [[65, 96, 1], [97, 128, 64], [129, 193, 40], [256, 33, 80]])
def test_grouped_gemm_row_tiles(session, fmt, lo, e8, rows):
    """Members whose last row tile is short or tall and ends inside and at
    the edges of its 16- and 32-row blocks; ragged columns (400) and output
    blocks (17 and 25 row tiles of 16 and 8 a block)."""
    rng = np.random.default_rng(900 + fmt + 10 * lo + rows[0])
    D, I = 400, 272
    layer = Layer(rng, fmt, D, I, len(rows), e8_range=e8 or (119, 123))
    hs = layer.upload(session)
    n = sum(rows)
    x = rng.standard_normal((n, D)).astype(np.float32) if lo else rand_x(rng, n, D)
    try:
        y = session.expert_group([h[0] for h in hs], [h[1] for h in hs], [h[2] for h in hs], rows, x)
    finally:
        for h in hs:
            for t in h:
                session.free(t)
    o = 0
    for e, r in enumerate(rows):
        h, ref = layer.expert_forward(e, x[o:o + r])
        mag = np.abs(h.astype(np.float64)) @ layer.deq(layer.experts[e][2], I)
        assert rel_err(y[o:o + r], ref, mag).max() <= TOL
        o += r


@pytest.mark.parametrize("fmt,half,O,I,S", [
    (4, True, 4096, 14336, 17),     # one short tile, K split
    (4, False, 2064, 7184, 200),    # f32 scales, tall tiles, K split, ragged block and columns
    (7, True, 4112, 4112, 193),     # MXFP4, a short tile of one row behind a tall one
    (4, True, 14336, 1040, 129),    # blocks enough for the chip
])
def test_dense_rows_on_the_gemm(session, fmt, half, O, I, S):
    """pipe_gemm of more rows than a GEMV batch tile, where the GEMM is the
    faster: the same product, also on a second call of fewer rows."""
    rng = np.random.default_rng(O + S)
    if fmt == 7:
        q, sc = rand_mxfp4(rng, O, I)
        h, deq = session.upload_mxfp4(q, sc, I, O), deq_mxfp4(q, sc, I)
    else:
        q, sc = rand_i4(rng, O, I, 32, fp16_scales=half)
        h, deq = session.upload(q, sc, 4, I, O, 32), deq_i4(q, sc, I, 32)
    x = rng.standard_normal((S, I)).astype(np.float32)
    try:
        got = {s: session.matmul(h, x[:s], fmt, I, O, 0 if fmt == 7 else 32) for s in (S, S - 1)}
    finally:
        session.free(h)
    ref = cref.matmul_mxfp4(x, q, sc, O, I) if fmt == 7 else cref.matmul_i4_grouped(x, q, sc, O, I, 32)
    mag = magnitude(x, deq)
    for s, y in got.items():
        assert rel_err(y, ref[:s], mag[:s]).max() <= TOL
        assert (np.abs(y.astype(np.float64) - ref[:s]) / mag[:s]).max() <= 2 * err_bound(I)   # ref rounds as well


@pytest.mark.parametrize("S", [24, 130])
def test_idot_rows_on_the_gemm_bitwise(session, S):
    """fmt=2 with int8 activations for many rows: every sum is an exact
    integer, so the K split changes nothing and the result is the
    reference's."""
    rng = np.random.default_rng(S)
    O, I = 4096, 8192
    q, sc = rand_i4(rng, O, I, 0)
    x = rng.standard_normal((S, I)).astype(np.float32)
    h = session.upload(q, sc, 2, I, O)
    y = np.zeros((S, O), np.float32)
    try:
        f = C.POINTER(C.c_float)
        assert session.b.hip_matmul_i4_idot(h, y.ctypes.data_as(f), x.ctypes.data_as(f), S)
    finally:
        session.free(h)
    assert np.array_equal(y, cref.matmul_i4_idot(x, q, sc, O, I))
