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


@pytest.mark.parametrize("fmt,lo,e8", [(4, True, None), (4, False, None), (7, True, (114, 140)), (7, False, (100, 150))])
@pytest.mark.parametrize("rows", [[65, 129], [128, 40], [97, 64, 1]])
def test_grouped_gemm_split_k(session, fmt, lo, e8, rows):
    """The same with K split in both launches (17 and 9 quads, few enough
    blocks to leave the chip idle): tall and short tiles' gate/up partials
    through the reduction, and output widths (1040, 2064) that end inside a
    block."""
    rng = np.random.default_rng(1900 + fmt + 10 * lo + rows[0])
    D, I = 2064, 1040
    layer = Layer(rng, fmt, D, I, len(rows), e8_range=e8 or (119, 123))
    hs = layer.upload(session)
    x = rng.standard_normal((sum(rows), D)).astype(np.float32) if lo else rand_x(rng, sum(rows), D)
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


def upload_dense(session, rng, fmt, half, O, I):
    """(handle, group size, dequantized weights, oracle product)."""
    if fmt == 7:
        q, sc = rand_mxfp4(rng, O, I)
        return session.upload_mxfp4(q, sc, I, O), 0, deq_mxfp4(q, sc, I), lambda x: cref.matmul_mxfp4(x, q, sc, O, I)
    q, sc = rand_i4(rng, O, I, 32, fp16_scales=half)
    return (session.upload(q, sc, 4, I, O, 32), 32, deq_i4(q, sc, I, 32),
            lambda x: cref.matmul_i4_grouped(x, q, sc, O, I, 32))


@pytest.mark.parametrize("fmt,half,O,I,S", [
    (4, True, 4096, 14336, 18),     # one short tile, K split
    (4, False, 2064, 7184, 200),    # f32 scales, tall tiles, K split, ragged block and columns
    (7, True, 4112, 4112, 194),     # MXFP4, a short tile of two rows behind a tall one
    (4, True, 14336, 1040, 130),    # blocks enough for the chip
    (7, False, 528, 128, 100),      # one quad of K: every prefetch past the end is clamped
    (4, False, 528, 256, 97),       # two
])
def test_dense_rows_on_the_gemm(session, monkeypatch, fmt, half, O, I, S):
    """Dense matrices of more rows than a GEMV batch tile, pinned to the GEMM:
    the same product, also on a second call of one row less."""
    monkeypatch.setenv("COLI_HIP_GEMV", "gemm")
    rng = np.random.default_rng(O + S)
    h, gs, deq, product = upload_dense(session, rng, fmt, half, O, I)
    x = rng.standard_normal((S, I)).astype(np.float32)
    try:
        got = {s: session.matmul(h, x[:s], fmt, I, O, gs) for s in (S, S - 1)}
    finally:
        session.free(h)
    ref = product(x)
    mag = magnitude(x, deq)
    for s, y in got.items():
        assert rel_err(y, ref[:s], mag[:s]).max() <= TOL
        assert (np.abs(y.astype(np.float64) - ref[:s]) / mag[:s]).max() <= 2 * err_bound(I)   # ref rounds as well


@pytest.mark.parametrize("fmt,O,I,S,gemm", [(4, 4096, 14336, 48, True), (4, 14336, 4096, 512, True),
                                            (7, 4096, 4096, 320, True), (4, 512, 2048, 512, False),
                                            (4, 4096, 14336, 16, False)])
def test_dense_kernel_pin(session, monkeypatch, fmt, O, I, S, gemm):
    """COLI_HIP_GEMV pins dense matrices of more than 16 rows to either
    kernel (their sums round in another order, so the results differ in
    bits), and the rule without it takes the one expected for shapes well
    inside its side."""
    rng = np.random.default_rng(3 * O + S)
    h, gs, _, _ = upload_dense(session, rng, fmt, True, O, I)
    x = rng.standard_normal((S, I)).astype(np.float32)
    got = {}
    try:
        for pin in ("tiles", "gemm", None):
            if pin:
                monkeypatch.setenv("COLI_HIP_GEMV", pin)
            else:
                monkeypatch.delenv("COLI_HIP_GEMV", raising=False)
            got[pin] = session.matmul(h, x, fmt, I, O, gs)
    finally:
        session.free(h)
    assert np.array_equal(got["tiles"], got["gemm"]) == (S <= 16)
    assert np.array_equal(got[None], got["gemm" if gemm else "tiles"])


@pytest.mark.parametrize("S", [24, 48, 130])
def test_idot_rows_on_the_gemm_bitwise(session, monkeypatch, S):
    """fmt=2 with int8 activations for many rows on the GEMM: every sum is an
    exact integer, so the K split changes nothing and the result is the
    reference's."""
    monkeypatch.setenv("COLI_HIP_GEMV", "gemm")
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


@pytest.mark.parametrize("fmt,half,O,I,S", [
    (4, True, 14336, 4096, 512),    # unsplit tall tiles, two running sums
    (4, False, 4112, 4112, 200),    # a K split, a short tile behind a tall one, ragged block and columns
    (7, True, 8192, 4096, 300),     # MXFP4
    (7, True, 14336, 4096, 40),     # MXFP4, a short tile
    (4, True, 14336, 4096, 40),     # a short tile
    (4, True, 14336, 7168, 128),    # several running sums a split
])
def test_dense_gemm_rounds_no_more_than_the_gemv(session, monkeypatch, fmt, half, O, I, S):
    """The GEMM's distance from the 64-bit product (2-norm over the whole
    result) is at most the GEMV's, whose waves each sum a share of K: as many
    running sums bound the growth of the f32 rounding the same way. 3 %: both
    norms are sums over at least 5e5 values' independent errors (0.2 %), and
    a last running sum of another length."""
    rng = np.random.default_rng(11 * O + S)
    h, gs, deq, _ = upload_dense(session, rng, fmt, half, O, I)
    x = rng.standard_normal((S, I)).astype(np.float32)
    err = {}
    try:
        for pin in ("tiles", "gemm"):
            monkeypatch.setenv("COLI_HIP_GEMV", pin)
            got = session.matmul(h, x, fmt, I, O, gs)
            if not err:
                exact = x.astype(np.float64) @ deq.T.astype(np.float64)
            err[pin] = np.linalg.norm(got - exact) / np.linalg.norm(exact)
    finally:
        session.free(h)
    assert err["gemm"] <= 1.03 * err["tiles"], err


def test_dense_gemm_row_tiles_in_several_launches(session, monkeypatch):
    """More rows than the scratch memory for the running sums holds at once
    (24 row tiles of this shape): each launch's rows land where they belong."""
    rng = np.random.default_rng(60)
    O, I, S = 14336, 4096, 3077
    h, gs, _, _ = upload_dense(session, rng, 4, True, O, I)
    x = rng.standard_normal((S, I)).astype(np.float32)
    try:
        monkeypatch.setenv("COLI_HIP_GEMV", "gemm")
        y = session.matmul(h, x, 4, I, O, gs)
        monkeypatch.setenv("COLI_HIP_GEMV", "tiles")
        ref = session.matmul(h, x, 4, I, O, gs)
    finally:
        session.free(h)
    d = np.linalg.norm(y - ref, axis=1) / np.linalg.norm(ref, axis=1)
    assert d.max() <= 1e-6   # (two results with 1.3e-7 of rounding each)


def test_tall_mxfp4_tiles_round_no_more_than_short_ones(session):
    """Eight members of 128 rows (tall tiles) against the same rows as sixteen
    members of 64 (short tiles); both accumulate folded scales in the MFMA. The
    distance from the 64-bit result does not grow. Enough blocks that
    gate/up runs without a K split."""
    rng = np.random.default_rng(77)
    D, I = 2048, 4096
    layer = Layer(rng, 7, D, I, 1)
    hs = layer.upload(session)
    x = rng.standard_normal((1024, D)).astype(np.float32)
    q, u, d = (deq_mxfp4(*layer.experts[0][i], K) for i, K in enumerate((D, D, I)))
    a = x.astype(np.float64) @ q.T
    exact = (a / (1 + np.exp(-a)) * (x.astype(np.float64) @ u.T)) @ d.T
    err = {}
    try:
        for rows in (128, 64):
            n = 1024 // rows
            y = session.expert_group([hs[0][0]] * n, [hs[0][1]] * n, [hs[0][2]] * n, [rows] * n, x)
            err[rows] = np.linalg.norm(y - exact) / np.linalg.norm(exact)
    finally:
        for t in hs[0]:
            session.free(t)
    assert err[128] <= 1.03 * err[64], err
