"""Inputs with more rows, or more elements, than one round of a kernel's grid takes: the workgroups
that walk on to a second row (and reuse their shared memory for it) and the interpreter's second
tile. The input repeats a block of rows, so every repetition has the block's results."""
import numpy as np
import pytest

from synaptik_amd.native import HipProgram
from synaptik_amd.program import ProgramBuilder

pytestmark = pytest.mark.gpu

GRID = 1 << 20  # workgroups a row kernel's grid holds at most


def _repeat(ctx, block, rows):
    buf = ctx.buffer(rows * block[0].nbytes)
    for r in range(0, rows, len(block)):
        buf.upload(block[:rows - r], r * block[0].nbytes)
    return buf


def _rows(buf, first, count, width):
    return buf.download(np.float32, count * width, 4 * first * width).reshape(count, width)


def _spans(R):
    return [(0, 64), (GRID - 32, 64), (R - 64, 64)]


def _run(ctx, pb, ins, outs):
    bufs = [ctx.buffer(s.nbytes) for s in outs]
    prog = HipProgram(ctx, pb.image())
    prog.run(ins, bufs)
    prog.close()
    return bufs


def test_row_reductions(ctx):
    R, C = GRID + 70, 2045
    print(f"[many rows] reductions {R}x{C}", flush=True)
    rng = np.random.default_rng(1)
    block = rng.standard_normal((8191, C)).astype(np.float32)
    block[3, 7], block[4, :] = np.nan, -np.abs(block[4])
    block[4, 9], block[5, 11] = -0.0, np.inf
    pb = ProgramBuilder()
    sx, outs = pb.input(R * C), [pb.output(R) for _ in range(3)]
    for o, kind in zip(outs, ("sum", "max", "lse")):
        pb.row_reduce(sx, o, R, C, kind)
    got = [b.download(np.float32, R) for b in _run(ctx, pb, [_repeat(ctx, block, R)], outs)]
    for o in got:  # the same bits in every repetition
        for r in range(0, R, len(block)):
            assert np.array_equal(o[r:r + len(block)].view(np.uint32),
                                  o[:min(len(block), R - r)].view(np.uint32))
    d = block.astype(np.float64)
    ok = np.isfinite(d).all(1)
    mx = d.max(1)
    assert np.isnan([o[3] for o in got]).all() and got[1][5] == got[2][5] == np.inf
    assert np.array_equal(got[1][:8191][ok], mx[ok].astype(np.float32))
    # binary64 sums rounded once; exponentials of half a unit, and the logarithm's rounding
    np.testing.assert_allclose(got[0][:8191][ok], d.sum(1)[ok], rtol=2e-7, atol=1e-12)
    lse = mx[ok] + np.log(np.exp(d[ok] - mx[ok, None]).sum(1))
    np.testing.assert_allclose(got[2][:8191][ok], lse, rtol=1e-6)


@pytest.mark.parametrize("R,C", [(4 * GRID + 70, 5), (GRID + 70, 2047)])
def test_softmax(ctx, R, C):
    print(f"[many rows] softmax {R}x{C}", flush=True)
    rng = np.random.default_rng(C)
    block = (2 * rng.standard_normal((16381, C))).astype(np.float32)
    block[2, 1], block[3, 0], block[4, :] = np.nan, -np.inf, 0.0
    pb = ProgramBuilder()
    sx, y, l, dx = pb.input(R * C), pb.output(R * C), pb.output(R), pb.output(R * C)
    pb.softmax(sx, y, R, C, lse=l)
    pb.softmax_bwd(y, sx, dx, R, C)
    by, bl, bd = _run(ctx, pb, [_repeat(ctx, block, R)], [y, l, dx])
    lse = bl.download(np.float32, R)
    for r in range(0, R, len(block)):
        assert np.array_equal(lse[r:r + len(block)], lse[:min(len(block), R - r)], equal_nan=True)
    assert np.isnan(lse[2]) and np.isfinite(lse[4])
    for first, n in _spans(R) + [(4 * GRID - 32, 64)] * (R > 4 * GRID):
        x = block[np.arange(first, first + n) % len(block)].astype(np.float64)
        ok = np.isfinite(x).all(1)
        p = np.exp(x - x.max(1, keepdims=True))
        p /= p.sum(1, keepdims=True)
        got, grad = _rows(by, first, n, C), _rows(bd, first, n, C)
        assert np.array_equal(np.isnan(got).any(1), np.isnan(x).any(1))
        # one unit each of the exponential, the sum and the quotient, of x - max its rounding
        np.testing.assert_allclose(got[ok], p[ok], rtol=2e-6)
        x, p = x[ok], p[ok]
        want = p * (x - (x * p).sum(1, keepdims=True))
        assert np.all(np.abs(grad[ok] - want) <= 4e-6 * p * (np.abs(x) + 4.0))


def test_index_cross_entropy(ctx):
    R, C = GRID + 70, 1025
    print(f"[many rows] cross-entropy {R}x{C}", flush=True)
    rng = np.random.default_rng(2)
    block = rng.standard_normal((16381, C)).astype(np.float32)
    y = rng.integers(0, C, len(block))
    y[rng.random(len(y)) < 0.5] = -1
    target = np.resize(y, R).astype(np.int32)
    pb = ProgramBuilder()
    sx, sy = pb.input(R * C), pb.input(R, "i32")
    loss, grad = pb.output(1), pb.output(R * C)
    pb.index_ce(sx, sy, loss, R, C, grad=grad, ignore_index=-1)
    bl, bg = _run(ctx, pb, [_repeat(ctx, block, R), ctx.upload(target)], [loss, grad])
    x = block.astype(np.float64)
    lse = np.log(np.exp(x).sum(1))
    rows = np.where(y >= 0, lse - x[np.arange(len(y)), np.maximum(y, 0)], 0.0)
    count = int((target >= 0).sum())
    want = np.resize(rows, R).sum() / count
    assert abs(float(bl.download(np.float32, 1)[0]) - want) <= 1e-6 * want
    for first, n in _spans(R):
        i = np.arange(first, first + n) % len(block)
        p = np.exp(x[i] - lse[i, None])
        p[np.arange(n), np.maximum(y[i], 0)] -= 1.0
        p[y[i] < 0] = 0.0
        np.testing.assert_allclose(_rows(bg, first, n, C), p / count, rtol=2e-6, atol=2e-7 / count)


def test_chain_of_two_rounds(ctx):
    """65536 workgroups of 1024 elements are one round of the interpreter's grid."""
    C = 1001
    R = 65536 * 1024 // C + 5
    print(f"[many rows] chain {R}x{C}", flush=True)
    rng = np.random.default_rng(3)
    x = rng.standard_normal((R, C), dtype=np.float32)
    row, col = rng.standard_normal(C).astype(np.float32), rng.standard_normal(R).astype(np.float32)
    pb = ProgramBuilder()
    ins = [pb.input(v.size) for v in (x, row, col)]
    out = pb.output(R * C)
    code = [("load", 0, 0, 0, 0, 0.0), ("load", 1, 1, 0, 0, 0.0), ("sub", 2, 0, 1, 0, 0.0),
            ("load", 3, 2, 0, 0, 0.0), ("mul", 2, 2, 3, 0, 0.0), ("store", 0, 2, 0, 0, 0.0)]
    pb.pointwise(R, C, ins, [out], code, modes=["full", "row", "col"])
    (b,) = _run(ctx, pb, [ctx.upload(v) for v in (x, row, col)], [out])
    assert np.array_equal(b.download(np.float32, R * C).reshape(R, C), (x - row) * col[:, None])
