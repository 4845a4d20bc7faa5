"""Programs that end without the status publication (no step touches the status word): every way to
run them succeeds with the right result, also right after a run of another program that flagged the
word (runtime.cpp, Program::publishes)."""
import numpy as np
import pytest

from synaptik_amd.native import HipIndexError, HipProgram
from synaptik_amd.program import ProgramBuilder

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["graph", "direct", "profiled", "async", "static"])
def test_run_without_publication(ctx, mode):
    R, C = 48, 33
    fb = ProgramBuilder()
    fx, ft, fl = fb.input(R * C), fb.input(R, "i64"), fb.output(1)
    fb.index_ce(fx, ft, fl, R, C)
    flagging = HipProgram(ctx, fb.image())
    pb = ProgramBuilder()
    sx, h, sy = pb.input(R * C), pb.internal(R * C), pb.output(R)
    pb.softmax(sx, h, R, C)
    pb.row_reduce(h, sy, R, C, "max")
    prog = HipProgram(ctx, pb.image())
    prog.set_graph_mode(mode == "graph")
    prog.set_profiling(mode == "profiled")
    rng = np.random.default_rng(17)
    bad = ctx.upload(np.full(R, C, np.int64))
    by, bl = ctx.buffer(4 * R), ctx.buffer(4)
    for _ in range(4):
        x = rng.standard_normal((R, C)).astype(np.float32)
        bx = ctx.upload(x)
        with pytest.raises(HipIndexError):
            (flagging.run_static if mode == "static" else flagging.run)([bx, bad], [bl])
        if mode == "async":
            prog.run_async([bx], [by])
            prog.wait()
        else:
            (prog.run_static if mode == "static" else prog.run)([bx], [by])
        e = np.exp((x - x.max(1, keepdims=True)).astype(np.float64))
        want = (e / e.sum(1, keepdims=True)).max(1)
        # the maximum's exponential is exactly 1: the sum's and the quotient's rounding, with the
        # other exponentials of at most one unit
        assert np.all(np.abs(by.download(np.float32, R) - want) <= 3 * 2.0 ** -23 * want)
    prog.close()
    flagging.close()


@pytest.mark.parametrize("mode", ["graph", "direct", "profiled", "async", "static"])
def test_run_of_steps_without_elements(ctx, mode):
    """Nothing but steps of extent zero: such a program still publishes, so that its run, and its
    captured graph, hold a launch. The outputs stay as they were."""
    pb = ProgramBuilder()
    x, y, z = pb.input(8), pb.output(8), pb.output(8)
    pb.softmax(x, y, 0, 8)
    pb.row_reduce(x, y, 0, 8, "max")
    pb.colsum(x, y, 1, 0, ldx=8)
    pb.gemm(x, x, y, 0, 2, 4)
    pb.softmax_bwd(x, x, z, 4, 0)
    pb.lse_bwd(x, x, z, 0, 4)
    pb.pointwise(0, 4, [x], [z], [("load", 0, 0, 0, 0, 0.0), ("neg", 1, 0, 0, 0, 0.0),
                                  ("store", 0, 1, 0, 0, 0.0)])
    pb.transpose(x, z, 0, 4)
    pb.fill(z, 0)
    pb.copy(x, z, 0)
    prog = HipProgram(ctx, pb.image())
    prog.set_graph_mode(mode == "graph")
    prog.set_profiling(mode == "profiled")
    data = np.arange(8, dtype=np.float32)
    bx, by, bz = ctx.upload(data + 10), ctx.upload(data), ctx.upload(-data)
    for _ in range(3):
        if mode == "async":
            prog.run_async([bx], [by, bz])
            prog.wait()
        else:
            (prog.run_static if mode == "static" else prog.run)([bx], [by, bz])
        assert np.array_equal(by.download(np.float32, 8), data)
        assert np.array_equal(bz.download(np.float32, 8), -data)
    prog.close()
