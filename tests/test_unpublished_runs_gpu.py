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
