"""exp, tanh and the logistic function as the device evaluates them (fexp64.h; its quotient is formed
from a hardware reciprocal, which the host test does not run) against numpy's binary64 functions
rounded once, over every 1021st binary32 pattern."""
import numpy as np
import pytest

from synaptik_amd.program import ProgramBuilder
from tests.gpu_helpers import run_program

pytestmark = pytest.mark.gpu


def _logistic(x):
    e = np.exp(-np.abs(x))
    return np.where(x >= 0, 1.0, e) / (1.0 + e)


@pytest.mark.parametrize("op,function", [("exp", np.exp), ("tanh", np.tanh), ("sigmoid", _logistic)])
def test_binary64_evaluations_round_like_numpy(ctx, op, function):
    print(f"[fexp64] {op}", flush=True)
    t = np.arange(0, 1 << 32, 1021, dtype=np.uint64).astype(np.uint32).view(np.float32)
    pb = ProgramBuilder()
    x, o = pb.input(t.size), pb.output(t.size)
    pb.pointwise(1, t.size, [x], [o], [("load", 0, 0, 0, 0, 0.0), (op, 1, 0, 0, 0, 0.0),
                                       ("store", 0, 1, 0, 0, 0.0)])
    (got,) = run_program(ctx, pb, [t], [o])
    with np.errstate(all="ignore"):
        want = function(t.astype(np.float64)).astype(np.float32)
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan)
    zero = want == 0
    assert np.array_equal(np.signbit(got[zero]), np.signbit(want[zero]))
    g, w = (v[~nan].view(np.int32).astype(np.int64) for v in (got, want))
    g, w = (np.where(v < 0, -(v & 0x7fffffff), v) for v in (g, w))
    # both sides are a few units of 2^-52 from the exact value: they round apart only where it lies
    # that close to a tie, about one argument in 10^7
    assert np.abs(g - w).max() <= 1 and np.count_nonzero(g != w) <= 4
