"""The chain interpreter at the places where its index arithmetic can go wrong: widths around a
group of four, groups that span rows, the last partial group, and chains of both broadcast kinds,
against numpy in the same binary32 operations. (More than one round of the grid: test_many_rows_gpu.)"""
import numpy as np
import pytest

from synaptik_amd.program import ProgramBuilder
from tests.gpu_helpers import run_program

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R,C", [(1, 1), (7, 1), (1, 7), (5, 2), (5, 3), (9, 4), (33, 5), (3, 4099),
                                 (2700, 1001), (11000, 257), (1500000, 3)])
def test_broadcast_chain(ctx, R, C):
    print(f"[pointwise] {R}x{C}", flush=True)
    rng = np.random.default_rng(R + C)
    x, y = (rng.standard_normal((R, C)).astype(np.float32) for _ in range(2))
    row, col = rng.standard_normal(C).astype(np.float32), rng.standard_normal(R).astype(np.float32)
    sc = rng.standard_normal(1).astype(np.float32)
    pb = ProgramBuilder()
    ins = [pb.input(v.size) for v in (x, y, row, col, sc)]
    o0, o1 = pb.output(R * C), pb.output(R * C)
    code = [("load", 0, 0, 0, 0, 0.0), ("load", 1, 2, 0, 0, 0.0), ("sub", 2, 0, 1, 0, 0.0),
            ("load", 3, 3, 0, 0, 0.0), ("mul", 2, 2, 3, 0, 0.0), ("store", 0, 2, 0, 0, 0.0),
            ("load", 4, 1, 0, 0, 0.0), ("load", 5, 4, 0, 0, 0.0), ("add", 4, 4, 5, 0, 0.0),
            ("max", 4, 4, 2, 0, 0.0), ("store", 1, 4, 0, 0, 0.0)]
    pb.pointwise(R, C, ins, [o0, o1], code, modes=["full", "full", "row", "col", "scalar"])
    a, b = run_program(ctx, pb, [x, y, row, col, sc], [o0, o1])
    want = (x - row[None, :]) * col[:, None]
    assert np.array_equal(a.reshape(R, C), want)
    assert np.array_equal(b.reshape(R, C), np.maximum(y + sc[0], want))


@pytest.mark.parametrize("n", [1, 2, 3, 5, 1023, 2560 * 1024 + 3, 3 * 2560 * 1024 + 1])
def test_long_chain(ctx, n):
    """No broadcast: the last group and the last workgroup partly filled."""
    rng = np.random.default_rng(n)
    x, y = (rng.standard_normal(n).astype(np.float32) for _ in range(2))
    pb = ProgramBuilder()
    sx, sy, o = pb.input(n), pb.input(n), pb.output(n)
    code = [("load", 0, 0, 0, 0, 0.0), ("load", 1, 1, 0, 0, 0.0), ("gt", 2, 0, 1, 0, 0.0),
            ("where", 3, 0, 1, 2, 0.0), ("const", 4, 0, 0, 0, 0.5), ("mul", 3, 3, 4, 0, 0.0),
            ("neg", 3, 3, 0, 0, 0.0), ("store", 0, 3, 0, 0, 0.0)]
    pb.pointwise(1, n, [sx, sy], [o], code)
    (got,) = run_program(ctx, pb, [x, y], [o])
    assert np.array_equal(got, -(np.where(x > y, x, y) * np.float32(0.5)))
