"""MSE at the edges of its launch forms (one block of 256 threads up to 1024 elements, one of 1024 up
to 16384, two launches beyond) against the exact-reduction oracle."""
import numpy as np
import pytest

from oracle import oracle
from synaptik_amd.program import ProgramBuilder
from tests.gpu_helpers import run_program

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("reduction", ["mean", "sum"])
@pytest.mark.parametrize("n", [1, 1023, 1024, 1025, 4097, 16383, 16384, 16385])
def test_mse(ctx, n, reduction):
    print(f"[mse] n={n} {reduction}", flush=True)
    rng = np.random.default_rng(n)
    p, t = (rng.standard_normal(n).astype(np.float32) for _ in range(2))
    pb = ProgramBuilder()
    sp, st, sl, sg = pb.input(n), pb.input(n), pb.output(1), pb.output(n)
    pb.mse(sp, st, sl, n, grad=sg, g=0.7, reduction=reduction)
    loss, grad = run_program(ctx, pb, [p, t], [sl, sg])
    d = (p - t).astype(np.float32)
    total = np.float64((d * d).astype(np.float64).sum())
    want = total if reduction == "sum" else total / n
    # binary64 sums of the rounded squares, rounded once (the mean twice)
    assert abs(loss[0] - want) <= 2.0 ** -23 * want
    assert np.array_equal(grad, oracle.mse_grad(p, t, 0.7, reduction))
