"""Row, column and whole-tensor reductions at the edges of their kernels' widths: one wave a row up
to 2044 columns, one workgroup of 256 up to 8188, of 512 up to 16380 and of 1024 up to 32764, re-read
beyond; rows whose start is not 16-byte aligned; column sums whose last lane holds one to three columns."""
import numpy as np
import pytest

from oracle import oracle
from synaptik_amd.program import ProgramBuilder
from tests.gpu_helpers import run_program

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C", [1, 3, 65, 252, 253, 508, 509, 1001, 1020, 1021, 2044, 2045, 4092, 4093, 8188, 8189, 16380, 16381, 20003, 32764, 32767, 70001])
def test_row_reductions(ctx, C):
    print(f"[row_reduce] C={C}", flush=True)
    R = 9
    rng = np.random.default_rng(C)
    x = (rng.standard_normal((R, C)) * 3).astype(np.float32)
    x[1, C // 2] = np.nan
    x[2, :] = -np.inf
    x[3, C - 1] = np.inf
    x[4, :] = -0.0
    if C > 1:
        x[4, C - 1] = 0.0
    pb = ProgramBuilder()
    sx = pb.input(R * C)
    outs = [pb.output(R) for _ in range(4)]
    for o, kind in zip(outs, ("sum", "mean", "max", "lse")):
        pb.row_reduce(sx, o, R, C, kind)
    total, mean, mx, lse = run_program(ctx, pb, [x], outs)
    want_max, want_lse = oracle.max_rows(x), oracle.logsumexp_rows(x)
    assert np.array_equal(np.isnan(mx), np.isnan(want_max))
    ok = ~np.isnan(want_max)
    assert np.array_equal(mx[ok].view(np.uint32), want_max[ok].view(np.uint32))
    for got, want, tol in ((lse, want_lse, 1e-6),
                           (total, np.array([oracle.exact_sum(r) for r in x], np.float32), 2e-7),
                           (mean, np.array([oracle.exact_mean(r) for r in x], np.float32), 2e-7)):
        assert np.array_equal(np.isnan(got), np.isnan(want))
        inf = np.isinf(want)
        assert np.array_equal(got[inf], want[inf])
        fin = np.isfinite(want)
        # binary64 sums rounded once: within one unit of the exact sum's rounding
        np.testing.assert_allclose(got[fin], want[fin], rtol=tol, atol=0)


@pytest.mark.parametrize("R,N", [(40000, 64), (40000, 65), (40001, 100), (33000, 255), (32, 300),
                                 (33, 300), (1, 1000), (32, 301), (48, 301), (49, 301), (2, 262143),
                                 (48, 262145), (4, 262145), (5, 262145)])
def test_column_sums_at_the_dispatch_edges(ctx, R, N):
    """4-byte lanes up to 64 columns, for up to 48 unaligned rows of at most 2^18 columns and for up to
    four of any width; four columns a lane beyond, on four waves up to 32 rows."""
    test_column_sums(ctx, R, N, 0)


@pytest.mark.parametrize("R,N", [(70, 257), (1000, 1001), (17, 1023), (5000, 258), (3, 4099)])
@pytest.mark.parametrize("pad", [0, 3])
def test_column_sums(ctx, R, N, pad):
    print(f"[colsum] {R}x{N} pad={pad}", flush=True)
    rng = np.random.default_rng(R + N)
    x = np.full((R, N + pad), np.nan, np.float32)
    x[:, :N] = rng.standard_normal((R, N)).astype(np.float32)
    pb = ProgramBuilder()
    sx = pb.input(x.size)
    so, sm = pb.output(N), pb.output(N)
    pb.colsum(sx, so, R, N, ldx=N + pad)
    pb.colsum(sx, sm, R, N, ldx=N + pad, mean=True)
    got, mean = run_program(ctx, pb, [x], [so, sm])
    np.testing.assert_array_max_ulp(got, oracle.colsum(np.ascontiguousarray(x[:, :N])), maxulp=1)
    exact = x[:, :N].astype(np.float64).sum(0) / R
    np.testing.assert_allclose(mean, exact, rtol=2e-7, atol=1e-12)


@pytest.mark.parametrize("n", [1, 3, 4, 1025, 4 * 256 * 1024 * 4 + 7])
def test_whole_sum(ctx, n):
    rng = np.random.default_rng(n)
    x = rng.standard_normal(n).astype(np.float32)
    pb = ProgramBuilder()
    sx, so, sm = pb.input(n), pb.output(1), pb.output(1)
    pb.reduce_all(sx, so, n, "sum")
    pb.reduce_all(sx, sm, n, "mean")
    got, mean = run_program(ctx, pb, [x], [so, sm])
    exact = float(np.sum(x.astype(np.float64)))
    # a binary64 sum of n terms, then one rounding to binary32
    slack = n * 2.0 ** -53 * float(np.abs(x).sum())
    assert abs(float(got[0]) - exact) <= 2.0 ** -24 * abs(exact) + slack
    assert abs(float(mean[0]) - exact / n) <= 2.0 ** -23 * abs(exact / n) + slack / n
