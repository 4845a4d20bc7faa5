"""Softmax, log-softmax, log-sum-exp and the softmax gradient at the edges of their row forms (one
wave a row up to 2044 columns, one workgroup of 256, 512 or 1024 threads, streamed beyond 32764), on
rows whose start is not 16-byte aligned, with special-value rows, against the oracle."""
import numpy as np
import pytest

from oracle import oracle
from synaptik_amd.program import ProgramBuilder
from tests.gpu_helpers import run_program

pytestmark = pytest.mark.gpu

WIDTHS = [1, 2, 5, 252, 253, 508, 509, 1020, 1021, 2044, 2045, 4092, 4093, 4097, 8188, 8189, 16380,
          16383, 32764, 32767]


@pytest.mark.parametrize("log", [False, True])
@pytest.mark.parametrize("C", WIDTHS)
def test_forward(ctx, C, log):
    print(f"[softmax] C={C} log={log}", flush=True)
    R = 11
    rng = np.random.default_rng(C)
    x = (rng.standard_normal((R, C)) * 3).astype(np.float32)
    last = C - 1
    x[1, 0] = np.nan
    x[2, last] = np.inf
    x[3, last] = -np.inf
    x[4, :] = -np.inf
    x[5, :] = -np.abs(x[5]); x[5, last] = -0.0
    x[6, :] = -np.abs(x[6]); x[6, 0] = 0.0
    x[7, 0] = 120.0
    x[8, :] -= 200.0
    x[9, 0], x[9, last] = np.nan, np.inf
    pb = ProgramBuilder()
    sx, sy, sl = pb.input(R * C), pb.output(R * C), pb.output(R)
    pb.softmax(sx, sy, R, C, lse=sl, log=log)
    got, lse = run_program(ctx, pb, [x], [sy, sl])
    got = got.reshape(R, C)
    want = oracle.softmax_rows(x, log=log)  # the special-value classes
    assert np.array_equal(np.isnan(got), np.isnan(want))
    inf = np.isinf(want)
    assert np.array_equal(got[inf], want[inf])
    # Finite rows against 64 bits (the oracle's own binary32 Kahan sum is up to 4e-6 off on an
    # unshifted row): from the rounded difference on, an exponential of one unit, the sum's
    # rounding and the quotient's (or the logarithm's and the subtraction's).
    for r in np.flatnonzero(np.isfinite(want if not log else np.where(inf, 0, want)).all(1)):
        shift = np.float32(0) if np.isneginf(x[r]).any() else x[r].max()
        d = (x[r] - shift).astype(np.float64)
        total = np.exp(d).sum()
        if log:
            exact, size = d - np.log(total), np.abs(d) + 2 * abs(np.log(total)) + 1
        else:
            exact = np.exp(d) / total
            size = exact + 1e-31
        fin = np.isfinite(exact)
        assert np.all(np.abs(got[r][fin] - exact[fin]) <= 4e-7 * size[fin])
    w = oracle.logsumexp_rows(x)
    assert np.array_equal(np.isnan(lse), np.isnan(w))
    assert np.array_equal(lse[np.isinf(w)], w[np.isinf(w)])
    fin = np.isfinite(w)
    np.testing.assert_allclose(lse[fin], w[fin], rtol=2e-6, atol=2e-6)


@pytest.mark.parametrize("C", WIDTHS)
def test_backward(ctx, C, R=6):
    print(f"[softmax bwd] C={C} R={R}", flush=True)
    rng = np.random.default_rng(C + 1)
    y = oracle.softmax_rows((rng.standard_normal((R, C)) * 2).astype(np.float32))
    g = rng.standard_normal((R, C)).astype(np.float32)
    k = rng.standard_normal(R).astype(np.float32)
    pb = ProgramBuilder()
    sy, sg, sk = pb.input(R * C), pb.input(R * C), pb.input(R)
    plain, scaled = pb.output(R * C), pb.output(R * C)
    pb.softmax_bwd(sy, sg, plain, R, C)
    pb.softmax_bwd(sy, sg, scaled, R, C, rowscale=sk)
    a, b = (o.reshape(R, C) for o in run_program(ctx, pb, [y, g, k], [plain, scaled]))
    want = oracle.softmax_grad_rows(y, g)
    # y (g - s): s differs by a few units of its last place between sum orders
    tol = 4e-6 * (np.abs(y) * (np.abs(g) + 1.0)) + 1e-12
    assert np.all(np.abs(a - want) <= tol)
    assert np.all(np.abs(b - (want + k[:, None] * y)) <= tol + 2e-7 * np.abs(k[:, None] * y))


# NaN bit patterns: numpy's, the ones whose low payload bits are set, and memory poison. A row is in
# the binary32 exponential's range but for its NaN.
NANS = [0x7fc00000, 0x7fc00001, 0x7fffffff, 0xffffffff, 0x7f800001]


@pytest.mark.parametrize("R", [1024, 1025, 2048, 2049])
@pytest.mark.parametrize("C", [1, 5, 200, 253, 400, 509, 1020, 1021, 2043])
def test_backward_of_many_rows(ctx, C, R):
    """Rows of at most 2044: a workgroup a row up to 1024 or 2048 rows, a wave a row beyond."""
    test_backward(ctx, C, R)


@pytest.mark.parametrize("R,C", [(600, 900), (524288, 1), (524289, 1), (174763, 3), (131072, 4),
                                 (104858, 5), (7825, 67), (1025, 512), (525, 1001), (3, 300001)])
def test_log_sum_exp_gradient(ctx, R, C):
    """An element a thread below 2^19 elements or four columns, else groups of four over row ends."""
    print(f"[lse bwd] {R}x{C}", flush=True)
    rng = np.random.default_rng(R)
    x = rng.standard_normal((R, C)).astype(np.float32)
    lse, g = rng.standard_normal(R).astype(np.float32), rng.standard_normal(R).astype(np.float32)
    x[0, 0], x[R // 2, C - 1], x[R - 1, C - 1] = np.nan, np.inf, -np.inf
    pb = ProgramBuilder()
    sx, sl, sg = pb.input(R * C), pb.input(R), pb.input(R)
    each, same = pb.output(R * C), pb.output(R * C)
    pb.lse_bwd(sx, sl, each, R, C, g=sg)
    pb.lse_bwd(sx, sl, same, R, C, gconst=0.75)
    a, b = run_program(ctx, pb, [x, lse, g], [each, same])
    e = np.exp((x - lse[:, None]).astype(np.float64))
    # the exponential's rounding (up to one unit) and the product's
    np.testing.assert_allclose(a.reshape(R, C), g[:, None] * e, rtol=2e-7)
    np.testing.assert_allclose(b.reshape(R, C), 0.75 * e, rtol=2e-7)


@pytest.mark.parametrize("log", [False, True])
@pytest.mark.parametrize("C", [2, 101, 252, 512, 1021, 2044, 4096, 5003, 20001, 32768, 40000])
def test_every_nan_pattern_takes_its_row(ctx, C, log):
    print(f"[softmax nan] C={C} log={log}", flush=True)
    R = 2 * len(NANS) + 1
    x = np.random.default_rng(C).standard_normal((R, C)).astype(np.float32)
    bits = x.view(np.uint32)
    for i, pattern in enumerate(NANS):
        bits[i, C // 2] = pattern
        bits[len(NANS) + i, C - 1] = pattern
    pb = ProgramBuilder()
    sx, sy, sl = pb.input(R * C), pb.output(R * C), pb.output(R)
    pb.softmax(sx, sy, R, C, lse=sl, log=log)
    got, lse = run_program(ctx, pb, [x], [sy, sl])
    got = got.reshape(R, C)
    assert np.all(np.isnan(got[:-1])) and np.all(np.isnan(lse[:-1]))
    assert np.all(np.isfinite(got[-1])) and np.isfinite(lse[-1])
