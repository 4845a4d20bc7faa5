"""Index cross-entropy at the edges of its kernels' widths: the largest and smallest row of each
form (one wave a row up to 1024 classes, one workgroup a row, the streamed form beyond), rows whose
start is not 16-byte aligned, and sample counts formed in the kernel and by the launch before."""
import numpy as np
import pytest

from oracle import oracle
from synaptik_amd.program import ProgramBuilder
from tests.gpu_helpers import run_program

pytestmark = pytest.mark.gpu

WIDTHS = [1, 64, 65, 513, 1024, 1025, 2044, 2045, 4093, 8188, 8189, 16380, 16381, 32764, 32767,
          65532, 65535, 70001]


@pytest.mark.parametrize("ignore", [None, -100])
@pytest.mark.parametrize("C", WIDTHS)
def test_widths(ctx, C, ignore):
    print(f"[index_ce] C={C} ignore={ignore}", flush=True)
    R = 7
    rng = np.random.default_rng(C)
    logits = (rng.standard_normal((R, C)) * 3).astype(np.float32)
    y = rng.integers(0, C, R)
    y[0], y[1] = 0, C - 1
    if ignore is not None:
        y[2::3] = ignore
    pb = ProgramBuilder()
    sx, sy = pb.input(R * C), pb.input(R, "i64")
    sl, sl2, sg = pb.output(1), pb.output(1), pb.output(R * C)
    pb.index_ce(sx, sy, sl, R, C, grad=sg, ignore_index=ignore)
    pb.index_ce(sx, sy, sl2, R, C, ignore_index=ignore)  # the loss alone
    loss, loss2, grad = run_program(ctx, pb, [logits, y.astype(np.int64)], [sl, sl2, sg])
    want = oracle.index_ce_mean(logits, y, ignore_index=ignore)
    assert abs(loss[0] - want) <= 1e-5 * abs(want) + 1e-12
    assert loss2[0] == loss[0]
    np.testing.assert_allclose(grad.reshape(R, C),
                               oracle.index_ce_grad(logits, y, ignore_index=ignore),
                               rtol=1e-5, atol=1e-9)


@pytest.mark.parametrize("R,C", [(4096, 18), (4097, 18), (1024, 1030), (1025, 1030)])
def test_sample_count_of_many_rows(ctx, R, C):
    print(f"[index_ce] R={R} C={C}", flush=True)
    rng = np.random.default_rng(R)
    logits = rng.standard_normal((R, C)).astype(np.float32)
    y = rng.integers(0, C, R)
    y[rng.random(R) < 0.3] = -1
    pb = ProgramBuilder()
    sx, sy = pb.input(R * C), pb.input(R, "i32")
    sl, sg = pb.output(1), pb.output(R * C)
    pb.index_ce(sx, sy, sl, R, C, grad=sg, ignore_index=-1)
    loss, grad = run_program(ctx, pb, [logits, y.astype(np.int32)], [sl, sg])
    want = oracle.index_ce_mean(logits, y, ignore_index=-1)
    assert abs(loss[0] - want) <= 1e-5 * abs(want)
    np.testing.assert_allclose(grad.reshape(R, C), oracle.index_ce_grad(logits, y, ignore_index=-1),
                               rtol=1e-5, atol=1e-9)


@pytest.mark.parametrize("R", [1, 3, 4, 251, 252, 253, 1023, 1025, 8191, 8193, 8199])
def test_mean_counts_samples_without_a_loss(ctx, R):
    """The mean's loads at the edges of its rounds; samples whose loss is exactly zero (of either sign
    of zero logits) count, ignored rows do not."""
    print(f"[index_ce] mean R={R}", flush=True)
    rng = np.random.default_rng(R)
    logits = rng.standard_normal((R, 2)).astype(np.float32)
    y = rng.integers(0, 2, R)
    kind = rng.integers(0, 4, R)
    kind[0] = 0
    logits[kind == 1] = [-0.0, -np.inf]
    logits[kind == 2] = [0.0, -200.0]
    y[(kind == 1) | (kind == 2)] = 0
    y[kind == 3] = -5
    pb = ProgramBuilder()
    sx, sy = pb.input(R * 2), pb.input(R, "i32")
    both, alone, grad = pb.output(1), pb.output(1), pb.output(R * 2)
    pb.index_ce(sx, sy, both, R, 2, grad=grad, ignore_index=-5)
    pb.index_ce(sx, sy, alone, R, 2, ignore_index=-5)
    valid = kind != 3
    x = logits.astype(np.float64)
    with np.errstate(divide="ignore"):
        rows = np.log(np.exp(x).sum(1)) - x[np.arange(R), np.maximum(y, 0)]
    a, b, _ = run_program(ctx, pb, [logits, y.astype(np.int32)], [both, alone, grad])
    want = rows[valid].sum() / valid.sum()
    assert abs(a[0] - want) <= 1e-6 * abs(want) + 1e-12 and a[0] == b[0]


def test_special_rows(ctx):
    """NaN and infinite logits and a row of nothing but -inf, on both row forms."""
    for C in (70, 1500):
        rng = np.random.default_rng(C)
        logits = rng.standard_normal((6, C)).astype(np.float32)
        logits[0, 3] = np.nan
        logits[1, 4] = np.inf
        logits[2, :] = -np.inf
        logits[3, 5] = -np.inf
        logits[4, :] = -0.0
        y = np.array([3, 5, 1, 7, 0, 2])
        pb = ProgramBuilder()
        sx, sy = pb.input(6 * C), pb.input(6, "i64")
        sl, sg = pb.output(1), pb.output(6 * C)
        pb.index_ce(sx, sy, sl, 6, C, grad=sg)
        loss, grad = run_program(ctx, pb, [logits, y.astype(np.int64)], [sl, sg])
        want = oracle.index_ce_grad(logits, y)
        got = grad.reshape(6, C)
        assert np.isnan(loss[0])
        assert np.array_equal(np.isnan(got), np.isnan(want))
        fin = ~np.isnan(want)
        np.testing.assert_allclose(got[fin], want[fin], rtol=1e-5, atol=1e-9)


@pytest.mark.parametrize("R,C", [(70003, 3), (33000, 70), (1030, 1100), (9, 70001)])
def test_mostly_ignored_rows(ctx, R, C):
    """Ignored rows are not read: their logits are NaN here, their gradient is zero; the counts of
    four parts of the rows, and a mean over more rows than one round of loads."""
    print(f"[index_ce] ignored R={R} C={C}", flush=True)
    rng = np.random.default_rng(R)
    logits = rng.standard_normal((R, C)).astype(np.float32)
    y = rng.integers(0, C, R)
    skipped = rng.random(R) < 0.85
    skipped[0] = False
    y[skipped] = -7
    read = logits.copy()
    read[skipped] = np.nan
    pb = ProgramBuilder()
    sx, sy = pb.input(R * C), pb.input(R, "i64")
    sl, sl2, sg = pb.output(1), pb.output(1), pb.output(R * C)
    pb.index_ce(sx, sy, sl, R, C, grad=sg, ignore_index=-7)
    pb.index_ce(sx, sy, sl2, R, C, ignore_index=-7)
    loss, loss2, grad = run_program(ctx, pb, [read, y.astype(np.int64)], [sl, sl2, sg])
    d = (logits - logits.max(1, keepdims=True)).astype(np.float64)
    total = np.exp(d).sum(1)
    rows = np.flatnonzero(~skipped)
    exact = float(np.mean(np.log(total[rows]) - d[rows, y[rows]]))
    # a row's loss is off by a few units of its largest term, about 2^-22 of the mean
    assert abs(loss[0] - exact) <= 1e-6 * abs(exact) and loss2[0] == loss[0]
    grad = grad.reshape(R, C)
    assert not grad[skipped].any()
    want = np.exp(d[rows]) / total[rows, None]
    want[np.arange(len(rows)), y[rows]] -= 1.0
    np.testing.assert_allclose(grad[rows], want / len(rows), rtol=2e-6, atol=2e-7 / len(rows))
