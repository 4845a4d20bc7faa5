"""GEMMs of odd extents and leading dimensions on every kernel and plan that takes them: the
direct-to-LDS kernel's unaligned form (tiles moved back at the operand's end, the chunk K cuts,
operands of less than a tile), the register kernel's 32x32 and 64x64 tiles with their K groups, and
split-K slices of both.
Operands are small integers, so every product sum is exact and the results must be equal bit for
bit, whatever the order of the sums; each epilogue is checked the same way."""
import numpy as np
import pytest

from synaptik_amd.native import HipProgram
from synaptik_amd.program import ProgramBuilder
from tests.gpu_helpers import run_program

pytestmark = pytest.mark.gpu

SHAPES = [
    (17, 17, 17), (33, 47, 31), (100, 101, 129),   # 32x32 tiles, K below and above a step a wave
    (97, 301, 515), (20, 21, 2001),                # ... in slices
    (1023, 1025, 19),                              # 64x64 LDS tiles, one k-tile
    (1025, 513, 67), (575, 1087, 33), (512, 1024, 1027),  # 64x64 LDS tiles, whole and in slices
    (2047, 2047, 35), (2049, 2050, 34),            # 128x128 LDS tiles; 64x64 past their last round
    (385, 387, 2051), (65, 130, 1100),             # deep: slices of 64x64 tiles
    (40, 1500, 1030), (1500, 40, 1030),            # an extent below a tile: no moved tile
]
LAYOUTS = [(False, False), (False, True), (True, False), (True, True)]


def _operands(rng, M, N, K, ta, tb, pad):
    A = rng.integers(-3, 4, (M, K)).astype(np.float32)
    B = rng.integers(-3, 4, (K, N)).astype(np.float32)
    a, b = (A.T if ta else A), (B.T if tb else B)
    sa = np.full((a.shape[0], a.shape[1] + pad), np.nan, np.float32)  # never read into a result
    sb = np.full((b.shape[0], b.shape[1] + pad), np.nan, np.float32)
    sa[:, :a.shape[1]], sb[:, :b.shape[1]] = a, b
    return A, B, sa, sb


@pytest.mark.parametrize("pad", [0, 1])
@pytest.mark.parametrize("ta,tb", LAYOUTS)
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_exact_products(ctx, M, N, K, ta, tb, pad):
    print(f"[gemm] {M}x{N}x{K} ta={ta} tb={tb} pad={pad}", flush=True)
    rng = np.random.default_rng(M * 7 + N * 3 + K)
    A, B, sa, sb = _operands(rng, M, N, K, ta, tb, pad)
    pb = ProgramBuilder()
    xa, xb = pb.input(sa.size), pb.input(sb.size)
    xc = pb.output(M * N)
    pb.gemm(xa, xb, xc, M, N, K, trans_a=ta, trans_b=tb, lda=sa.shape[1], ldb=sb.shape[1])
    (got,) = run_program(ctx, pb, [sa, sb], [xc])
    want = (A.astype(np.float64) @ B.astype(np.float64)).astype(np.float32)
    assert np.array_equal(got.reshape(M, N), want)


# M/N-contiguous operands of less than a 64-wide tile, many tiles along the other extent: LDS tiles
# whose chunks run past the operand's row, 64x64 register tiles (the last three), by layout and K
NARROW = [(33, 17000, 67), (17000, 63, 97), (61, 16500, 520), (20, 16500, 200), (33000, 33, 33),
          (27, 16500, 313), (16500, 45, 257),            # ... in two K groups a workgroup
          (16500, 17, 19), (31, 16500, 19), (16385, 32, 127)]


@pytest.mark.parametrize("pad", [0, 1])
@pytest.mark.parametrize("ta,tb", LAYOUTS)
@pytest.mark.parametrize("M,N,K", NARROW)
def test_narrow_operands(ctx, M, N, K, ta, tb, pad):
    test_exact_products(ctx, M, N, K, ta, tb, pad)


@pytest.mark.parametrize("ta,tb", LAYOUTS)
@pytest.mark.parametrize("M,N,K", [(33, 17000, 67), (17000, 61, 97), (16500, 17, 19),
                                   (16450, 27, 200), (27, 16450, 313), (16450, 45, 257),
                                   (16450, 70, 40)])  # (column sums of over 256 partial rows)
def test_narrow_epilogues(ctx, M, N, K, ta, tb):
    test_epilogues(ctx, M, N, K, ta, tb)


@pytest.mark.parametrize("ta,tb", LAYOUTS)
@pytest.mark.parametrize("M,N,K", [(33, 47, 31), (97, 301, 515), (1025, 513, 67), (2047, 2047, 35),
                                   (385, 387, 2051)])
def test_epilogues(ctx, M, N, K, ta, tb):
    """Bias + ReLU, accumulation, the ReLU gradient with its column sum, the forward with its
    cotangent and column sum, and a staged SGD update (lr and momentum powers of two)."""
    print(f"[gemm] epilogues {M}x{N}x{K} ta={ta} tb={tb}", flush=True)
    rng = np.random.default_rng(M + N + K)
    A, B, sa, sb = _operands(rng, M, N, K, ta, tb, 0)
    prod = (A.astype(np.float64) @ B.astype(np.float64)).astype(np.float32)
    bias = rng.integers(-5, 6, N).astype(np.float32)
    y = rng.integers(-1, 2, (M, N)).astype(np.float32)
    dy = rng.integers(-4, 5, (M, N)).astype(np.float32)
    p0 = rng.integers(-9, 10, (M, N)).astype(np.float32)
    m0 = rng.integers(-9, 10, (M, N)).astype(np.float32)
    kw = dict(trans_a=ta, trans_b=tb)
    pb = ProgramBuilder()
    xa, xb, xbias, xy, xdy = (pb.input(v.size) for v in (sa, sb, bias, y, dy))
    xp, xm, cnt = pb.input(M * N), pb.input(M * N), pb.input(1, "i64")
    fwd, grad, gsum, act, dz, zsum, pn, mn = (pb.output(c) for c in
                                              (M * N, M * N, N, M * N, M * N, N, M * N, M * N))
    pb.gemm(xa, xb, fwd, M, N, K, bias=xbias, act="relu", **kw)
    pb.gemm(xa, xb, fwd, M, N, K, accumulate=True, **kw)
    pb.gemm(xa, xb, grad, M, N, K, aux=xy, act="relu", act_grad=True, colsum=gsum, **kw)
    pb.gemm(xa, xb, act, M, N, K, bias=xbias, act="relu", dy=xdy, dz=dz, colsum=zsum, **kw)
    pb.gemm_update(xa, xb, M, N, K, cnt, (xp, xm, None, pn, mn, None), kind="sgd", lr=0.25,
                   momentum=0.5, has_momentum_slot=True, **kw)
    outs = run_program(ctx, pb, [sa, sb, bias, y, dy, p0, m0, np.ones(1, np.int64)],
                       [fwd, grad, gsum, act, dz, zsum, pn, mn])
    shape = lambda i: outs[i].reshape(M, N)  # noqa: E731
    relu = np.maximum(prod + bias, 0)
    assert np.array_equal(shape(0), relu + prod)
    g = np.where(y > 0, prod, 0)
    assert np.array_equal(shape(1), g)
    assert np.array_equal(outs[2], g.astype(np.float64).sum(0).astype(np.float32))
    assert np.array_equal(shape(3), relu)
    z = np.where(relu > 0, dy, 0)
    assert np.array_equal(shape(4), z)
    assert np.array_equal(outs[5], z.astype(np.float64).sum(0).astype(np.float32))
    mom = np.float32(0.5) * m0 + prod
    assert np.array_equal(shape(7), mom)
    assert np.array_equal(shape(6), p0 - np.float32(0.25) * mom)


def test_infinities_stay_in_their_rows(ctx):
    """Rows and columns past an edge tile's operand are never read into a result: an infinite
    operand element changes only its own row."""
    for M, N, K, ta, tb in [(1025, 513, 67, False, True), (1025, 513, 67, True, False),
                            (100, 101, 129, True, False)]:
        rng = np.random.default_rng(K)
        A, B, sa, sb = _operands(rng, M, N, K, ta, tb, 0)
        B[:] = 1.0
        sb[:] = 1.0
        A[5, 3] = np.inf
        (sa.T if ta else sa)[5, 3] = np.inf
        pb = ProgramBuilder()
        xa, xb, xc = pb.input(sa.size), pb.input(sb.size), pb.output(M * N)
        pb.gemm(xa, xb, xc, M, N, K, trans_a=ta, trans_b=tb)
        (got,) = run_program(ctx, pb, [sa, sb], [xc])
        got = got.reshape(M, N)
        assert np.all(np.isposinf(got[5]))
        rest = np.delete(np.arange(M), 5)
        want = np.broadcast_to(A[rest].sum(1, dtype=np.float64)[:, None], (M - 1, N))
        assert np.array_equal(got[rest], want.astype(np.float32))



def _run_periodic(ctx, M, N, K, ta, tb, block, B):
    """C = op(A).op(B) with A the rows of `block` over and over, uploaded one repetition a time."""
    rows, width = (K, M) if ta else (M, K)
    a = ctx.buffer(4 * rows * width)
    for r in range(0, rows, len(block)):
        a.upload(block[:rows - r], 4 * r * width)
    pb = ProgramBuilder()
    xa, xb, xc = pb.input(M * K), pb.input(K * N), pb.output(M * N)
    pb.gemm(xa, xb, xc, M, N, K, trans_a=ta, trans_b=tb)
    prog = HipProgram(ctx, pb.image())
    c = ctx.buffer(4 * M * N)
    prog.run([a, ctx.upload(np.ascontiguousarray(B.T) if tb else B)], [c])
    prog.close()
    return c.download(np.float32, M * N).reshape(M, N)


def _assert_periodic(got, block, B):
    want = (block.astype(np.float64) @ B.astype(np.float64)).astype(np.float32)
    for r in range(0, len(got), len(want)):
        assert np.array_equal(got[r:r + len(want)], want[:len(got) - r]), r


@pytest.mark.parametrize("M,N,K,ta,tb", [
    (2097153, 64, 1024, False, True),    # aligned operands, ragged M
    (2097153, 68, 1027, False, False),   # the unaligned form
    (1024, 96, 2097155, True, False),    # a contraction over as many rows, in slices
])
def test_operands_beyond_two_to_the_31_elements(ctx, M, N, K, ta, tb):
    print(f"[gemm] large {M}x{N}x{K} ta={ta} tb={tb}", flush=True)
    rng = np.random.default_rng(N)
    block = rng.integers(-1, 2, (40009, M if ta else K)).astype(np.float32)
    B = rng.integers(-1, 2, (K, N), dtype=np.int8).astype(np.float32)
    got = _run_periodic(ctx, M, N, K, ta, tb, block, B)
    if not ta:
        _assert_periodic(got, block, B)
        return
    folded = np.zeros((len(block), N))  # the rows of B that meet one row of the block
    for r in range(0, K, len(block)):
        folded[:min(len(block), K - r)] += B[r:r + len(block)]
    # whole numbers below 2^24: exact in any order
    assert np.array_equal(got, (block.T.astype(np.float64) @ folded).astype(np.float32))


def test_more_tiles_than_one_grid_plane(ctx):
    """More than 2^20 64x64 tiles of the register kernel: its grid has planes."""
    M, N, K = 64 * (1 << 20) + 65, 17, 17
    print(f"[gemm] planes {M}x{N}x{K}", flush=True)
    rng = np.random.default_rng(17)
    block = rng.integers(-3, 4, (1000003, K)).astype(np.float32)
    B = rng.integers(-3, 4, (K, N)).astype(np.float32)
    _assert_periodic(_run_periodic(ctx, M, N, K, False, False, block, B), block, B)
