"""The fp32 product through bf16 pieces (csrc/hy_gemm.hip), against float64.

Bound: every element adds at most 6 K / 16 matrix-core results (and the K / 32 stage
pieces of a cut tile) in fp32, each rounding at most 2^-24 of a partial sum that is at
most S = sum_k |a_k w_k|, and drops piece products below 2^-24 |a_k w_k|:
|c - exact| <= (6 K / 16 + K / 32 + 4) 2^-24 S.  A first-order term as large again covers
roundings inside a matrix instruction.

That worst case is far above what happens at large K, so a row's error is also held to
1.5e-6 of the row's norm.  Independent roundings of up to 2^-23 of a growing partial sum
add up to sqrt(6 K / 16 / 2) 2^-23 / sqrt(3) = 1.9e-6 in the extreme at K = 4096 and
measure 0.1e-6 to 1.1e-6; a product that lacks any one of its six piece products is at
2.4e-6 or more whatever K (test_split_cpu.py).  Missing pieces in less than a third of the
stages of K stay unseen."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def check(got, x, w, r=None):
    K = x.shape[1]
    x64, w64 = x.astype(np.float64), w.astype(np.float64)
    want = x64 @ w64.T + (0.0 if r is None else r)
    bound = 2 * (6 * K / 16 + K / 32 + 4) * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64).T)
    if r is not None:
        bound += 2.0 ** -24 * (np.abs(want) + np.abs(r))
    assert np.all(np.abs(got - want) <= bound)
    err, norm = np.linalg.norm(got - want, axis=1), np.linalg.norm(want, axis=1)
    assert np.all(err <= 1.5e-6 * norm), (err / norm).max()


# one to four 32-row tiles and their edges; N below, at and past a 128-row tile; one stage
# of K, fewer stages than work groups, and ranges that cut every tile
@pytest.mark.parametrize("M,N,K", [(17, 100, 32), (32, 128, 64), (33, 129, 96), (64, 517, 1024), (65, 257, 4096),
                                   (96, 6150, 4096), (97, 4096, 512), (128, 10003, 2048)])
def test_small_batches(gpu, M, N, K):
    rng = np.random.default_rng(M)
    x = rng.standard_normal((M, K)).astype(np.float32) * np.exp2(rng.integers(-20, 20, (M, 1))).astype(np.float32)
    w = rng.standard_normal((N, K)).astype(np.float32)
    r = rng.standard_normal((M, N)).astype(np.float32)
    check(gpu.lm_head_f32(x, w), x, w)
    check(gpu.lm_head_f32(x, w, r), x, w, r)


# five to eight 32-row subtiles a tile, odd counts (a wave with one subtile less), several
# row tiles, N at and past a 256-row tile, cut tiles and whole ones; the last four take
# whole tiles without scratch (up to 128 rows, and 256, of A each), K of one to three
# stages
@pytest.mark.parametrize("M,N,K", [(129, 4200, 4096), (192, 4097, 2080), (200, 4352, 4096), (256, 6150, 1056),
                                   (300, 6144, 4096), (1100, 2049, 512), (2300, 1024, 1024),
                                   (129, 65600, 32), (300, 33000, 48), (300, 65600, 32), (513, 45000, 16)])
def test_larger_batches(gpu, M, N, K):
    rng = np.random.default_rng(M)
    x = rng.standard_normal((M, K)).astype(np.float32) * np.exp2(rng.integers(-20, 20, (M, 1))).astype(np.float32)
    w = rng.standard_normal((N, K)).astype(np.float32)
    r = rng.standard_normal((M, N)).astype(np.float32)
    check(gpu.lm_head_f32(x, w), x, w)
    check(gpu.lm_head_f32(x, w, r), x, w, r)


@pytest.mark.parametrize("M,N,K", [(40, 300, 256), (128, 9000, 1024), (300, 6144, 512)])
def test_values_without_a_split(gpu, M, N, K):
    """Infinities, NaNs and values that round up to infinity in bf16 give what an fp32
    product gives; the other elements keep their bound."""
    rng = np.random.default_rng(1)
    x = rng.standard_normal((M, K)).astype(np.float32)
    w = rng.standard_normal((N, K)).astype(np.float32)
    x[3, 7] = np.inf
    x[5, K - 1] = np.nan
    w[11, 0] = -np.inf
    w[N - 1, 9] = np.float32(3.4e38)  # finite; its nearest bf16 is infinity
    x[:, 9] = np.float32(2.0 ** -40)
    got = gpu.lm_head_f32(x, w)
    with np.errstate(all="ignore"):
        want = x.astype(np.float64) @ w.astype(np.float64).T
    assert np.array_equal(np.isnan(got), np.isnan(want))
    inf = np.isinf(want)
    assert inf.any() and np.array_equal(got[inf], want[inf].astype(np.float32))
    rows, cols = [i for i in range(M) if i not in (3, 5)], [j for j in range(N) if j != 11]
    check(got[np.ix_(rows, cols)], x[rows], w[cols])


@pytest.mark.parametrize("M,N,K", [(48, 200, 512), (300, 6144, 512)])
def test_denormal_pieces(gpu, M, N, K):
    """Operands of 2^-110 to 2^-108 split exactly, their last pieces mostly into bf16 denormals,
    and stay on the bf16 matrix cores, which must not flush these (2.4e-6 of the norm)."""
    rng = np.random.default_rng(4)
    x = np.ldexp(rng.choice([-1.0, 1.0], (M, K)) * rng.uniform(1.0, 4.0, (M, K)), -110).astype(np.float32)
    w = np.ldexp(rng.standard_normal((N, K)), 60).astype(np.float32)
    check(gpu.lm_head_f32(x, w), x, w)
    x, w = (rng.standard_normal((M, K)) * 2.0 ** 60).astype(np.float32), np.resize(x, (N, K))
    check(gpu.lm_head_f32(x, w), x, w)


def test_tiny_values(gpu):
    """Operands down at 2^-100 keep their significand (bf16 pieces down to denormals)."""
    rng = np.random.default_rng(2)
    x = (rng.standard_normal((48, 512)) * 2.0 ** -100).astype(np.float32)
    w = (rng.standard_normal((200, 512)) * 2.0 ** 20).astype(np.float32)
    check(gpu.lm_head_f32(x, w), x, w)


@pytest.mark.parametrize("M,N,K", [(77, 6144, 4096), (128, 33000, 2048), (300, 6144, 4096), (2300, 3000, 1024)])
def test_errors_have_no_mean(gpu, M, N, K):
    """The errors' mean is far below their rms (accumulators of one sign leave 0.21 of it at
    K = 4096, 0.11 at 1024).  An average over as many elements of independent errors would be
    below 0.01 of the rms; a fortieth leaves room for the last turn of the signs."""
    rng = np.random.default_rng(3)
    x = rng.standard_normal((M, K)).astype(np.float32)
    w = rng.standard_normal((N, K)).astype(np.float32)
    e = gpu.lm_head_f32(x, w) - x.astype(np.float64) @ w.astype(np.float64).T
    rms = np.sqrt((e * e).mean())
    assert abs(e.mean()) <= 0.025 * rms
    assert rms <= 1.5e-6 * np.sqrt(K)  # the results' rms is sqrt(K)


# nine to sixteen rows in one pass (N of 4096 and more, not a multiple of a wave's four rows)
# and in two; K past and below the lanes' chunks
@pytest.mark.parametrize("M", [9, 12, 13, 16])
@pytest.mark.parametrize("N,K", [(4096, 272), (5003, 1040), (4095, 1024)])
def test_nine_to_sixteen_rows(gpu, M, N, K):
    rng = np.random.default_rng(M)
    x = rng.standard_normal((M, K)).astype(np.float32)
    w = rng.standard_normal((N, K)).astype(np.float32)
    r = rng.standard_normal((M, N)).astype(np.float32)
    got = gpu.lm_head_f32(x, w)
    check(got, x, w)
    check(gpu.lm_head_f32(x, w, r), x, w, r)
    # a row's bits do not depend on how many rows share the pass
    assert np.array_equal(got[:8].view(np.uint32), gpu.lm_head_f32(x[:8], w).view(np.uint32))


# small-batch tiles of every height, cut and whole, and the larger kernel with and without
# scratch
@pytest.mark.parametrize("e", [-104, -109, -112, -116, -124, -134, -146])
@pytest.mark.parametrize("M,N,K", [(20, 300, 512), (48, 2048, 1024), (90, 257, 256), (128, 517, 512),
                                   (300, 6144, 512), (300, 33000, 48)])
def test_operands_without_an_exact_split(gpu, M, N, K, e):
    """Below 2^-110 three bf16 pieces do not hold an fp32 value: rows of such values, on either
    side, keep fp32's accuracy (6e-7 of a row's norm measured; unmended pieces leave 2e-6 at
    2^-116 and 5e-4 at 2^-124).  Their neighbours, and sums that mix both, too."""
    rng = np.random.default_rng(-e)

    def tiny(*shape):
        return np.ldexp(rng.standard_normal(shape), e).astype(np.float32)

    def rel(got, x, w):
        ref = x.astype(np.float64) @ w.astype(np.float64).T
        return (np.linalg.norm(got - ref, axis=1) / np.linalg.norm(ref, axis=1)).max()

    x = rng.standard_normal((M, K)).astype(np.float32)
    w = np.ldexp(rng.standard_normal((N, K)), 60).astype(np.float32)
    x[M // 2:] = tiny(M - M // 2, K)
    got = gpu.lm_head_f32(x, w)
    assert rel(got[:M // 2], x[:M // 2], w) <= 1.5e-6
    assert rel(got[M // 2:], x[M // 2:], w) <= 1.5e-6
    x = np.ldexp(rng.standard_normal((M, K)), 60).astype(np.float32)
    w = tiny(N, K)
    w[0] = 0.0
    got = gpu.lm_head_f32(x, w)
    assert rel(got, x, w) <= 1.5e-6 and not got[:, 0].any()
    # a single such operand that carries its row: 2^60 against zeros
    x[:] = 0.0
    x[:, K - 1] = np.float32(2.0 ** 60)
    assert np.array_equal(gpu.lm_head_f32(x, w), np.ldexp(w[:, K - 1], 60)[None].repeat(M, 0))
