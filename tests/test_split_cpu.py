"""What the fp32-product tests can see, on the CPU: products of three bf16 pieces with all six
significant piece products pass their checks, with any one of them missing none does."""
import numpy as np
import pytest

from test_gemm_gpu import check


def bf16(x):
    """Round to nearest even, as fp32."""
    u = x.astype(np.float32).view(np.uint32)
    return ((u + (((u >> 16) & 1) + np.uint32(0x7FFF))) & np.uint32(0xFFFF0000)).view(np.float32)


def pieces(x):
    hi = bf16(x)
    mid = bf16(x - hi)
    lo = bf16(x - hi - mid)
    return [p.astype(np.float64) for p in (hi, mid, lo)]


SIX = [(0, 0), (0, 1), (1, 0), (1, 1), (0, 2), (2, 0)]


@pytest.mark.parametrize("K", [32, 512, 4096])
def test_check_sees_every_piece_product(K):
    rng = np.random.default_rng(K)
    x = rng.standard_normal((24, K)).astype(np.float32) * np.exp2(rng.integers(-20, 20, (24, 1))).astype(np.float32)
    w = rng.standard_normal((200, K)).astype(np.float32)
    prod = {(i, j): pieces(x)[i] @ pieces(w)[j].T for i, j in SIX}
    check(sum(prod.values()), x, w)
    for missing in SIX:
        with pytest.raises(AssertionError):
            check(sum(p for k, p in prod.items() if k != missing), x, w)


def test_check_sees_flushed_denormal_pieces():
    """test_denormal_pieces: its operands' last pieces without bf16's denormals."""
    rng = np.random.default_rng(4)
    x = np.ldexp(rng.choice([-1.0, 1.0], (48, 512)) * rng.uniform(1.0, 4.0, (48, 512)), -110).astype(np.float32)
    w = np.ldexp(rng.standard_normal((200, 512)), 60).astype(np.float32)
    px, pw = pieces(x), pieces(w)
    assert np.array_equal(sum(px).astype(np.float32), x)
    check(sum(px[i] @ pw[j].T for i, j in SIX), x, w)
    px[2] = np.where(np.abs(px[2]) < 2.0 ** -126, 0.0, px[2])
    with pytest.raises(AssertionError):
        check(sum(px[i] @ pw[j].T for i, j in SIX), x, w)
