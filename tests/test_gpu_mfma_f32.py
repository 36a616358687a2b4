"""F32 expert products on the fp32 matrix cores (csrc/hy_mfma_f32.hip): batches past
about 3 pairs per expert give, bit for bit, what the decode GEMV (HY_PATH_VALU) and the oracle give."""
import numpy as np
import pytest

import hy_oracle as O

pytestmark = pytest.mark.gpu


def layer_and_x(H, I, E, K, T, shared=True, seed=3):
    layer = O.synth_layer(H, I, E, K, O.F32, seed=seed, std=0.05, shared=shared)
    return layer, O.synth(seed + 10, 0, O.T_X, 0, (T, H), 1.0)


def run_both(gpu, layer, x, K, shared=True, **kw):
    T, H = x.shape
    E, I = layer.router.shape[0], layer.I
    m = gpu.Moe(H, I, E, K, gpu.F32, max_tokens=T, has_shared=shared, **kw)
    m.upload(0, layer)
    got = m.run(0, x)
    m.set_path(gpu.PATH_VALU)
    want = m.run(0, x)
    m.close()
    return got, want


# one row group (2 I = 64) and odd group counts; one block of K; tiles (of 32 and of 64
# pairs) holding 1, 4, 16, 17, 32, 33, 63, 64 and 65 pairs (the shared expert's T tokens, the routed experts' shares); one expert
@pytest.mark.parametrize("H,I,E,K,T,shared", [(64, 32, 2, 1, 17, True), (192, 96, 3, 2, 40, True),
                                              (128, 160, 1, 1, 63, True),
                                              (192, 64, 2, 2, 4, True), (64, 96, 4, 2, 64, True), (128, 64, 4, 4, 64, False),
                                              (256, 96, 16, 4, 65, True), (320, 128, 8, 3, 300, True)])
def test_matches_gemv_and_oracle(gpu, H, I, E, K, T, shared):
    layer, x = layer_and_x(H, I, E, K, T, shared)
    got, want = run_both(gpu, layer, x, K, shared)
    np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
    np.testing.assert_array_equal(got.view(np.uint32), O.moe_forward_q(layer, x).view(np.uint32))


def test_full_width_skewed(gpu):
    """HunyuanImage-3's widths; every token on the same experts (tiles of 64 and a rest)."""
    layer, x = layer_and_x(4096, 3072, 4, 2, 150)
    layer.router[:, 0] = [3.0, 2.0, -50.0, -50.0]
    x[:, 0] = 5.0
    got, want = run_both(gpu, layer, x, 2)
    np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))


def test_denormals_and_non_finite(gpu):
    layer, x = layer_and_x(128, 64, 4, 2, 48)
    x[5] *= np.float32(2.0 ** -130)
    x[7, 3] = np.inf
    x[9, 100] = np.nan
    got, want = run_both(gpu, layer, x, 2)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    ok = ~np.isnan(want)
    assert ok[5].all() and np.array_equal(got[ok].view(np.uint32), want[ok].view(np.uint32))


def test_dropped_pairs(gpu):
    layer, x = layer_and_x(128, 64, 8, 2, 90)
    got, want = run_both(gpu, layer, x, 2, drop_tokens=1, capacity_factor=0.7)
    np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
