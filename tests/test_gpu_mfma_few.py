"""The grouped GEMM's stream for experts of few tokens (csrc/hy_mfma_few.hip) against the
oracle, bit for bit: tiles of 1 to 32 pairs and a second tile, row groups that do not fill
a work group of four, reductions shorter than and no multiple of the blocks it keeps in
flight, and the first batch past its range."""
import numpy as np
import pytest

import hy_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wtype", [O.Q8_0, O.Q4_0])
@pytest.mark.parametrize("H,I,shared", [(128, 64, True), (384, 192, True), (640, 320, False), (256, 1344, True)])
def test_few(gpu, wtype, H, I, shared):
    E, K = 3, 2
    layer = O.synth_layer(H, I, E, K, wtype, seed=H + I, std=0.05, shared=shared)
    m = gpu.Moe(H, I, E, K, wtype, max_tokens=128, has_shared=shared)
    m.set_path(gpu.PATH_MFMA)
    m.upload(0, layer)
    for T in (1, 2, 16, 17, 31, 32, 33, 96, 97):  # 64 pairs per expert end at T = 96
        x = O.synth(70 + T, 0, O.T_X, 0, (T, H), 1.0)
        got, ref = m.run(0, x), O.moe_forward_q(layer, x)
        assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), f"T={T}"
    m.close()


@pytest.mark.parametrize("wtype", [O.Q8_0, O.Q4_0])
def test_few_one_expert(gpu, wtype):
    """Every token on one expert: full tiles and a ragged last one."""
    H, I = 256, 128
    layer = O.synth_layer(H, I, 8, 1, wtype, seed=9, std=0.05)
    layer.router[3] = 10.0
    m = gpu.Moe(H, I, 8, 1, wtype, max_tokens=128)
    m.set_path(gpu.PATH_MFMA)
    m.upload(0, layer)
    for T in (64, 65, 95, 128):
        x = np.abs(O.synth(80 + T, 0, O.T_X, 0, (T, H), 1.0))
        got, ref = m.run(0, x), O.moe_forward_q(layer, x)
        assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), f"T={T}"
    m.close()
