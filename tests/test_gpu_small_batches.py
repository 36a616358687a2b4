"""The kernels between the products at small batches, bit for bit against the oracle: the
weighted RMSNorm with the row in registers (and the loop of other widths), in place too;
the <2,4> router; the dispatch in one launch and the first batch past its 1024 pairs."""
import ctypes as C

import numpy as np
import pytest

import hy_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,T", [(256, 2048), (256, 2049), (1024, 2049), (1280, 2049), (4096, 300)])
def test_rms_norm_w_many_rows(gpu, H, T):
    test_rms_norm_w(gpu, H, T)


@pytest.mark.parametrize("H", [256, 320, 2048, 4096, 4352])
@pytest.mark.parametrize("T", [1, 5])
def test_rms_norm_w(gpu, H, T):
    rng = np.random.default_rng(H + T)
    x, w = rng.standard_normal((T, H)).astype(np.float32), rng.standard_normal(H).astype(np.float32)
    ref = O.rms_norm_blocked(x, w)
    f = gpu.lib().hy_rms_norm_w
    vp = C.c_void_p
    f.argtypes, f.restype = [vp, vp, C.c_uint32, C.c_uint32, C.c_float, vp, vp], C.c_int
    xb, wb, ob = gpu.Buf.from_array(x), gpu.Buf.from_array(w), gpu.Buf.empty((T, H))
    for dst in (ob, xb):  # in place last
        assert f(xb.ptr, wb.ptr, T, H, 1e-5, dst.ptr, None) == 0
        assert np.array_equal(dst.numpy().view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("T,E,K", [(33, 7, 2), (37, 64, 8), (128, 12, 8), (129, 12, 8), (256, 5, 4), (257, 5, 4)])
@pytest.mark.parametrize("drop", [0, 1])
def test_routing(gpu, T, E, K, drop):
    H, I = 192, 64
    layer = O.synth_layer(H, I, E, K, O.Q8_0, seed=T + E, std=0.05)
    m = gpu.Moe(H, I, E, K, O.Q8_0, max_tokens=T, drop_tokens=drop, capacity_factor=1.0, min_capacity=2)
    m.upload(0, layer)
    x = O.synth(T, 0, O.T_X, 0, (T, H), 1.0)
    out, lg, w, idx = m.run(0, x, debug=True)
    layer.capacity = O.drop_capacity(T, E, K, 1.0, 2) if drop else 0
    ref, rlg, rw, ridx = O.moe_forward_q(layer, x, debug=True)
    assert np.array_equal(lg.view(np.uint32), rlg.view(np.uint32)) and np.array_equal(idx, ridx)
    assert np.array_equal(out.view(np.uint32), ref.view(np.uint32))
    m.close()
