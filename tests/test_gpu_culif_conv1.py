"""The engine's conv1 on the matrix cores (32 steps a product) at the sizes
where it can go wrong: one to three input channels (an odd number of taps in
the last pair), c_out past one and two 32-wide tiles, windows that end inside
32 steps or 8, inputs other than 1.0, dense and silent input, thresholds that
fire at step 0; every neuron against the oracle, bit for bit."""
import numpy as np
import pytest

import oracle
import vdttfs
from vdttfs import models

pytestmark = pytest.mark.gpu
INF = np.float32(9999.0)


@pytest.mark.parametrize("decay,th", [(0.5, 1.0), (0.9, 0.4), (-0.7, 0.5), (0.5, 0.0), (0.5, -0.5)])
@pytest.mark.parametrize("C_in,C_out,T,delta", [(1, 64, 24, 8), (2, 33, 64, 32), (3, 70, 40, 8), (2, 130, 96, 32),
                                                (3, 20, 160, 32), (1, 5, 33, 33)])
def test_engine_conv1(gpu_ctx_factory, C_in, C_out, T, delta, decay, th):
    print(f"culif conv1 C_in={C_in} C_out={C_out} T={T} decay={decay} th={th}", flush=True)
    B, H, W = 3, 9, 11
    rng = np.random.default_rng(C_in * 1000 + C_out + T)
    ev = (rng.random((B, C_in, H, W, T)) < 0.08).astype(np.float32)
    ev[0, :, :4] = 0.0                      # silent rows
    ev[1, :, 5:7, :, : T // 2] = 1.0        # dense steps
    ev[2] *= rng.choice(np.array([1.0, 1.0, 0.5, -2.0, -0.0], np.float32), ev[2].shape)
    k = models.kaiming
    L = [vdttfs.CulifLayerSpec(vdttfs.CULIF_RAW_CONV, C_in, H, W, C_out, k(3, 0, (C_out, C_in, 3, 3), 9 * C_in), None,
                               decay, th),
         vdttfs.CulifLayerSpec(vdttfs.CULIF_FC, C_out * H * W, 1, 1, 4, k(3, 1, (4, C_out * H * W), 99), None, 0.5,
                               1.0)]
    ref, _ = oracle.culif_net_forward(L, ev, B, T, delta)
    if th == 1.0:
        assert (ref[0] < INF).any() and (ref[0] == INF).any()
    net = vdttfs.CulifNet(gpu_ctx_factory(vdttfs.task3_consts(T=T, delta=delta)), L, B)
    try:
        net.forward(net.ctx.to_device(ev))
        net.ctx.synchronize()
        got = net.layer_output(0)
    finally:
        net.close()
    np.testing.assert_array_equal(got.reshape(-1), ref[0].reshape(-1))
