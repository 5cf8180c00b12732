"""The time-driven layer kernel (a neuron's steps in one launch) at the sizes
where it can go wrong: fields that end inside the 16 loads ahead, partial
waves, one and many input channels, windows of one and four
blocks of 64 steps, fractional fire starts, an encoder whose times are not
steps, a pool first, fire windows apart from the integration window, and
weights that are not finite; against the oracle, bit for bit."""
import numpy as np
import pytest

import oracle
import vdttfs
from vdttfs import core
from vdttfs.core import Layer

pytestmark = pytest.mark.gpu


def net(rng, H, C0, C1, C2, K, same, pool_first, td, out_kind):
    def w(fan, *shape):
        return (rng.standard_normal(shape) * np.sqrt(4.0 / fan)).astype(np.float32)

    def bias(n):
        return (rng.standard_normal(n) * 0.1).astype(np.float32)

    L, h = [], H
    if pool_first:
        L.append(Layer(core.LAYER_POOL, h, h, C0, h // 2, h // 2, C0))
        h //= 2
    ho = h if same else h - K + 1
    L.append(Layer(core.LAYER_CONV, h, h, C0, ho, ho, C1, K, K, w(K * K * C0, K, K, C0, C1), bias(C1), 8.0, td))
    L.append(Layer(core.LAYER_POOL, ho, ho, C1, ho // 2, ho // 2, C1))
    f = (ho // 2) ** 2 * C1
    L.append(Layer(core.LAYER_FC, ho // 2, ho // 2, C1, 1, 1, C2, 1, 1, w(f, f, C2), bias(C2), 8.0, td))
    L.append(Layer(out_kind, 1, 1, C2, 1, 1, 5, 1, 1, w(C2, C2, 5), bias(5), 8.0, -1.0))
    return L


@pytest.mark.parametrize("mode", [vdttfs.STEP_T1, vdttfs.STEP_T2], ids=["t1", "t2"])
@pytest.mark.parametrize("T,tfs,H,C0,C1,C2,K,B,pool,odd", [
    (1, 0.0, 8, 1, 3, 7, 3, 3, False, ""),
    (16, 16.0, 9, 2, 17, 33, 3, 5, False, ""),
    (64, 10.5, 14, 5, 6, 40, 5, 4, True, ""),
    (65, 65.0, 8, 3, 70, 130, 3, 2, False, "inf"),
    (130, 0.0, 8, 20, 9, 12, 3, 2, False, "nan"),
    (255, 200.0, 8, 1, 4, 10, 3, 3, False, ""),
    (255, 255.0, 12, 16, 8, 64, 1, 2, True, ""),
])
def test_step_layers(gpu_ctx_factory, mode, T, tfs, H, C0, C1, C2, K, B, pool, odd):
    t1 = mode == vdttfs.STEP_T1
    print(f"step layers mode={mode} T={T} tfs={tfs} {H}x{H}x{C0} {C1} {C2} K={K} {odd}", flush=True)
    tc = vdttfs.task1_consts(T=T, delta=8) if t1 else vdttfs.task2_consts(T=T, delta=8, tfs=tfs)
    rng = np.random.default_rng(T + H + C1)
    L = net(rng, H, C0, C1, C2, K, not t1, pool, 2.5, core.LAYER_FC if t1 else core.LAYER_VMEM)
    if odd:
        conv = L[1 if pool else 0].kernel
        conv[0, K - 1, 0, C1 // 2] = np.inf if odd == "inf" else np.nan
    img = rng.random((B, H, H, C0)).astype(np.float32) * (rng.random((B, H, H, C0)) < 0.6)
    n_img = H * H * C0
    for enc, oenc in ((vdttfs.ENCODE_LINEAR, oracle.ENC_LINEAR), (vdttfs.ENCODE_LOG, oracle.ENC_LOG)):
        ref = oracle.stepnet_forward(oracle.Consts.from_task(tc), L, B, img, n_img, oenc, T / 4.0, 0.0,
                                     oracle.STEP_T1 if t1 else oracle.STEP_T2, same_pad=not t1)
        sn = vdttfs.StepNet(gpu_ctx_factory(tc), L, B, n_img, enc, T / 4.0, 0.0, mode)
        try:
            x, p = sn.ctx.to_device(img), sn.ctx.empty(B, np.int32)
            for _ in range(2):  # nothing is left of the first pass
                sn.forward(x, p)
            sn.ctx.synchronize()
            out, steps = sn.output()
            pred = p.download()
        finally:
            sn.close()
        assert steps == ref["steps"]
        np.testing.assert_array_equal(out, ref["final"], err_msg=f"encode {enc}")
        np.testing.assert_array_equal(pred, ref["pred"])
