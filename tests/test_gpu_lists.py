"""Integration from the column lists over every bin (windows past 64 steps)
against the oracle, bit for bit: LUT layers with fire start 0 at two and four
bin blocks, tap counts of each kernel, C_out below and past a wave, an FC
layer's group and several, lists past a window's capacity and of every wave
count; CuLIF layers in the engine with bins without events, silent fields and
thresholds that fire without input."""
import numpy as np
import pytest

import oracle
import vdttfs
from vdttfs import models
from test_gpu_split import case, reference, run

pytestmark = pytest.mark.gpu
INF = np.float32(9999.0)

# name, T, tfs, task2, is_fc, B, H, W, C_in, C_out, K
SHAPES = [
    ("t80-conv3-9-33", 80, 0, True, False, 3, 7, 5, 9, 33, 3),
    ("t65-conv3-20-131", 65, 0, False, False, 2, 6, 7, 20, 131, 3),
    ("t80-conv1-70-100", 80, 0, True, False, 5, 9, 4, 70, 100, 1),
    ("t129-conv3-40-260", 129, 0, True, False, 2, 6, 5, 40, 260, 3),
    ("t255-conv5-32-64", 255, 0, False, False, 3, 9, 8, 32, 64, 5),
    ("t100-conv3-200-70", 100, 0, True, False, 2, 4, 3, 200, 70, 3),
    ("t255-conv3-24-1024", 255, 0, True, False, 1, 3, 3, 24, 1024, 3),
    ("t80-fc-1600-128", 80, 0, True, True, 9, 1, 1, 1600, 128, 1),
    ("t80-fc-128-10", 80, 0, True, True, 17, 1, 1, 128, 10, 1),
    ("t200-fc-4100-700", 200, 0, False, True, 3, 1, 1, 4100, 700, 1),
    ("t65-fc-3-1", 65, 0, True, True, 5, 1, 1, 3, 1, 1),
]


@pytest.mark.parametrize("kind", ["random", "silent", "bin0", "one-late-bin", "last-bin", "dense", "fractional"])
@pytest.mark.parametrize("shape", SHAPES, ids=[s[0] for s in SHAPES])
def test_lists_match_oracle(gpu_ctx_factory, shape, kind):
    tc, ho, wo, Wt, bias, sp = case(shape, kind)
    T = tc.T
    alpha, theta = vdttfs.build_luts_host(tc, 0.75 * T, 0.5, 1.5 * T, 2.5)
    ref = reference(shape, tc, ho, wo, Wt, bias, sp, alpha, theta, 3)
    got = run(gpu_ctx_factory(tc), shape, ho, wo, Wt, bias, sp, alpha, theta, 3)
    np.testing.assert_array_equal(got, ref, err_msg=f"{shape[0]} {kind}")


@pytest.mark.parametrize("shape", [SHAPES[0], SHAPES[4], SHAPES[7]], ids=lambda s: s[0])
@pytest.mark.parametrize("what", ["shuffled", "level", "below", "steep", "inf-weight", "nan-weight"])
def test_lists_odd_tables_and_weights(gpu_ctx_factory, shape, what):
    tc, ho, wo, Wt, bias, sp = case(shape, "random")
    T = tc.T
    rng = np.random.default_rng(5)
    alpha, theta = vdttfs.build_luts_host(tc, 0.75 * T, 0.5, 1.5 * T, 2.5)
    if what == "shuffled":
        theta = rng.permutation(theta)
    elif what == "level":
        theta = np.full(T, 0.7, np.float32)
    elif what == "below":
        theta = np.where(np.arange(T) < T // 2, theta, 1e-6).astype(np.float32)
    elif what == "steep":
        theta = np.exp(-np.arange(T, dtype=np.float32) ** 2 / 40).astype(np.float32)
    else:
        Wt[rng.integers(0, Wt.shape[0], 6), rng.integers(0, Wt.shape[1], 6)] = np.nan if what == "nan-weight" else np.inf
    ref = reference(shape, tc, ho, wo, Wt, bias, sp, alpha, theta, 0)
    got = run(gpu_ctx_factory(tc), shape, ho, wo, Wt, bias, sp, alpha, theta, 0)
    np.testing.assert_array_equal(got, ref, err_msg=f"{shape[0]} {what}")


@pytest.mark.parametrize("decay,th", [(0.5, 1.0), (0.95, 0.3), (-0.7, 0.5), (0.5, 0.0), (0.5, -0.5)])
@pytest.mark.parametrize("T,delta,C1,C2,C3", [(65, 13, 64, 128, 40), (128, 32, 9, 260, 33), (160, 32, 70, 64, 128),
                                              (255, 51, 33, 32, 600)])
def test_culif_engine_lists(gpu_ctx_factory, T, delta, C1, C2, C3, decay, th):
    print(f"culif lists T={T} {C1}-{C2}-{C3} decay={decay} th={th}", flush=True)
    B, H, W = 2, 7, 6
    rng = np.random.default_rng(T + C1)
    ev = (rng.random((B, 2, H, W, T)) < 0.06).astype(np.float32)
    ev[0, :, :4] = 0.0
    k = models.kaiming
    L = [vdttfs.CulifLayerSpec(vdttfs.CULIF_RAW_CONV, 2, H, W, C1, k(3, 0, (C1, 2, 3, 3), 18), None, 0.5, 1.0),
         vdttfs.CulifLayerSpec(vdttfs.CULIF_CONV, C1, H, W, C2, k(3, 1, (C2, C1, 3, 3), 9 * C1), None, decay, th),
         vdttfs.CulifLayerSpec(vdttfs.CULIF_CONV, C2, H, W, C3, k(3, 2, (C3, C2, 3, 3), 9 * C2), None, decay, th),
         vdttfs.CulifLayerSpec(vdttfs.CULIF_FC, C3 * H * W, 1, 1, 4, k(3, 3, (4, C3 * H * W), 99), None, 0.5, 1.0)]
    ref, _ = oracle.culif_net_forward(L, ev, B, T, delta)
    if th == 1.0:
        assert (ref[1] < INF).any() and (ref[1] == INF).any()
    net = vdttfs.CulifNet(gpu_ctx_factory(vdttfs.task3_consts(T=T, delta=delta)), L, B)
    try:
        net.forward(net.ctx.to_device(ev))
        net.ctx.synchronize()
        got = [net.layer_output(i) for i in range(4)]
    finally:
        net.close()
    for i in range(4):
        np.testing.assert_array_equal(got[i].reshape(-1), ref[i].reshape(-1), err_msg=f"layer {i}")
