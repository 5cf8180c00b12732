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
    ("t80-conv5-1-6", 80, 0, False, False, 3, 28, 28, 1, 6, 5),
    ("t80-conv5-6-16", 80, 0, False, False, 3, 12, 12, 6, 16, 5),
    ("t65-conv3-7-31", 65, 0, True, False, 3, 5, 6, 7, 31, 3),
    ("t80-fc-1600-128", 80, 0, True, True, 9, 1, 1, 1600, 128, 1),
    ("t80-fc-128-10", 80, 0, True, True, 17, 1, 1, 128, 10, 1),
    ("t200-fc-4100-700", 200, 0, False, True, 3, 1, 1, 4100, 700, 1),
    ("t65-fc-3-1", 65, 0, True, True, 5, 1, 1, 3, 1, 1),
]
# either side of the lengths up to which a layer takes the lists
LENGTHS = [
    ("t80-fc-4096-70", 80, 0, True, True, 33, 1, 1, 4096, 70, 1),
    ("t80-fc-4097-70", 80, 0, True, True, 33, 1, 1, 4097, 70, 1),
    ("t80-fc-8192-140", 80, 0, True, True, 4, 1, 1, 8192, 140, 1),
    ("t80-fc-8193-140", 80, 0, True, True, 4, 1, 1, 8193, 140, 1),
    ("t80-fc-8192-132-b65", 80, 0, True, True, 65, 1, 1, 8192, 132, 1),
    ("t80-conv3-256-140", 80, 0, True, False, 2, 5, 4, 256, 140, 3),
    ("t80-conv3-257-140", 80, 0, True, False, 2, 5, 4, 257, 140, 3),
    ("t80-conv3-455-20", 80, 0, True, False, 1, 5, 4, 455, 20, 3),
    ("t80-conv3-456-20", 80, 0, True, False, 1, 5, 4, 456, 20, 3),
    ("t80-conv5-128-20", 80, 0, True, False, 1, 5, 4, 128, 20, 5),
    ("t80-conv5-129-20", 80, 0, True, False, 1, 5, 4, 129, 20, 5),
    ("t80-conv5-200-140", 80, 0, True, False, 1, 5, 4, 200, 140, 5),
    ("t80-conv5-201-140", 80, 0, True, False, 1, 5, 4, 201, 140, 5),
]


@pytest.mark.parametrize("kind", ["random", "dense"])
@pytest.mark.parametrize("shape", LENGTHS, ids=[s[0] for s in LENGTHS])
def test_lists_lengths(gpu_ctx_factory, shape, kind):
    test_lists_match_oracle(gpu_ctx_factory, shape, kind)


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


@pytest.mark.parametrize("T,delta,K,C_in,C_out,is_fc", [(64, 16, 3, 20, 70, False), (80, 7, 5, 3, 6, False),
                                                        (255, 256, 1, 130, 33, False), (48, 1, 1, 300, 260, True)])
def test_any_bucket_contents(gpu_ctx_factory, T, delta, K, C_in, C_out, is_fc):
    """Buckets a caller may hand over: offsets that run backwards or past the
    column, times outside the chunk or the window, infinite and NaN, inputs
    past the width and repeated.  Past 1024 outputs the loop nest over the
    chunks runs; its first C_out outputs are the reference."""
    print(f"buckets T={T} delta={delta} K={K} {C_in}->{C_out}", flush=True)
    WIDE, B, H, W = 1030, 2, 5, 6
    if is_fc:
        H = W = 1
    tc = vdttfs.task2_consts(T=T, delta=delta, tfs=5.0)
    ctx = gpu_ctx_factory(tc)
    rng = np.random.default_rng(T)
    cols, NC = B * H * W, (T + delta - 1) // delta
    cin = rng.integers(-2, C_in + 3, (cols, C_in)).astype(np.int32)
    tin = np.sort(rng.random((cols, C_in)) * (T + 12) - 4, axis=1).astype(np.float32)
    tin[rng.random(tin.shape) < 0.02] = np.inf
    tin[rng.random(tin.shape) < 0.02] = np.nan
    tb = np.clip(np.nan_to_num(tin - 5.0, nan=0.0, posinf=1e6), 0, T).astype(int)
    off = np.stack([(tb < delta * i).sum(1) for i in range(NC + 1)], axis=1).astype(np.int32)
    wild = rng.random(off.shape) < 0.1
    off[wild] += rng.integers(-C_in, C_in, int(wild.sum())).astype(np.int32)
    Wt = (rng.standard_normal((K * K * C_in, WIDE)) * np.sqrt(2.0 / (K * K * C_in))).astype(np.float32)
    bias = (rng.standard_normal(WIDE) * 0.2).astype(np.float32)
    alpha, theta = vdttfs.build_luts_host(tc, 0.75 * T, 0.5, 1.5 * T, 2.5)
    d = [ctx.to_device(x) for x in (cin.reshape(-1), tin.reshape(-1), off.reshape(-1), alpha, theta)]
    outs = []
    for co in (WIDE, C_out):
        k, b = ctx.to_device(np.ascontiguousarray(Wt[:, :co])), ctx.to_device(bias[:co].copy())
        o = ctx.empty(cols * co).fill(0xFF)
        ctx.integrate(o, d[0], d[1], d[2], k, b, d[3], d[4], 2, B=B, H_in=H, W_in=W, C_in=C_in, H_out=H, W_out=W,
                      C_out=co, K_h=K, K_w=K, is_fc=is_fc)
        ctx.synchronize()
        outs.append(o.download().reshape(cols, co))
    assert (outs[1] < INF).any() and (outs[1] == INF).any()
    np.testing.assert_array_equal(outs[1], outs[0][:, :C_out])
