"""Narrow convolutions (one pixel per lane or per four lanes) against
the oracle, bit for bit: every field and output width of the kernel, odd ones
between them, padding, windows of one to four blocks of 64 bins, fire starts,
thresholds that do not fall, weights that are not finite, partial waves."""
import ctypes

import numpy as np
import pytest

import vdttfs
from test_gpu_split import case, reference, run

pytestmark = pytest.mark.gpu
INF = np.float32(9999.0)

# name, T, tfs, task2, is_fc, B, H, W, C_in, C_out, K
SHAPES = [
    ("t64-conv5-1-6", 64, 0, False, False, 3, 28, 28, 1, 6, 5),
    ("t64-conv3-1-4-same", 64, 0, True, False, 2, 7, 9, 1, 4, 3),
    ("t255-conv1-16-8", 255, 0, False, False, 5, 3, 4, 16, 8, 1),
    ("t80-conv3-3-16-same", 80, 20, True, False, 3, 9, 5, 3, 16, 3),
    ("t1-conv1-1-1", 1, 0, False, False, 2, 3, 3, 1, 1, 1),
    ("t65-conv2-8-11", 65, 0, False, False, 3, 6, 5, 8, 11, 2),
    ("t130-conv5-1-13-same", 130, 7, True, False, 2, 11, 6, 1, 13, 5),
    ("t33-conv3-2-9", 33, 0, False, False, 4, 5, 5, 2, 9, 3),
    ("t64-conv5-1-3-big", 64, 0, False, False, 90, 32, 32, 1, 3, 5),  # 256 threads a workgroup
    # four lanes a pixel: every width of theirs, odd sizes, padding
    ("t64-conv3-4-16-same", 64, 0, True, False, 9, 31, 30, 4, 16, 3),
    ("t80-conv3-7-5", 80, 0, False, False, 11, 30, 29, 7, 5, 3),
    ("t64-conv3-12-13-same", 64, 9, True, False, 9, 31, 30, 12, 13, 3),
    ("t64-conv5-6-16", 64, 0, False, False, 90, 31, 32, 6, 16, 5),
    ("t140-conv1-160-10", 140, 0, True, False, 80, 29, 29, 160, 10, 1),
    # nine outputs and more up to 64 steps: a lane per output below 12,288 pixels
    ("t64-conv5-1-16-few", 64, 0, False, False, 15, 32, 32, 1, 16, 5),
    ("t64-conv5-1-16-many", 64, 0, False, False, 16, 32, 32, 1, 16, 5),
    ("t64-conv3-3-9-same-few", 64, 0, True, False, 12, 32, 31, 3, 9, 3),
    ("t64-conv3-3-9-same-many", 64, 0, True, False, 13, 32, 31, 3, 9, 3),
    ("t64-conv1-16-10-few", 64, 0, True, False, 2, 9, 7, 16, 10, 1),
]
KINDS = ["random", "silent", "bin0", "last-bin", "dense", "fractional"]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("shape", SHAPES, ids=[s[0] for s in SHAPES])
def test_pixel_matches_oracle(gpu_ctx_factory, shape, kind):
    tc, ho, wo, Wt, bias, sp = case(shape, kind)
    T = tc.T
    alpha, theta = vdttfs.build_luts_host(tc, 0.75 * T, 0.5, 1.5 * T, 2.5)
    t_min = min(3, T - 1)
    ref = reference(shape, tc, ho, wo, Wt, bias, sp, alpha, theta, t_min)
    got = run(gpu_ctx_factory(tc), shape, ho, wo, Wt, bias, sp, alpha, theta, t_min)
    np.testing.assert_array_equal(got, ref, err_msg=f"{shape[0]} {kind}")


@pytest.mark.parametrize("shape", [SHAPES[0], SHAPES[3], SHAPES[6]], ids=lambda s: s[0])
@pytest.mark.parametrize("what", ["shuffled", "level", "below", "nan", "zero", "inf-weight", "nan-weight"])
def test_pixel_odd_tables_and_weights(gpu_ctx_factory, shape, what):
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
    elif what == "nan":
        theta = np.where(np.arange(T) == T // 3, np.nan, theta).astype(np.float32)
    elif what == "zero":
        theta = np.zeros(T, np.float32)
    else:
        Wt[rng.integers(0, Wt.shape[0], 4), rng.integers(0, Wt.shape[1], 4)] = np.nan if what == "nan-weight" else np.inf
    ref = reference(shape, tc, ho, wo, Wt, bias, sp, alpha, theta, 2)
    got = run(gpu_ctx_factory(tc), shape, ho, wo, Wt, bias, sp, alpha, theta, 2)
    np.testing.assert_array_equal(got, ref, err_msg=f"{shape[0]} {what}")


@pytest.mark.parametrize("T", [64, 80])
def test_pixel_layers_allocate_nothing(gpu_ctx_factory, T):
    """LeNet-5's conv2 at batch 1024 runs without lists, which would take 90 MB."""
    print(f"pixel scratch T={T}", flush=True)
    ctx = gpu_ctx_factory(vdttfs.task1_consts(T=T, delta=16))
    B, H, C_in, C_out, K = 1024, 12, 6, 16, 5
    rng = np.random.default_rng(T)
    sp = np.where(rng.random(B * H * H * C_in) < 0.3, np.floor(rng.random(B * H * H * C_in) * T), INF)
    alpha, theta = vdttfs.build_luts_host(vdttfs.task1_consts(T=T, delta=16), 16.0, 0.0, 16.0, 0.0)
    d = [ctx.to_device(v.astype(np.float32)) for v in (sp, rng.standard_normal((150, C_out)) * 0.1, np.zeros(C_out),
                                                       alpha, theta)]
    out = ctx.empty(B * 8 * 8 * C_out)

    def free_bytes():
        ctx.synchronize()
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert ctypes.CDLL("libamdhip64.so").hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    before = free_bytes()
    ctx.layer_forward(out, *d, 0, B, H, H, C_in, 8, 8, C_out, K, K, False)
    assert before - free_bytes() < 16 << 20  # a kernel's first launch may load its code
