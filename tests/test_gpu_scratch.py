"""The context's scratch of the split and list kernels: a call that has run once
can be captured, and the captured graph stays right when later calls grow the
scratch; a call whose scratch is not there yet is refused under capture without
ending it."""
import ctypes
import zlib

import numpy as np
import pytest

import oracle
import vdttfs
from vdttfs import _lib
from test_gpu_split import case, reference

pytestmark = pytest.mark.gpu
RELAXED = 2  # hipStreamCaptureModeRelaxed


def hip():
    lib = ctypes.CDLL("libamdhip64.so")
    for f in ("hipStreamBeginCapture", "hipStreamEndCapture", "hipGraphInstantiate", "hipGraphLaunch",
              "hipGraphExecDestroy", "hipGraphDestroy", "hipStreamIsCapturing", "hipMemGetInfo"):
        getattr(lib, f).restype = ctypes.c_int
    return lib


def stream_of(ctx):
    """The context's stream: the first pointer after its constants and three ints."""
    at = (ctypes.sizeof(_lib.Consts) + 3 * 4 + 7) // 8 * 8
    h = ctx.handle
    return ctypes.c_void_p.from_address((h.value if isinstance(h, ctypes.c_void_p) else int(h)) + at)


class Captured:
    def __init__(self, ctx, call):
        self.h, self.s = hip(), stream_of(ctx)
        graph, self.exe = ctypes.c_void_p(), ctypes.c_void_p()
        assert self.h.hipStreamBeginCapture(self.s, RELAXED) == 0
        try:
            call()
        finally:
            rc = self.h.hipStreamEndCapture(self.s, ctypes.byref(graph))
        assert rc == 0 and graph
        assert self.h.hipGraphInstantiate(ctypes.byref(self.exe), graph, None, None, ctypes.c_size_t(0)) == 0
        assert self.h.hipGraphDestroy(graph) == 0

    def replay(self):
        assert self.h.hipGraphLaunch(self.exe, self.s) == 0

    def close(self):
        self.h.hipGraphExecDestroy(self.exe)


# name, T, tfs, task2, is_fc, B, H, W, C_in, C_out, K
SHAPES = [
    ("t80-conv3-9-33", 80, 40, True, False, 3, 7, 5, 9, 33, 3),
    ("t80-conv3-40-70", 80, 0, True, False, 3, 7, 5, 40, 70, 3),
    ("t80-fc-600-260", 80, 40, True, True, 19, 1, 1, 600, 260, 1),
    ("t64-conv5-70-36", 64, 32, True, False, 3, 9, 8, 70, 36, 5),
    ("t80-conv5-1-6", 80, 0, False, False, 3, 28, 28, 1, 6, 5),
]


def layer_call(ctx, shape, seed_kind="random", batch=None):
    name, T, tfs, task2, is_fc, B, H, W, C_in, C_out, K = shape
    if batch:
        shape = shape[:5] + (batch,) + shape[6:]
        B = batch
    tc, ho, wo, Wt, bias, sp = case(shape, seed_kind)
    alpha, theta = vdttfs.build_luts_host(tc, 0.75 * T, 0.5, 1.5 * T, 2.5)
    d = [ctx.to_device(v) for v in (sp, Wt, bias, alpha, theta)]
    out = ctx.empty(B * ho * wo * C_out).fill(0xFF)

    def call():
        ctx.layer_forward(out, *d, 3, B, H, W, C_in, ho, wo, C_out, 1 if is_fc else K, 1 if is_fc else K, is_fc)

    return call, out, reference(shape, tc, ho, wo, Wt, bias, sp, alpha, theta, 3)


def test_captured_after_one_call(gpu_ctx_factory):
    for shape in SHAPES:
        print(f"scratch capture {shape[0]}", flush=True)
        tc = vdttfs.TaskConsts(T=shape[1], tfs=float(shape[2]), delta=8, vth=1.0, alpha_by_time=shape[3],
                               conv_same_pad=shape[3])
        ctx = gpu_ctx_factory(tc)
        call, out, ref = layer_call(ctx, shape)
        call()
        ctx.synchronize()
        np.testing.assert_array_equal(out.download(), ref)
        g = Captured(ctx, call)
        big, big_out, big_ref = layer_call(ctx, shape, batch=4 * shape[5])  # grows the scratch that the graph holds
        for _ in range(3):
            out.fill(0xFF)
            g.replay()
            ctx.synchronize()
            np.testing.assert_array_equal(out.download(), ref, err_msg=shape[0])
            big_out.fill(0xFF)
            big()
            ctx.synchronize()
            np.testing.assert_array_equal(big_out.download(), big_ref, err_msg=shape[0])
        g.close()


def test_bucket_integration_captured(gpu_ctx_factory):
    """vdttfs_integrate under capture, without lists' scratch (the loop nest)
    and with it, against an eager call."""
    print("scratch capture integrate", flush=True)
    tc = vdttfs.task2_consts(T=48, delta=8, tfs=12.0)
    B, H, W, C_in, C_out, K = 2, 6, 5, 24, 70, 3
    rng = np.random.default_rng(zlib.crc32(b"capture-integrate"))
    sp = np.where(rng.random(B * H * W * C_in) < 0.5, np.floor(rng.random(B * H * W * C_in) * 56), 9999.0)
    c = oracle.Consts.from_task(tc)
    cin, tin, off = oracle.bucketize(c, sp.astype(np.float32), B * H * W, C_in)
    Wt = (rng.standard_normal((K * K * C_in, C_out)) * np.sqrt(2.0 / (K * K * C_in))).astype(np.float32)
    bias = (rng.standard_normal(C_out) * 0.3).astype(np.float32)
    alpha, theta = vdttfs.build_luts_host(tc, 36.0, 0.5, 72.0, 2.5)
    ref = oracle.integrate(c, cin, tin, off, Wt, bias, alpha, theta, 2, B, H, W, C_in, H, W, C_out, K, K, K // 2,
                           False)[0]
    ctx = gpu_ctx_factory(tc)
    d = [ctx.to_device(np.ascontiguousarray(v).reshape(-1)) for v in (cin, tin, off, Wt, bias, alpha, theta)]
    out = ctx.empty(B * H * W * C_out)

    def call():
        ctx.integrate(out, *d, 2, B=B, H_in=H, W_in=W, C_in=C_in, H_out=H, W_out=W, C_out=C_out, K_h=K, K_w=K,
                      is_fc=False)

    for warm in (False, True):
        if warm:
            call()
            ctx.synchronize()
        g = Captured(ctx, call)
        for _ in range(3):
            out.fill(0xFF)
            g.replay()
            ctx.synchronize()
            np.testing.assert_array_equal(out.download(), ref, err_msg=f"warm={warm}")
        g.close()


def test_capture_without_scratch_is_refused_whole(gpu_ctx_factory):
    print("scratch capture refused", flush=True)
    shape = SHAPES[3]  # 25 taps past the dense merge: bucketize and merged lists where the split has no scratch
    tc = vdttfs.TaskConsts(T=64, tfs=32.0, delta=8, vth=1.0, alpha_by_time=True, conv_same_pad=True)
    ctx = gpu_ctx_factory(tc)
    call, out, ref = layer_call(ctx, shape)

    def refused():
        with pytest.raises(vdttfs.VdttfsError) as e:
            call()
        assert e.value.code == _lib.E_UNSUPPORTED and "capture" in str(e.value)

    g = None
    h, s = hip(), stream_of(ctx)
    graph = ctypes.c_void_p()
    assert h.hipStreamBeginCapture(s, RELAXED) == 0
    refused()
    assert h.hipStreamEndCapture(s, ctypes.byref(graph)) == 0
    h.hipGraphDestroy(graph)
    call()  # the context goes on
    ctx.synchronize()
    np.testing.assert_array_equal(out.download(), ref)
    g = Captured(ctx, call)
    out.fill(0xFF)
    g.replay()
    ctx.synchronize()
    np.testing.assert_array_equal(out.download(), ref)
    g.close()


@pytest.mark.parametrize("shape", [SHAPES[1], SHAPES[3]], ids=lambda s: s[0])
def test_counting_call_finds_its_scratch(gpu_ctx_factory, shape):
    """A layer's first call also sizes what its counting call takes (merged
    lists of 50 MB and more here): the counting call allocates nothing."""
    print(f"scratch counting {shape[0]}", flush=True)
    shape = shape[:5] + (96, 12, 12) + shape[8:]
    name, T, tfs, task2, is_fc, B, H, W, C_in, C_out, K = shape
    tc, ho, wo, Wt, bias, sp = case(shape, "random")
    ctx = gpu_ctx_factory(tc)
    alpha, theta = vdttfs.build_luts_host(tc, 0.75 * T, 0.5, 1.5 * T, 2.5)
    d = [ctx.to_device(v) for v in (sp, Wt, bias, alpha, theta)]
    out, again = ctx.empty(B * ho * wo * C_out), ctx.empty(B * ho * wo * C_out)
    free, total = ctypes.c_size_t(), ctypes.c_size_t()

    def free_bytes():
        ctx.synchronize()
        assert hip().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    ctx.layer_forward(out, *d, 3, B, H, W, C_in, ho, wo, C_out, K, K, False)
    before = free_bytes()
    eproc, _ = ctx.layer_forward(again, *d, 3, B, H, W, C_in, ho, wo, C_out, K, K, False, count=True)
    assert eproc > 0 and before - free_bytes() < 16 << 20  # a kernel's first launch may load its code
    np.testing.assert_array_equal(again.download(), out.download())


def test_network_sizes_lists_for_the_layers_that_use_them(gpu_ctx_factory):
    """An FC layer at T = 64 never takes the split kernels, whose scratch would
    be half as large again as its merged lists (402 against 269 MB)."""
    print("scratch network creation", flush=True)
    B, cin, cout, T = 2048, 16384, 64, 64
    ctx = gpu_ctx_factory(vdttfs.task2_consts(T=T, delta=8, tfs=32.0))
    layer = vdttfs.Layer(vdttfs.LAYER_FC, 1, 1, cin, 1, 1, cout, kernel=np.zeros((cin, cout), np.float32),
                         bias=np.zeros(cout, np.float32), tc_fire=16.0)
    free, total = ctypes.c_size_t(), ctypes.c_size_t()

    def free_bytes():
        ctx.synchronize()
        assert hip().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    before = free_bytes()
    net = vdttfs.Net(ctx, [layer], B, cin, vdttfs.ENCODE_LINEAR, 16.0, 0.0, vdttfs.READOUT_ARGMIN)
    used = before - free_bytes()
    net.close()
    lists, events, maps = B * (cin + 64) * 8, B * cin * 8, 4 * B * (cin + cout)
    assert used < lists + events + maps + 4 * cin * cout + (64 << 20), used
