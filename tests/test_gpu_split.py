"""The split integrator (bin 0 on the matrix cores, the later bins from
per-column lists) against the oracle, bit for bit.

SHAPES are layers of all kinds with few pixels: one to 25 taps, two bin blocks,
odd C_out (one load per column), C_in outside multiples of 8 and 16, lists past
a window's capacity, thresholds that are not monotone, non-finite weights,
t_min > 0, valid and same padding, and FC layers.  Those that the split takes
run its 16x16 tiles; the others run on the fused kernels or the column lists
and are compared all the same.  TILES are layers that the split takes (checked
against its size rule), with each tile of its matrix product: odd and even
C_out past whole tiles, C_in outside multiples of 8, partial pixel tiles, rows
in image and in (position, image) order, non-finite weights.
"""
import sys
import zlib

import numpy as np
import pytest

import oracle
import vdttfs

pytestmark = pytest.mark.gpu
INF = np.float32(9999.0)

# name, T, tfs, task2, is_fc, B, H, W, C_in, C_out, K
SHAPES = [
    ("t80-conv3-9-33", 80, 40, True, False, 3, 7, 5, 9, 33, 3),            # odd C_out, one wave
    ("t128-conv3-20-131", 128, 64, True, False, 2, 6, 7, 20, 131, 3),      # odd C_out past 128: three blocks
    ("t80-conv1-70-100", 80, 24, True, False, 5, 9, 4, 70, 100, 1),        # one tap, two events per load
    ("t80-conv3-valid-40-260", 80, 20, False, False, 4, 6, 5, 40, 260, 3),  # alpha by bin, several groups
    ("t80-conv2x2-130-140-b40", 80, 40, True, False, 40, 2, 2, 130, 140, 3),  # (position, image) rows
    ("t64-conv5-70-36", 64, 32, True, False, 3, 9, 8, 70, 36, 5),          # 25 taps, C_in past the dense merge
    ("t64-conv5-6-96", 64, 16, True, False, 2, 11, 6, 6, 96, 5),
    ("t64-conv3-128-96", 64, 32, True, False, 4, 3, 4, 128, 96, 3),        # a long field
    ("t48-conv3-256-256", 48, 24, True, False, 3, 3, 2, 256, 256, 3),
    ("t80-fc-600-260", 80, 40, True, True, 19, 1, 1, 600, 260, 1),
    ("t65-fc-30-40", 65, 17, False, True, 70, 1, 1, 30, 40, 1),
    ("t64-conv3-64-64-big", 64, 32, True, False, 40, 16, 16, 64, 64, 3),
]
# k_gemm0's tile of a wave (pixels x c_out), then a shape that takes it
TILES = [
    ((16, 16), ("t64-conv5-5-33-small", 64, 32, True, False, 7, 6, 7, 5, 33, 5)),
    ((16, 16), ("t128-conv3-65-131", 128, 64, True, False, 2, 6, 7, 65, 131, 3)),         # two bin blocks
    ((32, 32), ("t64-conv5-5-33", 64, 32, True, False, 147, 13, 11, 5, 33, 5)),
    ((32, 32), ("t64-conv5-3-34", 64, 32, False, False, 149, 13, 14, 3, 34, 5)),
    ((32, 32), ("t64-conv5-5-33-pos", 64, 32, True, False, 353, 5, 7, 5, 33, 5)),         # (position, image) rows
    ((32, 32), ("t64-conv3-20-70", 64, 32, True, False, 58, 13, 11, 20, 70, 3)),          # nine taps
    ((32, 64), ("t64-conv5-5-67", 64, 32, True, False, 153, 13, 11, 5, 67, 5)),
    ((32, 64), ("t64-conv5-3-66", 64, 16, True, False, 153, 13, 11, 3, 66, 5)),
    ((32, 64), ("t64-conv5-5-67-pos", 64, 32, True, False, 645, 5, 7, 5, 67, 5)),
    ((64, 64), ("t64-conv5-2-131", 64, 32, True, False, 737, 13, 11, 2, 131, 5)),
    ((64, 64), ("t64-conv5-2-130", 64, 32, True, False, 737, 13, 11, 2, 130, 5)),
    ((64, 64), ("t64-conv5-2-131-pos", 64, 32, True, False, 3001, 5, 7, 2, 131, 5)),
]
KINDS = ["random", "silent", "bin0", "one-late-bin", "last-bin", "late", "dense", "fractional"]


def spike_times(kind, n, T, tfs, rng):
    if kind == "random":
        t = np.floor(rng.random(n) * (T + tfs + 2)).astype(np.float32)
        return np.where(rng.random(n) < 0.5, t, INF).astype(np.float32)
    if kind == "dense":
        return np.floor(rng.random(n) * (T + tfs)).astype(np.float32)
    if kind == "late":  # every event past bin 0: lists in windows
        return np.floor(tfs + 1 + rng.random(n) * (T - 1)).astype(np.float32)
    if kind == "fractional":
        t = (rng.random(n) * (T + tfs + 1) - 2).astype(np.float32)
        return np.where(rng.random(n) < 0.6, t, INF).astype(np.float32)
    v = {"silent": INF, "bin0": float(tfs), "one-late-bin": float(tfs) + 5.0, "last-bin": float(T - 1) + tfs}[kind]
    return np.full(n, v, np.float32)


def case(shape, kind):
    name, T, tfs, task2, is_fc, B, H, W, C_in, C_out, K = shape
    print(f"split {name} {kind}", flush=True)
    sys.stdout.flush()
    rng = np.random.default_rng(zlib.crc32(f"split-{name}-{kind}".encode()))
    tc = vdttfs.TaskConsts(T=T, tfs=float(tfs), delta=8, vth=1.0, alpha_by_time=task2, conv_same_pad=task2)
    ho, wo = (1, 1) if is_fc else ((H, W) if task2 else (H - K + 1, W - K + 1))
    fan = C_in if is_fc else K * K * C_in
    Wt = (rng.standard_normal((fan, C_out)) * np.sqrt(2.0 / fan)).astype(np.float32)
    bias = (rng.standard_normal(C_out) * 0.4).astype(np.float32)
    sp = spike_times(kind, B * H * W * C_in, T, tfs, rng)
    return tc, ho, wo, Wt, bias, sp


def reference(shape, tc, ho, wo, Wt, bias, sp, alpha, theta, t_min):
    _, T, _, task2, is_fc, B, H, W, C_in, C_out, K = shape
    c = oracle.Consts.from_task(tc)
    cin, tin, off = oracle.bucketize(c, sp, B * H * W, C_in)
    res = oracle.integrate(c, cin, tin, off, Wt, bias, alpha, theta, t_min, B, H, W, C_in, ho, wo, C_out,
                           1 if is_fc else K, 1 if is_fc else K, K // 2 if task2 and not is_fc else 0, is_fc)
    return res[0]


def run(ctx, shape, ho, wo, Wt, bias, sp, alpha, theta, t_min):
    _, T, _, task2, is_fc, B, H, W, C_in, C_out, K = shape
    x, k, b = ctx.to_device(sp), ctx.to_device(Wt), ctx.to_device(bias)
    al, th = ctx.to_device(alpha), ctx.to_device(theta)
    out = ctx.empty(B * ho * wo * C_out).fill(0xFF)
    ctx.layer_forward(out, x, k, b, al, th, t_min, B, H, W, C_in, ho, wo, C_out, 1 if is_fc else K,
                      1 if is_fc else K, is_fc)
    ctx.synchronize()
    return out.download()


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("shape", SHAPES, ids=[s[0] for s in SHAPES])
def test_split_matches_oracle(gpu_ctx_factory, shape, kind):
    tc, ho, wo, Wt, bias, sp = case(shape, kind)
    T = tc.T
    alpha, theta = vdttfs.build_luts_host(tc, 0.75 * T, 0.5, 1.5 * T, 2.5)
    ref = reference(shape, tc, ho, wo, Wt, bias, sp, alpha, theta, 3)
    if kind in ("random", "late"):
        assert (ref < INF).any() and (ref == INF).any(), "the case must fire some neurons and not others"
    got = run(gpu_ctx_factory(tc), shape, ho, wo, Wt, bias, sp, alpha, theta, 3)
    np.testing.assert_array_equal(got, ref, err_msg=f"{shape[0]} {kind}")


def tile_of(shape):
    """The split's tile for a layer, or None where the split does not take it
    (its rules on sizes for at most 25 taps)."""
    _, T, tfs, task2, is_fc, B, H, W, C_in, C_out, K = shape
    taps = 1 if is_fc else K * K
    pix = B * (1 if is_fc else (H * W if task2 else (H - K + 1) * (W - K + 1)))
    nel = taps * C_in
    tiles = -(-pix // 32) * -(-C_out // 32)
    if C_out < 32 or 4 * tfs < T or T > 128:
        return None
    if taps > 9 and nel > (6400 if C_out > 128 and pix <= 512 else 3750):
        return None
    if T > 64:
        if nel <= 300 or taps == 1 or (nel <= 576 and pix <= 1024):
            return None
    elif taps > 9:
        if nel < 4:
            return None
    elif is_fc or tiles < 768 or nel < 144 or nel * pix * C_out < 10**8 or (2 * tfs < T and tiles < 4096):
        return None
    return (64, 64) if tiles >= 16384 else (32, 64) if tiles >= 2048 else (32, 32) if tiles >= 768 else (16, 16)


@pytest.mark.parametrize("kind", ["random", "bin0", "fractional"])
@pytest.mark.parametrize("tile,shape", TILES, ids=[t[1][0] for t in TILES])
def test_split_tiles(gpu_ctx_factory, tile, shape, kind):
    assert tile_of(shape) == tile
    test_split_matches_oracle(gpu_ctx_factory, shape, kind)


LINES = [  # either side of the lines that the split is chosen by
    ((32, 32), ("t64-conv3-20-70-768", 64, 32, True, False, 16, 32, 16, 20, 70, 3)),
    (None, ("t64-conv3-20-70-767", 64, 32, True, False, 15, 34, 16, 20, 70, 3)),
    (None, ("t64-conv3-20-70-early", 64, 31, True, False, 16, 32, 16, 20, 70, 3)),
    ((32, 64), ("t64-conv3-20-66-early", 64, 31, True, False, 45, 31, 32, 20, 66, 3)),
    # past 64 steps short fields and single taps take the column lists
    (None, ("t80-conv5-12-40", 80, 40, True, False, 17, 9, 7, 12, 40, 5)),
    ((16, 16), ("t80-conv5-13-40", 80, 40, True, False, 17, 9, 7, 13, 40, 5)),
    (None, ("t80-conv3-64-40", 80, 40, True, False, 3, 9, 7, 64, 40, 3)),
    ((16, 16), ("t80-conv3-65-40", 80, 40, True, False, 3, 9, 7, 65, 40, 3)),
    (None, ("t80-conv1-601-40", 80, 40, True, False, 3, 9, 7, 601, 40, 1)),
    # long fields of many taps the merged lists
    ((16, 16), ("t64-conv5-150-40", 64, 32, True, False, 2, 6, 5, 150, 40, 5)),
    (None, ("t64-conv5-151-40", 64, 32, True, False, 2, 6, 5, 151, 40, 5)),
    (None, ("t80-conv5-151-128", 80, 40, True, False, 2, 6, 5, 151, 128, 5)),
    ((16, 16), ("t64-conv5-256-132", 64, 32, True, False, 2, 6, 5, 256, 132, 5)),
    (None, ("t64-conv5-257-132", 64, 32, True, False, 2, 6, 5, 257, 132, 5)),
    (None, ("t64-conv5-151-132-513", 64, 32, True, False, 9, 19, 3, 151, 132, 5)),
    (None, ("t64-conv3-15-99", 64, 32, True, False, 16, 32, 16, 15, 99, 3)),
    ((32, 32), ("t64-conv3-16-99", 64, 32, True, False, 16, 32, 16, 16, 99, 3)),
]


@pytest.mark.parametrize("tile,shape", LINES, ids=[t[1][0] for t in LINES])
def test_split_lines(gpu_ctx_factory, tile, shape):
    assert tile_of(shape) == tile
    test_split_matches_oracle(gpu_ctx_factory, shape, "random")


@pytest.mark.parametrize("what", ["inf-weight", "nan-weight", "inf-row0"])
@pytest.mark.parametrize("tile,shape", [TILES[k] for k in (2, 4, 7, 8, 9, 10)],
                         ids=[TILES[k][1][0] for k in (2, 4, 7, 8, 9, 10)])
def test_split_tiles_non_finite_weights(gpu_ctx_factory, tile, shape, what):
    assert tile_of(shape) == tile
    test_split_odd_tables_and_weights(gpu_ctx_factory, shape, what)


@pytest.mark.parametrize("shape", [SHAPES[0], SHAPES[4], SHAPES[7]], ids=lambda s: s[0])
@pytest.mark.parametrize("what", ["shuffled", "level", "below", "steep", "inf-weight", "nan-weight", "inf-row0"])
def test_split_odd_tables_and_weights(gpu_ctx_factory, shape, what):
    """Thresholds that defeat the tail's guess (shuffled, all equal, a run
    below 1e-5, a steep fall), and weights that are not finite: only elements
    with an event may bring them into a sum."""
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
        bad = np.float32(np.nan if what == "nan-weight" else np.inf)
        at = [0] if what == "inf-row0" else rng.integers(0, Wt.shape[0], 6)
        Wt[at, rng.integers(0, Wt.shape[1], len(at))] = bad
        Wt[at[0], :] = bad
    ref = reference(shape, tc, ho, wo, Wt, bias, sp, alpha, theta, 0)
    got = run(gpu_ctx_factory(tc), shape, ho, wo, Wt, bias, sp, alpha, theta, 0)
    np.testing.assert_array_equal(got, ref, err_msg=f"{shape[0]} {what}")
