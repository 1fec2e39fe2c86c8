"""Implicit-GEMM convs on the bf16 matrix cores (fp32 operands as three bf16 parts each).

Forced onto shapes at the edges of its tiles and loaders and compared with a float64
convolution. Bound: an operand's three parts are exact, the products left out stay below
2^-24 of theirs, and the sum is rounded once per 32 k, so the relative L2 error stays below
2^-24 (2 + sqrt(K / 32)); twice that is allowed. Inputs that bf16 parts cannot carry
(infinities, NaN, magnitudes that round to infinity or lose bits) must give what fp32
arithmetic gives.
"""
import ctypes as C
import math
import zlib

import numpy as np
import pytest

from tests.hipops import conv_desc, run_conv

pytestmark = pytest.mark.gpu

# (n, c, h, w, oc, k, stride, pad, group, act)
SHAPES = [
    (1, 16, 8, 8, 64, 1, 1, 0, 1, 0),      # smallest K, one column tile, one row tile
    (2, 64, 7, 10, 65, 1, 1, 0, 1, 5),     # even plane, 2-pixel loads, one row past a tile, residual
    (3, 72, 7, 7, 130, 1, 1, 0, 1, 3),     # odd plane: gather loads; K no multiple of a slice group
    (2, 61, 9, 11, 128, 1, 1, 0, 1, 1),    # channels no multiple of 8, ragged columns
    (1, 16, 13, 13, 96, 3, 2, 1, 1, 1),    # two octets per tap, stride 2
    (2, 24, 12, 9, 64, 3, 1, 1, 1, 4),     # three octets per tap, residual
    (1, 19, 10, 10, 80, 5, 2, 2, 1, 0),    # 5x5, channel tail, asymmetric remainder
    (1, 96, 9, 9, 192, 3, 1, 1, 3, 3),     # grouped
    (2, 512, 6, 6, 128, 3, 1, 0, 1, 1),    # long K, no padding
]


@pytest.fixture
def tune(hip):
    L = hip.lib()
    yield L.spinn_hip_tune_split_conv
    L.spinn_hip_tune_split_conv(-1, 0, 0)
    L.spinn_hip_tune_streamk(-1)


def _case(shape):
    n, c, h, w, oc, k, s, p, g, act = shape
    rng = np.random.default_rng(zlib.crc32(repr(shape).encode()))
    x = rng.standard_normal((n, c, h, w)).astype(np.float32)
    wt = (rng.standard_normal((oc, c // g, k, k)) * math.sqrt(2.0 / (c // g * k * k))).astype(np.float32)
    b = rng.normal(0, 0.1, oc).astype(np.float32)
    oh, ow = (h + 2 * p - k) // s + 1, (w + 2 * p - k) // s + 1
    r = rng.standard_normal((n, oc, oh, ow)).astype(np.float32) if act in (4, 5) else None
    return x, wt, b, r


def _exact(torch, shape, x, wt, b, r):
    n, c, h, w, oc, k, s, p, g, act = shape
    y = torch.nn.functional.conv2d(torch.from_numpy(x).double(), torch.from_numpy(wt).double(),
                                   torch.from_numpy(b).double(), s, p, 1, g)
    if r is not None:
        y = y + torch.from_numpy(r).double()
    if act in (1, 5):
        y = torch.where(y < 0, torch.zeros_like(y), y)
    elif act == 3:
        y = torch.nn.functional.silu(y)
    return y.numpy()


@pytest.mark.parametrize("bm,split,streamk", [(64, 1, -1), (128, 1, -1), (64, 3, -1), (128, 2, -1), (64, 0, 1)],
                         ids=["64", "128", "64_ksplit3", "128_ksplit2", "64_streamk"])
@pytest.mark.parametrize("shape", SHAPES, ids=[repr(s) for s in SHAPES])
def test_split_conv(hip, torch_gpu, tune, shape, bm, split, streamk):
    torch = torch_gpu
    n, c, h, w, oc, k, s, p, g, act = shape
    if streamk == 1 and g == 1:  # more than a tile per CU (test_split_conv_streamk: real cuts)
        tune(1, bm, split)
        hip.lib().spinn_hip_tune_streamk(streamk)
        n = 256 * 64 // (((h + 2 * p - k) // s + 1) * ((w + 2 * p - k) // s + 1) * ((oc + 63) // 64))
        while hip.lib().spinn_hip_conv_workspace_size(C.byref(conv_desc(
                hip, n, c, h, w, oc, k, k, s, s, p, p, g, act, hip.ALGO_IMPLICIT_GEMM))) == 0:
            n += 1
        shape = (n,) + shape[1:]
    print(f"[split conv] {shape} bm {bm} split {split} stream-K {streamk}", flush=True)
    tune(1, bm, split)
    hip.lib().spinn_hip_tune_streamk(streamk)
    x, wt, b, r = _case(shape)
    d = conv_desc(hip, n, c, h, w, oc, k, k, s, s, p, p, g, act, hip.ALGO_IMPLICIT_GEMM)
    y, _ = run_conv(hip, torch, d, x, wt, b, r)
    ref = _exact(torch, shape, x, wt, b, r)
    rel = np.linalg.norm(y - ref) / np.linalg.norm(ref)
    bound = 2 * 2.0 ** -24 * (2 + math.sqrt(c // g * k * k / 32))
    if act == 3:
        bound += 1e-6  # the hardware exp2 and reciprocal of SiLU
    assert rel <= bound, f"relative error {rel:.2e} above {bound:.2e}"


@pytest.mark.parametrize("shape", [SHAPES[1], SHAPES[4]], ids=["1x1", "3x3s2"])
def test_split_conv_special_values(hip, torch_gpu, tune, shape):
    """Infinities, NaN, values that round to infinity in bf16 and tiny ones, in the input,
    the weights and the residual."""
    torch = torch_gpu
    n, c, h, w, oc, k, s, p, g, act = shape
    tune(1, 64, 1)
    x, wt, b, r = _case(shape)
    x[0, 3, 2, 2], x[0, 5, 4, 7] = np.inf, np.nan
    x[-1, 2, 5, 5] = 3.4e38
    x[-1, 7, 0, 0] = 1e-30
    x[:, 1] *= 1e-3
    x[0, 1, 6, 5] = -np.inf
    wt[1] *= 1e-6
    wt[2, 0, 0, 0], wt[4, 1, 0, 0] = np.inf, 3.4e38
    if r is not None:
        r[0, 5, 1, 1] = np.inf
    d = conv_desc(hip, n, c, h, w, oc, k, k, s, s, p, p, g, act, hip.ALGO_IMPLICIT_GEMM)
    y, _ = run_conv(hip, torch, d, x, wt, b, r)
    with np.errstate(over="ignore", invalid="ignore"):
        ref = _exact(torch, shape, x, wt, b, r)
    big = np.abs(ref) > 1e37
    bad = np.argwhere(np.isnan(y) != np.isnan(ref))
    assert len(bad) == 0, [(tuple(i), y[tuple(i)], ref[tuple(i)]) for i in bad[:8]]
    inf = np.isinf(ref)
    assert np.array_equal(y[inf], ref[inf].astype(np.float32))
    ok = np.isfinite(ref) & ~big
    assert ok.any() and inf.any()
    assert np.abs(y[ok] - ref[ok]).max() <= 1e-5 * max(1.0, np.abs(ref[ok]).max())


@pytest.mark.parametrize("sx,sw", [(1e-36, 1.0), (1.0, 1e-36), (1e-20, 1e-16), (1e30, 1e5)])
@pytest.mark.parametrize("shape", [(2, 64, 7, 10, 65, 1, 1, 0, 1, 0), (1, 19, 10, 10, 80, 3, 1, 1, 1, 0)],
                         ids=["1x1", "3x3_tail"])
def test_split_conv_scales(hip, torch_gpu, tune, shape, sx, sw):
    """Magnitudes whose low parts lie under bf16's least number, and large ones: the error
    stays relative to the result."""
    n, c, h, w, oc, k, s, p, g, act = shape
    tune(1, 64, 1)
    x, wt, _, _ = _case(shape)
    x, wt = (x * np.float32(sx)).astype(np.float32), (wt * np.float32(sw)).astype(np.float32)
    d = conv_desc(hip, n, c, h, w, oc, k, k, s, s, p, p, g, act, hip.ALGO_IMPLICIT_GEMM)
    y, _ = run_conv(hip, torch_gpu, d, x, wt)
    ref = _exact(torch_gpu, shape, x, wt, np.zeros(oc, np.float32), None)
    scale = ref.std()
    rel = np.linalg.norm(y / scale - ref / scale) / np.linalg.norm(ref / scale)
    # fp32 sums of K terms in two-term steps on the fp32 path
    assert rel <= 2 * 2.0 ** -24 * (2 + math.sqrt(c * k * k / 2))


@pytest.mark.parametrize("bm,split", [(64, 1), (128, 1), (64, 3), (128, 2)])
@pytest.mark.parametrize("sx,sw", [(1e-36, 1e30), (1e30, 1e-36), (1e-37, 1e37), (1e37, 1e-37), (1e-40, 1e37),
                                   (1e37, 1e-40), (1e-36, 1e14), (1e-42, 1e30), (1e-42, 1e4), (1.0, 1e-30)])
@pytest.mark.parametrize("shape", [(2, 64, 7, 10, 65, 1, 1, 0, 1, 0), (1, 19, 10, 10, 80, 3, 1, 1, 1, 0),
                                   (2, 256, 6, 6, 130, 1, 1, 0, 2, 0)], ids=["1x1", "3x3_tail", "grouped"])
def test_split_conv_tiny_times_large(hip, torch_gpu, tune, shape, sx, sw, bm, split):
    """Operands that three bf16 parts cannot hold, in ordinary sums: the other operand makes up
    for them, or every part is zero."""
    n, c, h, w, oc, k, s, p, g, act = shape
    print(f"[split conv] {shape} x {sx} w {sw} bm {bm} split {split}", flush=True)
    tune(1, bm, split)
    x, wt, _, _ = _case(shape)
    x, wt = (x * np.float32(sx)).astype(np.float32), (wt * np.float32(sw)).astype(np.float32)
    d = conv_desc(hip, n, c, h, w, oc, k, k, s, s, p, p, g, act, hip.ALGO_IMPLICIT_GEMM)
    y, _ = run_conv(hip, torch_gpu, d, x, wt)
    ref = _exact(torch_gpu, shape, x, wt, np.zeros(oc, np.float32), None)
    scale = ref.std()
    rel = np.linalg.norm(y / scale - ref / scale) / np.linalg.norm(ref / scale)
    # fp32 sums of K terms in two-term steps, and fp32's own least number in sums near it
    kk = c // g * k * k
    assert rel <= 2 * 2.0 ** -24 * (2 + math.sqrt(kk / 2)) + math.sqrt(kk) * 2.0 ** -149 / scale


@pytest.mark.parametrize("bm,split", [(64, 1), (128, 1), (64, 2)])
@pytest.mark.parametrize("k", [1, 3])
def test_split_conv_tiny_operand_of_one_channel(hip, torch_gpu, tune, k, bm, split):
    """One channel holds tiny inputs under large weights, or the reverse; the others are ordinary
    but meet zeros, so the sums are the odd channel's alone and look like any others."""
    n, c, hw, oc = 2, 96, 8, 128
    tune(1, bm, split)
    rng = np.random.default_rng(5)
    x = rng.standard_normal((n, c, hw, hw)).astype(np.float32)
    wt = rng.standard_normal((oc, c, k, k)).astype(np.float32)
    x[:, ::2], wt[:, 1::2] = 0, 0           # every product is zero ...
    x[:, 70] = rng.uniform(1, 2, x[:, 70].shape) * 2.0 ** -130
    wt[:64, 70] *= np.float32(2.0 ** 100)   # ... but this channel's
    wt[64:, 70] *= np.float32(2.0 ** 10)
    x[0, 70] *= np.float32(2.0 ** 120)
    wt[5, 70] *= np.float32(2.0 ** -225)
    d = conv_desc(hip, n, c, hw, hw, oc, k, k, 1, 1, k // 2, k // 2, 1, 0, hip.ALGO_IMPLICIT_GEMM)
    y, _ = run_conv(hip, torch_gpu, d, x, wt)
    shape = (n, c, hw, hw, oc, k, 1, k // 2, 1, 0)
    ref = _exact(torch_gpu, shape, x, wt, np.zeros(oc, np.float32), None)
    size = np.sqrt((ref ** 2).mean((2, 3), keepdims=True))  # per image and output channel
    # nine terms at most; 2^-149 where a sum is that small
    assert (np.abs(y - ref) <= 16 * 2.0 ** -24 * size + 9 * 2.0 ** -149).all()


@pytest.mark.parametrize("bm", [64, 128])
@pytest.mark.parametrize("hw", [8, 9])  # whole and ragged tiles; 2-pixel and 1-pixel loads
@pytest.mark.parametrize("row", [16, 33, 50, 67])
def test_split_conv_tiny_sums_of_one_row(hip, torch_gpu, tune, row, hw, bm):
    """Tiny inputs that reach a single output channel, among channels of ordinary sums."""
    n, c, oc = 1, 64, 128
    tune(1, bm, 1)
    rng = np.random.default_rng(row)
    x = rng.standard_normal((n, c, hw, hw)).astype(np.float32)
    wt = rng.standard_normal((oc, c, 1, 1)).astype(np.float32)
    x[:, 9] = rng.uniform(1, 2, x[:, 9].shape) * 2.0 ** -126
    wt[:, 9], wt[row], wt[row, 9] = 0, 0, 1.5
    d = conv_desc(hip, n, c, hw, hw, oc, 1, 1, 1, 1, 0, 0, 1, 0, hip.ALGO_IMPLICIT_GEMM)
    y, _ = run_conv(hip, torch_gpu, d, x, wt)
    ref = x[:, 9].astype(np.float64) * 1.5
    assert (np.abs(y[:, row] - ref) <= 2.0 ** -149).all()


# (n, c, h, w, oc, k, stride, pad, group, act), tile rows: what the cut is
STREAMK = [
    ((64, 256, 14, 14, 128, 1, 1, 0, 1, 1), 64),    # 392 tiles of 4 groups: extra workgroups
    ((64, 256, 14, 14, 256, 1, 1, 0, 1, 5), 128),   # the same, 128 rows and a residual
    ((136, 256, 14, 14, 128, 1, 1, 0, 1, 1), 64),   # 834: parts in whole-tile workgroups
    ((32, 256, 14, 14, 1024, 1, 1, 0, 1, 5), 0),    # 784 128-row tiles, by the rule
    ((64, 64, 14, 14, 128, 3, 1, 1, 1, 5), 64),     # 1-pixel loads, 9 groups
    ((64, 64, 14, 14, 256, 3, 1, 1, 1, 0), 128),
    ((64, 250, 14, 14, 128, 1, 1, 0, 1, 3), 64),    # a channel tail
    ((64, 250, 14, 14, 256, 1, 1, 0, 1, 1), 128),
]


@pytest.mark.parametrize("special", [False, True], ids=["plain", "special"])
@pytest.mark.parametrize("case", STREAMK, ids=[repr(c) for c in STREAMK])
def test_split_conv_streamk(hip, torch_gpu, tune, case, special):
    """Remaining tiles cut along K, each part starting inside it."""
    shape, bm = case
    n, c, h, w, oc, k, s, p, g, act = shape
    print(f"[split conv stream-K] {case} special {special}", flush=True)
    if bm:
        tune(1, bm, 0)
        hip.lib().spinn_hip_tune_streamk(1)
    d = conv_desc(hip, n, c, h, w, oc, k, k, s, s, p, p, g, act, hip.ALGO_IMPLICIT_GEMM)
    assert hip.lib().spinn_hip_conv_uses_bf16_parts(C.byref(d)) == 1
    ws = hip.lib().spinn_hip_conv_workspace_size(C.byref(d))
    assert ws > 0 and ws % (4 * n * oc * h * w) != 0, "a K split's workspace holds whole outputs"
    x, wt, b, r = _case(shape)
    if special:
        _plant(shape, x, wt, r)
    y, _ = run_conv(hip, torch_gpu, d, x, wt, b, r)
    _check(torch_gpu, shape, x, wt, b, r, y)


def _plant(shape, x, wt, r):
    """Infinities, NaN, values that round to infinity in bf16, tiny and subnormal ones."""
    n, c, h, w = shape[:4]
    ww = wt.reshape(wt.shape[0], -1)
    x[0, 3, 2, 2], x[0, 5, 4, 3] = np.inf, np.nan
    x[-1, 2, 5, 5], x[-1, 7, 0, 0], x[n // 2, c - 1, h - 1, w - 1] = 3.4e38, 1e-30, -np.inf
    x[:, 1] *= np.float32(1e-3)
    x[:, 4] *= np.float32(1e-36)
    wt[1] *= np.float32(1e-6)
    wt[3] *= np.float32(1e-36)
    wt[5] *= np.float32(1e-42)
    wt[7] *= np.float32(1e20)
    wt[9] = 0
    ww[2, 0], ww[4, ww.shape[1] - 1], ww[6, ww.shape[1] // 2] = np.inf, 3.4e38, np.nan
    if r is not None:
        r[0, 5, 1, 1] = np.inf


def _check(torch, shape, x, wt, b, r, y):
    """Every element against fp32 arithmetic: the same non-finite ones; finite ones within the
    roundings of a sum of K terms in two-term steps, each at most 2^-24 of the terms' magnitudes
    (and six products each off by fp32's least number). Sums near fp32's largest are skipped."""
    n, c, h, w, oc, k, s, p, g, act = shape
    kk = c // g * k * k
    with np.errstate(over="ignore", invalid="ignore"):
        ref = _exact(torch, shape, x, wt, b, r)
    ab = [None if a is None else np.abs(np.nan_to_num(a, nan=0.0, posinf=0.0, neginf=0.0)) for a in (x, wt, b, r)]
    size = _exact(torch, shape[:9] + ((4,) if r is not None else (0,)), *ab)
    fits = size < 1e38
    assert fits.mean() > 0.5
    nan = np.isnan(ref)
    bad = np.argwhere((np.isnan(y) != nan) & (fits | nan))
    assert len(bad) == 0, [(tuple(i), y[tuple(i)], ref[tuple(i)]) for i in bad[:8]]
    inf = np.isinf(ref) & fits
    assert np.array_equal(y[inf], ref[inf].astype(np.float32))
    ok = np.isfinite(ref) & fits
    assert ok.any()
    err = np.abs(y[ok] - ref[ok])
    lim = (kk / 2 + 8) * 2.0 ** -24 * size[ok] + 6 * kk * 2.0 ** -149
    if act == 3:
        lim = lim * 1.2 + 1e-6 * np.abs(ref[ok])  # silu's slope stays under 1.1; hardware exp2
    worst = np.argmax(err - lim)
    assert err[worst] <= lim[worst], (err[worst], lim[worst], y[ok][worst], ref[ok][worst])


@pytest.mark.parametrize("bm,split", [(64, 1), (128, 1), (64, 3), (128, 2)])
@pytest.mark.parametrize("shape", SHAPES, ids=[repr(s) for s in SHAPES])
def test_split_conv_special_elements(hip, torch_gpu, tune, shape, bm, split):
    """Special values on every loader, tile and K split, each element on its own."""
    n, c, h, w, oc, k, s, p, g, act = shape
    print(f"[split conv special] {shape} bm {bm} split {split}", flush=True)
    tune(1, bm, split)
    x, wt, b, r = _case(shape)
    _plant(shape, x, wt, r)
    d = conv_desc(hip, n, c, h, w, oc, k, k, s, s, p, p, g, act, hip.ALGO_IMPLICIT_GEMM)
    y, _ = run_conv(hip, torch_gpu, d, x, wt, b, r)
    _check(torch_gpu, shape, x, wt, b, r, y)
