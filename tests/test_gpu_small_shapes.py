"""Gemms on 16 x 16 wave-K tiles and on few 64 x 64 tiles, and ReduceMax over short rows.

Gemm bound: an fp32 sum of K terms in at most K / 8 roundings of at most 2^-24 each, which
add like a random walk: 2^-24 (4 + sqrt(K / 8)); twice that is allowed.
"""
import math

import numpy as np
import pytest

from tests.hipops import run_gemm

pytestmark = pytest.mark.gpu

# (m, n, k, trans_a, trans_b, batch)
GEMMS = [
    (5, 16, 64, 0, 1, 1),        # one row of tiles, the shortest K
    (33, 49, 67, 0, 0, 1),       # ragged in every direction
    (256, 256, 1024, 1, 0, 1),   # exactly one 16 x 16 tile per CU, the longest K
    (17, 130, 1021, 1, 1, 1),
    (64, 400, 400, 0, 1, 2),
    (64, 400, 400, 0, 1, 32),    # 224 64 x 64 tiles
    (65, 129, 576, 0, 0, 22),    # ragged 64 x 64 tiles
    (500, 1000, 130, 1, 1, 1),   # 128 of them
    (960, 1088, 128, 0, 1, 1),   # 255: the most with four accumulator sets
    (1024, 1024, 128, 0, 1, 1),  # 256: one set
    (832, 1024, 576, 0, 1, 1),   # 208: the fewest on 64 x 64 tiles
    (832, 960, 576, 0, 0, 1),    # 195: 32 x 32 wave-K
    (32, 8192, 128, 0, 1, 1),    # 32 rows: 32 x 32 wave-K
    (32, 400, 400, 0, 1, 32),
    (512, 1024, 512, 1, 0, 1),   # 128 tiles at K = 512: 32 x 32 wave-K, not split K
]


@pytest.mark.parametrize("case", GEMMS, ids=[repr(c) for c in GEMMS])
def test_gemm_few_tiles(hip, torch_gpu, case):
    m, n, k, ta, tb, batch = case
    print(f"[gemm few tiles] {case}", flush=True)
    rng = np.random.default_rng(m * 7919 + n * 31 + k)
    lead = (batch,) if batch > 1 else ()
    a = rng.standard_normal(lead + ((k, m) if ta else (m, k))).astype(np.float32)
    b = rng.standard_normal(lead + ((n, k) if tb else (k, n))).astype(np.float32)
    y = run_gemm(hip, torch_gpu, a, b, None, 1.0, 0.0, ta, tb, batch)
    A = np.swapaxes(a, -1, -2) if ta else a
    B = np.swapaxes(b, -1, -2) if tb else b
    ref = A.astype(np.float64) @ B.astype(np.float64)
    rel = np.linalg.norm(y - ref) / np.linalg.norm(ref)
    assert rel <= 2 * 2.0 ** -24 * (4 + math.sqrt(k / 8)), rel


def _quarters(x):
    """First maximal element of each quarter from its first element, later quarters replacing
    the running one only when strictly greater."""
    out = []
    for row in x:
        m = None
        for q in np.split(row, 4):
            b = q[0]
            for v in q[1:]:
                if v > b:
                    b = v
            if m is None or b > m:
                m = b
        out.append(m)
    return np.array(out, np.float32)


@pytest.mark.parametrize("block", [16, 32, 80, 240, 256])
@pytest.mark.parametrize("rows", [1, 63, 517])
def test_reduce_max_short_rows(hip, torch_gpu, rows, block):
    torch = torch_gpu
    rng = np.random.default_rng(rows * 1000 + block)
    x = rng.standard_normal((rows, block)).astype(np.float32)
    kinds = np.arange(rows) % 8
    x[kinds == 1] = -np.abs(x[kinds == 1])                              # all negative
    zero = np.where(rng.random((rows, block)) < 0.5, 0.0, -0.0).astype(np.float32)
    x[kinds == 2] = zero[kinds == 2]                                    # zeros of both signs
    x[kinds == 3] = np.minimum(x[kinds == 3], zero[kinds == 3])
    x[kinds == 4, block // 2] = np.nan
    x[kinds == 5, 0] = np.nan
    x[kinds == 6, block - 1] = np.inf
    x[kinds == 7] = -np.inf
    xd = torch.from_numpy(x).cuda()
    y = torch.full((rows,), 7.0, device="cuda")
    L = hip.lib()
    hip.check(L.spinn_hip_reduce_max(rows, block, hip.ptr(xd), hip.ptr(y), None), "reduce_max")
    torch.cuda.synchronize()
    assert _same(y.cpu().numpy(), _quarters(x))


def _same(a, b):
    """Bit for bit, NaN for NaN."""
    nan = np.isnan(a) & np.isnan(b)
    return np.array_equal(a.view(np.uint32)[~nan], b.view(np.uint32)[~nan])
