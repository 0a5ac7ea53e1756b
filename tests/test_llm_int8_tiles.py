"""Edges of llm_int8_linear's 128- and 256-row tiles, bit for bit against the CPU
oracle: rows and columns on both sides of a tile, one to four 128-deep k tiles,
ragged grids over the XCDs; sums that merge to zeros of either sign and to
infinities, whose division by 127 takes the special cases.  K in runs above 128
rows.  And the activation stages of a few rows, on both sides of the one-launch
form's limit."""
import numpy as np
import pytest

import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [H.F16, H.BF16])
@pytest.mark.parametrize("outliers", [0, 2])
@pytest.mark.parametrize("M,K,N", [(129, 128, 16), (255, 256, 272), (257, 384, 2064), (385, 512, 256), (2049, 128, 4112)])
def test_tile_edges(device, oracle, dt, outliers, M, K, N):
    import gpu_calls as G

    rng = np.random.default_rng(M + N)
    w = rng.integers(-127, 128, (N, K), dtype=np.int8)
    ws = (rng.random(N, dtype=np.float32) * np.float32(1e-3) + np.float32(1e-4)).astype(np.float32)
    w[::7] = 0
    ws[1::9] = -ws[1::9]        # zeros and results of the other sign
    ws[3::11] = np.float32(1e-44)  # a denormal: products that vanish in T
    if not outliers:
        # and results that overflow.  (Not with outlier columns: their products of two T values are exact in fp32, so
        # that fused and separate multiply-adds agree, up to where a product overflows and its fused sum does not.)
        ws[5::13] = np.float32(3e38)
    x = np.clip(rng.standard_normal((M, K), dtype=np.float32), -5, 5)
    if outliers:
        x[rng.integers(0, M, outliers), rng.permutation(K)[:outliers]] = 30.0
    xb = H.f32_to_bits(x, dt)
    bb = H.make_bias(N, dt, seed=3, std=1.0) if M % 2 else None
    rows = np.r_[0:min(M, 40), max(0, M - 40):M] if M > 1000 else np.arange(M)
    rows = np.unique(np.r_[rows, np.nonzero((np.abs(x) > 6).any(1))[0]])  # the outlier columns depend on these
    got = G.llm_int8_linear(xb, w, bb, ws, 6.0, dt)
    want = oracle.llm_int8_linear(xb[rows], w, bb, ws, 6.0, dt)["out"]
    g = got[rows]
    nan = np.isnan(H.bits_to_f32(want, dt))
    assert np.array_equal(np.isnan(H.bits_to_f32(g, dt)), nan)
    assert np.array_equal(g[~nan], want[~nan])


@pytest.mark.parametrize("dt", [H.F16, H.BF16])
@pytest.mark.parametrize("outliers", [0, 3, 40])
@pytest.mark.parametrize("M,K,N,runs", [
    (257, 1664, 528, 3),    # 13 k tiles in runs of 5: the last has 3; three row and three column tiles
    (385, 2176, 272, 4),    # 17 in runs of 5: the last has 2
    (129, 2688, 784, 5),    # 21 in runs of 5: the last has one
    (300, 3968, 1040, 7),   # 31 in runs of 5; five column tiles, no multiple of the XCDs with three row tiles
    (140, 8192, 272, 8),    # equal runs
])
def test_k_in_runs_above_128_rows(device, oracle, dt, outliers, M, K, N, runs):
    import gpu_calls as G

    rng = np.random.default_rng(M + K)
    w = rng.integers(-127, 128, (N, K), dtype=np.int8)
    ws = (rng.random(N, dtype=np.float32) * np.float32(1e-3) + np.float32(1e-4)).astype(np.float32)
    ws[1::9] = -ws[1::9]
    x = np.clip(rng.standard_normal((M, K), dtype=np.float32), -5, 5)
    cols = np.r_[[0, K - 1, 639], 640 + rng.permutation(K - 641)][:outliers]  # ends of K, the end of a run of 5 tiles, behind it
    x[rng.integers(0, M, cols.size), cols] = 20.0
    xb = H.f32_to_bits(x, dt)
    bb = H.make_bias(N, dt, seed=3, std=1.0) if M % 2 else None
    o = oracle.llm_int8_linear(xb, w, bb, ws, 6.0, dt)
    assert o["outlier"].sum() == outliers
    got, st = G.llm_int8_linear(xb, w, bb, ws, 6.0, dt, stages=True)
    assert st["runs"] == runs
    assert np.array_equal(got, o["out"])


@pytest.mark.parametrize("dt", [H.F16, H.BF16])
@pytest.mark.parametrize("M", [1, 2, 7, 8, 9])
@pytest.mark.parametrize("K", [64, 2112, 8256, 28736])  # one, more than one and more than four rounds of the mask's 64
                                                       # words; past the K up to which eight rows take the one launch
def test_few_rows(device, oracle, dt, M, K):
    import gpu_calls as G

    rng = np.random.default_rng(M * K)
    N = 48
    w = rng.integers(-127, 128, (N, K), dtype=np.int8)
    ws = (rng.random(N, dtype=np.float32) * np.float32(1e-3) + np.float32(1e-4)).astype(np.float32)
    x = np.clip(rng.standard_normal((M, K), dtype=np.float32), -5, 5)
    cols = np.unique(np.r_[0, K - 1, rng.integers(0, K, 5)])
    x[rng.integers(0, M, cols.size), cols] = 20.0
    x[M - 1, 3], x[0, 5] = np.nan, -0.0
    xb = H.f32_to_bits(x, dt)
    o = oracle.llm_int8_linear(xb, w, None, ws, 6.0, dt)
    got, st = G.llm_int8_linear(xb, w, None, ws, 6.0, dt, stages=True)
    assert np.array_equal(st["list"], np.nonzero(o["outlier"])[0]) and st["count"] == cols.size
    assert np.array_equal(st["outlier"], o["outlier"])
    assert np.array_equal(st["ranges"], o["ranges"])
    assert np.array_equal(st["qx"], o["qx"])
    assert np.array_equal(got, o["out"])
