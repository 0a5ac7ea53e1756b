"""Edges of the GEMM's 128- and 256-row tiles, against the CPU oracle: rows and
columns on both sides of a tile, runs of one to five 64-deep k tiles (odd ones,
int4's 128-deep raw tiles, groups of two tiles), ragged grids over the XCDs.
Tolerances are those of test_gpu_linear.py: fp32 sums within 2e-5, outputs the
rounded sums."""
import pytest

import helpers as H
from test_gpu_linear import G, check, check_sampled  # noqa: F401  (G is a fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [H.F16, H.BF16])
@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("g", [-1, 64, 128])
def test_half_tile_edges(G, oracle, dt, bits, g):
    for M, K, N in [(65, 128, 16), (127, 256, 272), (128, 384, 256), (129, 640, 240), (257, 256, 528)]:
        if bits == 8:
            K -= 64 if K > 128 else 0  # an odd number of k tiles
        if bits == 4 and N % 32:
            N += 16
        check(G, oracle, dt, bits, g, M, K, N, bias=(M % 2 == 1), seed=M)


@pytest.mark.parametrize("dt", [H.F16, H.BF16])
@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("g", [-1, 64, 128])
def test_whole_tile_edges(G, oracle, dt, bits, g):
    # one round of 256 x 256 tiles and some half-size ones behind it; the last row tile is partial
    for M, K, N in [(2047, 256, 8224), (1793, 128 if bits == 4 else 192, 8192)]:
        check_sampled(G, oracle, dt, bits, g, M, K, N, bias=(M % 2 == 1), seed=M)


@pytest.mark.parametrize("dt", [H.F16, H.BF16])
@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("g", [-1, 64, 128])
@pytest.mark.parametrize("M,K,N", [
    (300, 2048, 272),   # more row tiles than column tiles, both ragged: runs of 8 (int8) and 16 (int4) k tiles in plain order
    (129, 2176, 784),   # fewer: two row tiles on four column tiles; a shorter last run
    (65, 2176, 1296),   # one row tile, six column tiles, no multiple of the XCDs
    (129, 8448, 272),   # runs of 33 and 34
])
def test_half_tiles_with_k_in_runs(G, oracle, dt, bits, g, M, K, N):
    from paddle_amd import _lib

    ws = _lib.lib.wol_linear_workspace(M, K, N, bits, g)
    assert ws > 0 and "128x256 tiles on [0,%d) with K in runs" % N in G.linear_plan(M, K, N, bits, g, ws)
    check(G, oracle, dt, bits, g, M, K, N, bias=(M % 2 == 1), seed=M)
