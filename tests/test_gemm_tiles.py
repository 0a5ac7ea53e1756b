"""Edges of the GEMM's 128- and 256-row tiles, against the CPU oracle: rows and
columns on both sides of a tile, from the two (int8) or four (int4) 64-deep k
tiles these kernels start at, odd numbers of them, int4's 128-deep raw tiles,
groups of two tiles, ragged grids over the XCDs, K in runs.  Every case asserts
that wol_linear_plan names the tiles it is meant for.
Tolerances are those of test_gpu_linear.py: fp32 sums within 2e-5, outputs the
rounded sums."""
import pytest

import helpers as H
from test_gpu_linear import G, check, check_sampled  # noqa: F401  (G is a fixture)

pytestmark = pytest.mark.gpu

WIDE = "wol::gemm_dma_kernel_wide (v_mfma_f32_16x16x32):"
TALL = "wol::gemm_dma_kernel_tall (v_mfma_f32_32x32x16):"


def plan(G, M, K, N, bits, g):
    from paddle_amd import _lib

    return G.linear_plan(M, K, N, bits, g, _lib.lib.wol_linear_workspace(M, K, N, bits, g))


@pytest.mark.parametrize("dt", [H.F16, H.BF16])
@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("g", [-1, 64, 128])
def test_half_tile_edges(G, oracle, dt, bits, g):
    # int8: 2, 3, 5 and 9 k tiles; int4: 4, 6 and 10
    for M, K, N in [(65, 128, 16), (127, 256, 272), (128, 384, 256), (129, 640, 240), (257, 256, 528)]:
        if bits == 8:
            K -= 64 if K > 128 else 0  # an odd number of k tiles
        else:
            K = max(K, 256)            # one raw tile alone is the general kernel's
            N += 16 if N % 32 else 0
        assert plan(G, M, K, N, bits, g).startswith(WIDE + " 128x256 tiles on [0,%d)" % N)
        check(G, oracle, dt, bits, g, M, K, N, bias=(M % 2 == 1), seed=M)


@pytest.mark.parametrize("dt", [H.F16, H.BF16])
@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("g", [-1, 64, 128])
def test_whole_tile_edges(G, oracle, dt, bits, g):
    # one round of 256 x 256 tiles and some half-size ones behind it; the last row tile is partial
    for M, K, N in [(2047, 256, 8224), (1793, 384 if bits == 4 else 192, 8192)]:
        assert plan(G, M, K, N, bits, g).startswith((WIDE if g == -1 else TALL) + " 256x256 tiles on columns [0,8192)")
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
    assert plan(G, M, K, N, bits, g).startswith(WIDE + " 128x256 tiles on [0,%d) with K in runs" % N)
    check(G, oracle, dt, bits, g, M, K, N, bias=(M % 2 == 1), seed=M)
