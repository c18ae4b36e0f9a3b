"""GPU parity of the two matrix kernels of mi_mul_mat_q8_0 (more than 8 rows of x)
where the tile choice and the tiles' edges lie: the 64 x 64 kernel (4 key groups per
workgroup, stages of 4 blocks) at one row, one column and one block either side of
its tiles, groups and stages, with and without partials in the workspace, and the
128 x 128 kernel on grids past the rule.

The bar is the product's own, (K / 32 + 8) * 2^-24 * sum |w| |x'|: each order of
adding rounds once per block and once per added group or split (at most 3 + 3).
"""
import numpy as np
import pytest
from helpers import assert_mul_mat_q8_0, to_dev, to_np
from oracle import oracle as orc

from acestep_ops import ops

pytestmark = pytest.mark.gpu


def _case(n, k, m, seed):
    r = np.random.default_rng(seed)
    w = orc.quantize_q8_0(r.standard_normal((n, k)).astype(np.float32))
    x = r.standard_normal((m, k)).astype(np.float32)
    return r, w, x, ops.q8_0_repack(ops.Q8(to_dev(w)))


@pytest.mark.parametrize("k", [32, 96, 128, 160, 416, 544, 2048])  # 1, 3, 4, 5, 13, 17 and 64 blocks
@pytest.mark.parametrize("n,m", [(64, 9), (1, 64), (65, 65), (63, 33), (130, 100), (256, 129)])
def test_small_tile_edges(dev, n, k, m):
    print(f"mul_mat q8_0 64-tile n={n} k={k} m={m}", flush=True)
    _, w, x, wr = _case(n, k, m, n + k + m)
    assert_mul_mat_q8_0(to_np(ops.mul_mat_q8_0(wr, to_dev(x))), w, x)


@pytest.mark.parametrize("n,k,m", [(512, 6144, 70), (2048, 6144, 200), (2048, 2080, 20)])
def test_small_tile_key_splits(dev, n, k, m):
    """Partials of 4, 2 and 2 key splits on top of the key groups (2080: a ragged last stage)."""
    print(f"mul_mat q8_0 64-tile splits n={n} k={k} m={m}", flush=True)
    _, w, x, wr = _case(n, k, m, n + k + m)
    y = to_np(ops.mul_mat_q8_0(wr, to_dev(x)))
    assert_mul_mat_q8_0(y, w, x)
    assert np.array_equal(y, to_np(ops.mul_mat_q8_0(wr, to_dev(x))))  # the same bits on every call


@pytest.mark.parametrize("n,k,m", [(12288, 64, 700), (8200, 160, 1100), (2560, 3072, 1024), (2560, 6144, 1217), (2100, 96, 1000)])
def test_large_tile(dev, n, k, m):
    """Grids past the 64 x 64 tiles' share, with 3 and 2 key splits and with short keys."""
    print(f"mul_mat q8_0 128-tile n={n} k={k} m={m}", flush=True)
    _, w, x, wr = _case(n, k, m, n + k + m)
    assert_mul_mat_q8_0(to_np(ops.mul_mat_q8_0(wr, to_dev(x))), w, x)


@pytest.mark.parametrize("n,m", [(130, 70), (2048, 40), (64, 64)])
def test_small_tile_residual(dev, n, m):
    """The gated and the clamped residual in the epilogue, y in place of r: the bits of the separate ops."""
    k = 256
    print(f"mul_mat q8_0 64-tile residual n={n} m={m}", flush=True)
    r, w, _, wr = _case(n, k, m, n + m)
    gu = to_dev(r.standard_normal((m, 2 * k)).astype(np.float32))
    res = r.standard_normal((m, n)).astype(np.float32)
    gate = to_dev(r.standard_normal(n).astype(np.float32))
    p = ops.mul_mat_q8_0_swiglu(wr, gu)
    y = to_dev(res)
    ops.mul_mat_q8_0_swiglu_gated_add(wr, gu, y, gate, out=y)
    assert np.array_equal(to_np(y), to_np(ops.gated_add(to_dev(res), p, gate)))
    z = to_np(ops.mul_mat_q8_0_swiglu_add(wr, gu, to_dev(res), clamp=(-2.0, 2.0)))
    assert np.array_equal(z, to_np(ops.add_clamp(to_dev(res), p, -2.0, 2.0)))
