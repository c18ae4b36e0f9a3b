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


@pytest.mark.parametrize("n,k,m,splits", [(512, 6144, 70, 4), (2048, 6144, 200, 4), (2048, 2080, 20, 2), (2048, 6144, 375, 2),
                                          (2000, 6208, 300, 2), (2048, 6112, 375, 1)])
def test_small_tile_key_splits(dev, n, k, m, splits):
    """Partials on top of the key groups: grids under a quarter of the resident workgroups (2080: a
    ragged last stage), then under half with 96 blocks per split (6208: 97, a last stage of one
    block; 6112: one block too few)."""
    print(f"mul_mat q8_0 64-tile splits n={n} k={k} m={m}", flush=True)
    _, w, x, wr = _case(n, k, m, n + k + m)
    dx = to_dev(x)
    mp = (m + 127) // 128 * 128  # the workspace: quants and scales of the padded rows, then the partials
    partials = ops.mul_mat_q8_0_workspace(wr, dx) - mp * k - mp * (k // 32) * 4
    assert partials == (splits * mp * ((n + 63) // 64 * 64) * 4 if splits > 1 else 0)
    y = to_np(ops.mul_mat_q8_0(wr, dx))
    assert_mul_mat_q8_0(y, w, x)
    assert np.array_equal(y, to_np(ops.mul_mat_q8_0(wr, dx)))  # the same bits on every call


@pytest.mark.parametrize("n,k,m", [(130, 544, 70), (100, 4096, 20)])
def test_small_tile_not_finite(dev, n, k, m):
    """NaN and infinite elements of x, infinite and NaN scales of w, NaN bits left in the workspace
    (padding rows, partials): NaN and infinities where the matrix-vector kernel has them (a sum has
    them in any order), the other values within both kernels' bounds (K / 32 + 8) 2^-24 sum |w| |x'|,
    |x'| <= max |x| (1 + 2^-8) (the scale and a quant, rounded)."""
    print(f"mul_mat q8_0 64-tile not finite n={n} k={k} m={m}", flush=True)
    _, w, x, _ = _case(n, k, m, n + k)
    x[2, 40], x[9, k - 1], x[15], x[19, ::2] = np.nan, np.inf, -np.inf, np.nan
    big = np.max(np.abs(x[np.isfinite(x)]))
    w = w.copy().reshape(n, k // 32, 34)
    w[5, 2, :2], w[97, 0, :2] = np.frombuffer(np.float16([np.inf, np.nan]).tobytes(), np.uint8).reshape(2, 2)
    w = w.reshape(n, -1)
    wr = ops.q8_0_repack(ops.Q8(to_dev(w)))

    def mul(rows):
        dx = to_dev(rows)
        ws = to_dev(np.full(ops.mul_mat_q8_0_workspace(wr, dx), 0xff, np.uint8))
        return to_np(ops.mul_mat_q8_0(wr, dx, workspace=ws))

    y, ref = mul(x), np.concatenate([mul(x[i:i + 8]) for i in range(0, m, 8)])
    assert np.array_equal(np.isnan(y), np.isnan(ref)) and np.isnan(y[:, 97]).all()
    inf = np.isinf(y)
    assert np.array_equal(inf, np.isinf(ref)) and np.array_equal(y[inf], ref[inf])
    ok = np.isfinite(y)
    assert ok[np.ix_(np.r_[:2, 3:9, 10:15, 16:19], np.r_[:5, 6:97, 98:n])].all()
    sw = np.abs(orc.dequantize_q8_0(w).astype(np.float64))
    with np.errstate(invalid="ignore"):
        bound = np.broadcast_to(2 * (k / 32 + 8) * 2.0 ** -24 * sw.sum(1) * big * (1 + 2.0 ** -8), y.shape)
        assert np.all(np.abs(y.astype(np.float64) - ref)[ok] <= bound[ok])


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
