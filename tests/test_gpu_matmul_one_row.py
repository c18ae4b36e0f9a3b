"""GPU parity of mi_mul_mat_q8_0 on one row of x, where the prologue, the product and
the key sum are one launch (up to 32 blocks of keys, or 64 on 128 or more row groups; past
256 row groups where the waves' sets of blocks are nearly full):
the oracle's bar at ragged and smallest sizes and either side of the rule, each
prologue equal to its separate op followed by the plain product, and y sharing memory
with an input (which keeps the separate launches).
"""
import numpy as np
import pytest
from helpers import assert_mul_mat_q8_0, to_dev, to_np
from oracle import oracle as orc

from acestep_ops import ops

pytestmark = pytest.mark.gpu


def _case(n, k, seed):
    r = np.random.default_rng(seed)
    w = orc.quantize_q8_0(r.standard_normal((n, k)).astype(np.float32))
    return r, w, r.standard_normal((1, k)).astype(np.float32), ops.q8_0_repack(ops.Q8(to_dev(w)))


@pytest.mark.parametrize("n,k", [(1, 32), (64, 64), (65, 288), (130, 992), (1024, 1024), (32768, 96), (32769, 96), (300, 1056),
                                 (8128, 2048), (8129, 2016), (8192, 2048), (8192, 2080),
                                 (16384, 256), (16385, 256), (16385, 768), (16385, 1056)])
def test_sizes(dev, n, k):
    print(f"mul_mat q8_0 one row n={n} k={k}", flush=True)
    r, w, x, wr = _case(n, k, n + k)
    assert_mul_mat_q8_0(to_np(ops.mul_mat_q8_0(wr, to_dev(x))), w, x)
    x[:] = 0.0
    assert not to_np(ops.mul_mat_q8_0(wr, to_dev(x))).any()


@pytest.mark.parametrize("n,k,shift", [(130, 1024, 0), (200, 96, 1), (8200, 2048, 0)])
def test_prologues(dev, n, k, shift):
    """shift 1: operands 4-byte aligned only."""
    print(f"mul_mat q8_0 one row prologues n={n} k={k} shift={shift}", flush=True)
    r, w, x, wr = _case(n, k, n + k)
    up = lambda a: to_dev(np.concatenate([np.zeros(shift, np.float32), a.ravel()]))[shift:].view(*a.shape)  # noqa: E731
    f = lambda *s: r.standard_normal(s).astype(np.float32)  # noqa: E731
    dx, b, g, nw, sc, sh = up(x), up(f(1, k)), to_dev(f(k)), to_dev(f(k)), to_dev(f(k)), to_dev(f(k))
    gu, res = up(f(1, 2 * k)), to_dev(f(1, n))
    eq = lambda y, z: np.testing.assert_array_equal(to_np(y), to_np(z))  # noqa: E731
    eq(ops.mul_mat_q8_0_rms_norm(wr, dx, nw, 1e-6), ops.mul_mat_q8_0(wr, ops.rms_norm(dx, 1e-6, w=nw)))
    eq(ops.mul_mat_q8_0_swiglu_add(wr, gu, res), ops.add(ops.mul_mat_q8_0(wr, ops.swiglu(gu)), res))
    s, y = ops.mul_mat_q8_0_add_rms_norm(wr, dx, b, nw, 1e-6)
    s2, n2 = ops.add_rms_norm(dx, b, 1e-6, w=nw)
    eq(s, s2)
    eq(y, ops.mul_mat_q8_0(wr, n2))
    s, y = ops.mul_mat_q8_0_adaln(wr, dx, nw, 1e-6, b=b, gate=g, scale=sc, shift=sh)
    s2, n2 = ops.add_rms_norm(dx, b, 1e-6, gate=g, w=nw, scale=sc, shift=sh)
    eq(s, s2)
    eq(y, ops.mul_mat_q8_0(wr, n2))


def test_y_in_place_of_x(dev):
    print("mul_mat q8_0 one row in place", flush=True)
    _, w, x, wr = _case(1024, 1024, 5)
    dx = to_dev(x)
    ops.mul_mat_q8_0(wr, dx, out=dx)
    assert_mul_mat_q8_0(to_np(dx), w, x)


@pytest.mark.parametrize("bad", [False, True])
@pytest.mark.parametrize("n,k", [(1024, 1024), (6144, 1024), (130, 992), (65, 32), (10944, 992), (12288, 2048), (8200, 1056)])
def test_same_bits_as_separate_launches(dev, n, k, bad):
    """y sharing memory with an operand keeps the separate launches: the bits of the one launch,
    for each prologue and each operand that is checked (12288 x 2048: 3 splits of 3 blocks per
    wave, the last with one block; bad: NaN and infinite elements of x)."""
    print(f"mul_mat q8_0 one row, bits n={n} k={k} bad={bad}", flush=True)
    r, _, x, wr = _case(n, k, n + k)
    f = lambda *s: r.standard_normal(s).astype(np.float32)  # noqa: E731
    b, gu, nw, sc, sh, g = f(1, k), f(1, 2 * k), f(k), f(k), f(k), f(k)
    if bad:
        x[0, [3, 17]], gu[0, [5, k + 9]] = (np.nan, np.inf), (-np.inf, np.nan)

    def over(a):
        """(a on the device, y over its first n elements)"""
        d = to_dev(np.concatenate([a.ravel(), np.zeros(max(n - a.size, 0), np.float32)]))
        return d[:a.size].view(*a.shape), d[:n].view(1, n)

    eq = lambda y, z: np.testing.assert_array_equal(to_np(y), to_np(z))  # noqa: E731
    dx, y = over(x)
    eq(ops.mul_mat_q8_0(wr, dx, out=y), ops.mul_mat_q8_0(wr, to_dev(x)))
    dg, y = over(gu)
    eq(ops.mul_mat_q8_0_swiglu(wr, dg, out=y), ops.mul_mat_q8_0_swiglu(wr, to_dev(gu)))
    ops_ = {"x": x, "b": b, "nw": nw, "sc": sc, "sh": sh, "g": g}
    call = lambda d, **kw: ops.mul_mat_q8_0_adaln(  # noqa: E731
        wr, d["x"], d["nw"], 1e-6, b=d["b"], gate=d["g"], scale=d["sc"], shift=d["sh"], **kw)
    s0, y0 = call({q: to_dev(v) for q, v in ops_.items()})
    for name in ops_:
        d = {q: to_dev(v) for q, v in ops_.items() if q != name}
        d[name], y = over(ops_[name])
        s1, y1 = call(d, out=y)
        eq(s1, s0)
        eq(y1, y0)
    sm, y = over(np.zeros_like(x))  # y over the sum: the product comes last
    eq(call({q: to_dev(v) for q, v in ops_.items()}, out=y, out_sum=sm)[1], y0)


@pytest.mark.parametrize("over", ["norm", "shift"])
def test_sum_over_a_vector(dev, over):
    """The residual sum written over the norm weight or the modulate's shift, which every row's
    norm reads after it: the bits of the sum first, then the product with the sum in their place."""
    print(f"mul_mat q8_0 one row, sum over {over}", flush=True)
    n, k = 6144, 1024
    r, _, x, wr = _case(n, k, 11)
    f = lambda *s: r.standard_normal(s).astype(np.float32)  # noqa: E731
    dx, b, nw, sc, sh = to_dev(x), to_dev(f(1, k)), to_dev(f(k)), to_dev(f(k)), to_dev(f(k))
    s0 = ops.add(dx, b)
    nw2, sh2 = (s0.view(k), sh) if over == "norm" else (nw, s0.view(k))
    ref = ops.mul_mat_q8_0(wr, ops.add_rms_norm(dx, b, 1e-6, w=nw2, scale=sc, shift=sh2)[1])
    s, y = ops.mul_mat_q8_0_adaln(wr, dx, nw, 1e-6, b=b, scale=sc, shift=sh, out_sum=(nw if over == "norm" else sh).view(1, k))
    np.testing.assert_array_equal(to_np(s), to_np(s0))
    np.testing.assert_array_equal(to_np(y), to_np(ref))
