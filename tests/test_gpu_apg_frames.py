"""GPU parity of mi_apg_forward where its split over channels and frames changes:
one or two channels per workgroup (odd channel counts, operands 4-byte aligned
only), frame counts either side of a workgroup's 512 threads and of the 8192 frames
held in registers, and out in place of cond. The bar is the op's own: APG runs in
double and only the order of its sums differs from the oracle's, so the float output
is within 1 ulp of the oracle's.
"""
import numpy as np
import pytest
from helpers import to_dev, to_np
from oracle import oracle as orc

from acestep_ops import sampler as smp
from acestep_ops.device import DTensor

pytestmark = pytest.mark.gpu


def _ulps(y, ref):
    return np.abs(y.astype(np.float64) - ref) / np.spacing(np.abs(ref).astype(np.float32)).astype(np.float64)


@pytest.mark.parametrize("inplace", [False, True])
@pytest.mark.parametrize("n,t,oc,shift", [(1, 1, 64, 0), (2, 511, 6, 0), (1, 513, 7, 0), (1, 8192, 4, 0), (2, 8193, 2, 0),
                                          (1, 9300, 3, 0), (1, 6000, 64, 0), (1, 700, 64, 1)])
def test_apg_frames(dev, n, t, oc, shift, inplace):
    print(f"apg n={n} t={t} oc={oc} shift={shift} inplace={inplace}", flush=True)
    r = np.random.default_rng(n + t + oc)
    ra = np.zeros((n, t, oc))
    mb = None
    for step in range(2):
        cond = r.standard_normal((n, t, oc)).astype(np.float32)
        unc = (cond - 0.3 * r.standard_normal((n, t, oc))).astype(np.float32)
        up = lambda a: to_dev(np.concatenate([np.zeros(shift, np.float32), a.ravel()]))[shift:].view(n, t, oc)  # noqa: E731
        dc, du = up(cond), up(unc)
        mb = mb if mb is not None else smp.apg_buffer(dc)
        y = smp.apg_forward(dc, du, 7.0, mb, step == 0, out=dc if inplace else None)
        y = DTensor(y.buf, (y.buf.nbytes // 4,), "f32").numpy()[-n * t * oc:].reshape(n, t, oc) if inplace else to_np(y)
        ref = orc.apg_forward(cond, unc, 7.0, ra, step == 0)
        assert np.max(_ulps(y, ref)) <= 1.0


@pytest.mark.parametrize("n,t,oc", [(1, 31, 64), (40, 17, 64), (200, 40, 7), (3, 2, 1024), (130, 300, 64), (66000, 1, 2)])
def test_apg_many_samples(dev, n, t, oc):
    """A workgroup per sample: short ones, many, one frame more than the workgroup's phases, and
    more samples than a grid's second dimension holds."""
    print(f"apg by sample n={n} t={t} oc={oc}", flush=True)
    r = np.random.default_rng(n + t + oc)
    ra = np.zeros((n, t, oc))
    mb = None
    for step in range(2):
        cond = r.standard_normal((n, t, oc)).astype(np.float32)
        unc = (cond - 0.3 * r.standard_normal((n, t, oc))).astype(np.float32)
        dc, du = to_dev(cond), to_dev(unc)
        mb = mb if mb is not None else smp.apg_buffer(dc)
        y = to_np(smp.apg_forward(dc, du, 7.0, mb, step == 0))
        assert np.max(_ulps(y, orc.apg_forward(cond, unc, 7.0, ra, step == 0))) <= 1.0


@pytest.mark.parametrize("by", [1, -1, 3])
def test_apg_out_across_uncond(dev, by):
    """out of one sample laid over uncond, frames later or earlier."""
    print(f"apg out across uncond by={by}", flush=True)
    t, oc = 1200, 64
    r = np.random.default_rng(50 + by)
    cond = r.standard_normal((1, t, oc)).astype(np.float32)
    unc = (cond - 0.3 * r.standard_normal((1, t, oc))).astype(np.float32)
    whole = np.zeros(((t + 4) * oc,), np.float32)
    at, to = (0, by) if by > 0 else (-by, 0)
    whole[at * oc:(at + t) * oc] = unc.ravel()
    d = to_dev(whole)
    dc = to_dev(cond)
    v = lambda f: d[f * oc:(f + t) * oc].view(1, t, oc)  # noqa: E731
    smp.apg_forward(dc, v(at), 7.0, smp.apg_buffer(dc), True, out=v(to))
    y = to_np(d)[to * oc:(to + t) * oc].reshape(1, t, oc)
    assert np.max(_ulps(y, orc.apg_forward(cond, unc, 7.0, np.zeros((1, t, oc)), True))) <= 1.0
