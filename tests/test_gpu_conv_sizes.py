"""Conv2D forward by groups of output channels, at the edges of its dispatch
(kernels 1, 3 and 5, strides, padding up to and beyond the kernel's half, channel
counts that fill no group, four and eight channels per thread) against the
oracle.  The forward keeps the reference's order of float32 sums, so a linear or
ReLU layer's outputs are the same bits."""

import numpy as np
import pytest

from gpuutil import DBuf, TOL, log

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,inC,HW,outC,k,s,p,act", [
    (2, 5, 7, 4, 3, 1, 1, 6), (3, 6, 16, 5, 3, 1, 1, 1), (2, 5, 17, 9, 3, 1, 1, 6), (1, 7, 3, 4, 3, 1, 1, 6),
    (2, 5, 1, 4, 3, 1, 1, 6), (2, 5, 2, 7, 3, 1, 1, 6), (2, 1, 19, 7, 3, 1, 0, 6), (2, 8, 15, 12, 3, 2, 1, 1),
    (2, 3, 9, 6, 3, 1, 2, 6), (2, 9, 13, 11, 1, 1, 0, 6), (3, 4, 12, 4, 1, 2, 0, 6), (2, 6, 11, 5, 5, 1, 2, 6),
    (2, 3, 14, 8, 5, 2, 1, 1), (1, 2, 5, 4, 5, 1, 0, 6), (2, 5, 8, 3, 3, 1, 1, 6), (130, 5, 20, 12, 3, 1, 1, 6),
    (33, 17, 33, 21, 3, 1, 1, 3)])
def test_conv_forward_sizes(dev, oracle, B, inC, HW, outC, k, s, p, act):
    from goneuron_amd._lib import check, lib
    L = lib()
    log(f"conv2d forward B={B} inC={inC} HW={HW} outC={outC} k={k} s={s} p={p} act={act}")
    n_in, o = inC * HW * HW, (HW + 2 * p - k) // s + 1
    n_out = outC * o * o
    net = oracle.Net([oracle.spec(oracle.LAYER_CONV2D, in_size=n_in, in_channels=inC, out_channels=outC,
                                  kernel=k, stride=s, padding=p, act=act)], oracle.LOSS_MSE)
    rng = np.random.default_rng(B * 7 + HW * 3 + outC)
    params = (rng.normal(size=net.n) * 0.2).astype(np.float32)
    net.params[:] = params
    nd = min(B, 3)
    x = rng.normal(size=(nd, n_in)).astype(np.float32)
    want, _ = net.accumulate_grad(x, np.zeros((nd, n_out), np.float32), nd, n_in, n_out)
    want = want.reshape(nd, n_out)
    rows = np.arange(B) % nd
    dx, dp, dout = DBuf(dev, x[rows]), DBuf(dev, params), DBuf(dev, np.full((B, n_out), np.nan, np.float32))
    check(dev.h, L.gn_conv2d_forward(dev.h, dx.p, dp.p, dout.p, B, inC, HW, HW, outC, k, s, p, act))
    if act in (1, 6):
        np.testing.assert_array_equal(dout.get(), want[rows])
    else:
        assert np.abs(dout.get() - want[rows]).max() <= TOL * np.abs(want).max()
