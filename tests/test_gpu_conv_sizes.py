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


def _conv64(x, w, b, k, s, p):
    """Float64, with the reference's k3 s1 p1 rule: the first and last columns of
    interior rows hold the bias alone."""
    B, C, H, W = x.shape
    oH, oW = (H + 2 * p - k) // s + 1, (W + 2 * p - k) // s + 1
    xp = np.pad(x.astype(np.float64), ((0, 0), (0, 0), (p, p), (p, p)))
    z = np.zeros((B, w.shape[0], oH, oW))
    for i in range(k):
        for j in range(k):
            z += np.einsum("bchw,oc->bohw", xp[:, :, i:i + s * oH:s, j:j + s * oW:s][:, :, :oH, :oW], w[:, :, i, j].astype(np.float64))
    if (k, s, p) == (3, 1, 1):
        z[:, :, 1:oH - 1, 0] = 0
        z[:, :, 1:oH - 1, oW - 1] = 0
    return z + b[:, None, None]


# planes higher than wide and wider than high; more than 65535 (sample, channel)
# planes, which still are at most 65535 groups of eight, and more than that
@pytest.mark.parametrize("B,inC,H,W,outC,k,s,p", [
    (2, 5, 7, 19, 4, 3, 1, 1), (2, 6, 21, 3, 9, 3, 1, 1), (1, 7, 1, 40, 5, 3, 1, 1), (1, 7, 40, 1, 5, 3, 1, 1),
    (2, 5, 9, 30, 7, 3, 2, 1), (2, 5, 30, 9, 8, 5, 1, 2), (2, 8, 17, 6, 12, 1, 1, 0), (1, 5, 6, 33, 6, 1, 2, 0),
    (130, 5, 33, 12, 12, 3, 1, 1), (1100, 5, 4, 3, 64, 3, 1, 1), (9000, 1, 2, 3, 59, 1, 1, 0)])
def test_conv_forward_planes(dev, B, inC, H, W, outC, k, s, p):
    from goneuron_amd._lib import check, lib
    L = lib()
    log(f"conv2d forward B={B} inC={inC} {H}x{W} outC={outC} k={k} s={s} p={p}")
    rng = np.random.default_rng(B + H * 7 + W)
    x = rng.normal(size=(B, inC, H, W)).astype(np.float32)
    w, b = (rng.normal(size=(outC, inC, k, k)) * 0.2).astype(np.float32), rng.normal(size=outC).astype(np.float32)
    want = _conv64(x, w, b, k, s, p)
    dx, dp = DBuf(dev, x), DBuf(dev, np.concatenate([w.ravel(), b]))
    dout = DBuf(dev, np.full(want.shape, np.nan, np.float32))
    check(dev.h, L.gn_conv2d_forward(dev.h, dx.p, dp.p, dout.p, B, inC, H, W, outC, k, s, p, 6))
    assert np.abs(dout.get() - want).max() <= TOL * np.abs(want).max()


@pytest.mark.parametrize("B,inC,outC", [(6000, 32, 8), (1500, 57, 4), (70, 64, 16)])
def test_conv_weight_gradient_block_sums(dev, B, inC, outC):
    """The blocks' partials of many slots: one block per sample here, whose
    partial is one exact product (a single output gradient, inputs that are
    powers of two), so what is left is the rounding of their sum.  It must not
    exceed that of a wave per slot (64 chains, then a tree), restated in numpy;
    a tenth is allowed for the draw."""
    from goneuron_amd._lib import check, lib
    L = lib()
    log(f"conv2d weight gradient B={B} {inC} -> {outC} channels of 3x3")
    rng = np.random.default_rng(B)
    x = np.broadcast_to(np.exp2(rng.integers(-1, 2, size=(B, inC, 1, 1))), (B, inC, 3, 3)).astype(np.float32)
    g = np.zeros((B, outC, 3, 3), np.float32)
    g[:, :, 1, 1] = rng.uniform(1, 2, size=(B, outC))
    n = outC * inC * 9
    dx, dg = DBuf(dev, np.ascontiguousarray(x)), DBuf(dev, g)
    dp, dout, dgr = (DBuf(dev, np.zeros(k, np.float32)) for k in (n + outC, g.shape, n + outC))
    check(dev.h, L.gn_conv2d_backward(dev.h, dx.p, dp.p, dout.p, dg.p, dgr.p, None, B, inC, 3, 3, outC, 3, 1, 1, 6, 1.0))
    got = dgr.get()[:n].reshape(outC, inC, 9)
    terms = g[:, :, None, 1, 1] * x[:, None, :, 0, 0]  # exact
    ref = terms.astype(np.float64).sum(0)
    assert np.array_equal(got, np.broadcast_to(got[:, :, :1], got.shape))  # every tap meets the same products
    lanes = [np.zeros((outC, inC), np.float32) for _ in range(64)]
    for b in range(B):
        lanes[b % 64] = lanes[b % 64] + terms[b]
    while len(lanes) > 1:
        lanes = [a + b for a, b in zip(lanes[:len(lanes) // 2], lanes[len(lanes) // 2:])]
    rms = [np.sqrt(np.mean((v / ref - 1) ** 2)) for v in (got[:, :, 0], lanes[0])]
    log(f"  rounding {rms[0]:.2e}, a wave per slot {rms[1]:.2e}")
    assert rms[0] <= 1.1 * rms[1]


@pytest.mark.parametrize("B,inC,HW,outC,k,s,p", [
    (32, 5, 20, 8, 3, 1, 1), (33, 5, 20, 8, 3, 1, 1), (4, 8, 10, 12, 3, 1, 1), (4, 9, 10, 12, 3, 1, 1), (4, 2, 9, 7, 3, 2, 1)])
def test_conv_forward_tanh(dev, oracle, B, inC, HW, outC, k, s, p):
    """Both sides of the grid and window up to which tanh takes a channel per thread."""
    test_conv_forward_sizes(dev, oracle, B, inC, HW, outC, k, s, p, 3)
