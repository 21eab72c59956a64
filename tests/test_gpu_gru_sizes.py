"""SequenceUnroller(GRU) operators at the edges of their thread layouts, against
the oracle: one column group, sizes that are no multiple of 4, the largest
layer whose weights stay on the CU (256), the first ones that stream (257 and
260), and the largest accepted (1024).  Tolerance: the per-tensor 1e-4 of the
reference's largest magnitude that every operator is held to (float32 sums in
another order; float64 activations rounded to float32 on both sides)."""
import ctypes as C

import numpy as np
import pytest

from cfgutil import max_rel
from gpuutil import DBuf, TOL, log

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T,I,H,seq", [
    (3, 4, 2, 1, 0), (2, 5, 3, 7, 1), (3, 6, 5, 64, 0), (2, 5, 4, 66, 1), (2, 4, 4, 130, 0), (2, 4, 3, 200, 1),
    (2, 4, 4, 252, 0), (2, 4, 6, 256, 1), (2, 3, 4, 257, 1), (2, 3, 4, 260, 0), (1, 2, 3, 1024, 0)])
def test_gru_seq_sizes(dev, oracle, B, T, I, H, seq):
    from goneuron_amd._lib import check, lib
    L = lib()
    log(f"gru B={B} T={T} I={I} H={H} seq={seq}")
    net = oracle.Net([oracle.spec(oracle.LAYER_GRU_UNROLLER, in_size=I, out_size=H, seq_len=T,
                                  return_sequences=seq)], oracle.LOSS_MSE)
    rng = np.random.default_rng(H * 10 + T)
    p = (rng.normal(size=net.n) * min(0.3, 1.5 / np.sqrt(H))).astype(np.float32)
    net.params[:] = p
    x = rng.normal(size=(B, T * I)).astype(np.float32)
    OL = T * H if seq else H
    g = rng.normal(size=(B, OL)).astype(np.float32)
    out_r, gin_r = net.accumulate_grad(x, g, B, T * I, OL)
    gr = net.grads.copy()
    ws = C.c_int64()
    check(None, L.gn_gru_workspace(B, T, I, H, C.byref(ws)))
    dx, dp, dg = DBuf(dev, x), DBuf(dev, p), DBuf(dev, g)
    dout, dgr, dgin, dwk = (DBuf(dev, np.zeros(s, np.float32)) for s in ((B, OL), p.shape, (B, T * I), ws.value))
    check(dev.h, L.gn_gru_seq_forward(dev.h, dx.p, dp.p, dout.p, dwk.p, B, T, I, H, seq))
    check(dev.h, L.gn_gru_seq_backward(dev.h, dx.p, dp.p, dg.p, dgr.p, dgin.p, dwk.p, B, T, I, H,
                                       C.c_float(np.float32(1) / np.float32(B)), seq))
    assert max_rel(dout.get(), out_r) <= TOL
    assert max_rel(dgin.get(), gin_r) <= TOL
    got = dgr.get()
    nwx, nwh = 3 * H * I, 2 * H * H
    for name, sl in (("Wx", slice(0, nwx)), ("Wh_u", slice(nwx, nwx + H * H)),
                     ("Wh_r", slice(nwx + H * H, nwx + nwh)), ("b", slice(nwx + nwh, None))):
        assert max_rel(got[sl], gr[sl]) <= TOL, name
