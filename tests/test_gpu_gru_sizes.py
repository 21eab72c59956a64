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


# widths between the largest resident layer and the largest accepted, each rest of 4
@pytest.mark.parametrize("B,T,I,H,seq", [(2, 3, 4, 262, 0), (2, 3, 4, 383, 1), (1, 3, 4, 513, 0), (2, 2, 3, 770, 1),
                                         (1, 2, 3, 1021, 0), (1, 2, 3, 1022, 1), (1, 2, 3, 1023, 0)])
def test_gru_seq_streamed(dev, oracle, B, T, I, H, seq):
    test_gru_seq_sizes(dev, oracle, B, T, I, H, seq)


@pytest.mark.parametrize("B,T,I,H,shift", [(2, 4, 3, 64, 1), (2, 4, 4, 256, 3), (2, 3, 4, 260, 2), (1, 3, 4, 320, 1)])
def test_gru_seq_buffers_at_any_float(dev, B, T, I, H, shift):
    """Buffers that start at any float, the workspace among them, give what
    buffers that start at 16 bytes give (the GEMMs around the recurrence sum in
    another order there)."""
    from goneuron_amd._lib import check, lib
    L = lib()
    log(f"gru B={B} T={T} I={I} H={H} buffers {shift} floats past their start")
    rng = np.random.default_rng(H)
    ws = C.c_int64()
    check(None, L.gn_gru_workspace(B, T, I, H, C.byref(ws)))
    p = (rng.normal(size=3 * H * I + 2 * H * H + 3 * H) * min(0.3, 1.5 / np.sqrt(H))).astype(np.float32)
    x, g = rng.normal(size=(B, T * I)).astype(np.float32), rng.normal(size=(B, H)).astype(np.float32)
    res = []
    for k in (0, shift):
        buf = [DBuf(dev, np.concatenate([np.zeros(k, np.float32), np.ravel(a)])) for a in
               (x, p, g, np.zeros((B, H), np.float32), np.zeros_like(p), np.zeros_like(x), np.zeros(ws.value, np.float32))]
        dx, dp, dg, dout, dgr, dgin, dwk = (C.c_void_p(b.p.value + 4 * k) for b in buf)
        check(dev.h, L.gn_gru_seq_forward(dev.h, dx, dp, dout, dwk, B, T, I, H, 0))
        check(dev.h, L.gn_gru_seq_backward(dev.h, dx, dp, dg, dgr, dgin, dwk, B, T, I, H, C.c_float(1.0), 0))
        res.append([b.get()[k:] for b in buf[3:6]])
    for a, b in zip(*res):
        assert np.abs(a).max() > 0 and max_rel(b, a) <= TOL
