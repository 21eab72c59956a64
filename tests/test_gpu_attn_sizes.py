"""Attention beyond the LDS-resident kernels (T > 128 or heads wider than 32), at
the edges of its tiles and of its dispatch, against the oracle: head widths at
and beside each padded width, sequences around the 16-row tiles, the 32/64-row
stages and the 64-row workgroups, few (sample, head) pairs (16-row workgroups)
and many.  Tolerance: the per-tensor 1e-4 of the reference's largest magnitude
that every operator is held to."""
import ctypes as C

import numpy as np
import pytest

from cfgutil import max_rel
from gpuutil import DBuf, TOL, log

pytestmark = pytest.mark.gpu


def _mha(dev, B, T, D, NH, causal, p, x, g, shift=0):
    """shift: the workspace starts that many floats past its aligned start."""
    from goneuron_amd._lib import check, lib
    L = lib()
    ws = C.c_int64()
    check(None, L.gn_mha_workspace(B, T, D, NH, 0, C.byref(ws)))
    dx, dp, dg = DBuf(dev, x), DBuf(dev, p), DBuf(dev, g)
    dout, dgr, dgin, dwk = (DBuf(dev, np.full(s, np.nan, np.float32))
                            for s in ((B, T * D), p.shape, (B, T * D), ws.value + shift))
    whole, dwk.p = dwk.p, C.c_void_p(dwk.p.value + 4 * shift)
    check(dev.h, L.gn_mha_forward(dev.h, dx.p, dp.p, dout.p, dwk.p, B, T, D, NH, causal, 0))
    check(dev.h, L.gn_mha_backward(dev.h, dx.p, dp.p, dg.p, dgr.p, dgin.p, dwk.p, B, T, D, NH, causal, 0,
                                   C.c_float(np.float32(1) / np.float32(B))))
    dwk.p = whole
    return dout.get(), dgr.get(), dgin.get()


@pytest.mark.parametrize("B,T,D,NH,causal", [
    (1, 129, 8, 2, 1), (2, 130, 15, 3, 0), (1, 191, 33, 1, 1), (2, 33, 48, 1, 0), (1, 65, 98, 2, 1),
    (1, 64, 64, 1, 1), (2, 48, 63, 1, 0), (1, 193, 64, 1, 1), (1, 63, 80, 1, 0), (2, 31, 81, 1, 1),
    (1, 97, 96, 1, 1), (1, 66, 128, 1, 0), (1, 17, 125, 1, 1), (1, 16, 130, 1, 0), (4, 1, 64, 1, 1),
    (90, 65, 66, 2, 1), (140, 40, 128, 2, 0)])
def test_attn_sizes(dev, oracle, B, T, D, NH, causal):
    log(f"attention B={B} T={T} D={D} heads={NH} causal={causal}")
    nd = min(B, 2)  # distinct samples; a larger batch repeats them
    assert B % nd == 0
    net = oracle.Net([oracle.spec(oracle.LAYER_MHA, dim=D, num_heads=NH, seq_len=T, causal=causal, use_rope=0)],
                     oracle.LOSS_MSE)
    rng = np.random.default_rng(T * D + NH)
    p = (rng.normal(size=net.n) * (1.0 / np.sqrt(D))).astype(np.float32)
    net.params[:] = p
    x = rng.normal(size=(nd, T * D)).astype(np.float32)
    g = rng.normal(size=(nd, T * D)).astype(np.float32)
    out_r, gin_r = net.accumulate_grad(x, g, nd, T * D, T * D)
    gr = net.grads.copy()
    out, got, gin = _mha(dev, B, T, D, NH, causal, p, np.tile(x, (B // nd, 1)), np.tile(g, (B // nd, 1)))
    for r in (0, B // nd - 1):
        assert max_rel(out[r * nd:(r + 1) * nd], out_r) <= TOL
        assert max_rel(gin[r * nd:(r + 1) * nd], gin_r) <= TOL
    n1 = D * D + D
    scale = np.abs(gr).max()
    for i, name in enumerate(("wQ", "wK", "wV", "wOut")):
        ref = gr[i * n1:(i + 1) * n1]
        if np.abs(ref).max() <= 1e-6 * scale:  # sums that vanish (wK; wQ and wK at T = 1)
            assert np.abs(got[i * n1:(i + 1) * n1]).max() <= 1e-5 * scale, name
            continue
        assert max_rel(got[i * n1:i * n1 + D * D], ref[:D * D]) <= TOL, name


# heads of a multiple of four columns below the padded width (16-byte accesses),
# heads beyond 64 with 16-row workgroups (fewer than 256 of 64 rows) and 64-row ones
@pytest.mark.parametrize("B,T,D,NH,causal", [
    (1, 97, 24, 1, 1), (2, 70, 80, 2, 0), (1, 130, 100, 1, 0), (2, 65, 120, 1, 1), (130, 65, 48, 2, 1),
    (1, 193, 128, 1, 1), (1, 129, 80, 1, 0), (2, 64, 192, 2, 1), (1, 49, 68, 1, 0), (64, 66, 256, 2, 1),
    (64, 65, 168, 2, 0), (130, 40, 96, 1, 1), (1, 131, 4, 1, 1)])
def test_attn_head_widths(dev, oracle, B, T, D, NH, causal):
    test_attn_sizes(dev, oracle, B, T, D, NH, causal)


def test_attn_single_key_rows_have_no_score_gradient(dev):
    """Under the causal mask token 0 attends to itself alone: its probability is
    1 and gradScore an exact zero, so with a gradient on token 0 only the query
    and key projections get exactly none (Adam would turn rounding noise there
    into whole steps)."""
    for T, D, NH in ((150, 64, 2), (40, 96, 1), (200, 128, 1), (70, 80, 2)):
        rng = np.random.default_rng(T)
        p = (rng.normal(size=4 * (D * D + D)) / np.sqrt(D)).astype(np.float32)
        x = rng.normal(size=(3, T * D)).astype(np.float32)
        g = np.zeros((3, T * D), np.float32)
        g[:, :D] = rng.normal(size=(3, D))
        _, got, _ = _mha(dev, 3, T, D, NH, 1, p, x, g)
        assert not got[:2 * (D * D + D)].any(), (T, D, NH)
        assert got[2 * (D * D + D):].any()


def test_attn_infinite_last_row(dev):
    """Positions past the end weigh nothing: an infinite value (or output
    gradient) of the last token gives infinities, not NaN, in what it reaches."""
    for T, D, NH in ((130, 64, 2), (33, 48, 1), (100, 128, 1), (70, 80, 2), (131, 24, 3)):
        log(f"attention with an infinite last row T={T} D={D} heads={NH}")
        rng = np.random.default_rng(T)
        w = [np.zeros((D + 1, D), np.float32) for _ in range(4)]
        w[0][:D], w[1][:D] = (rng.normal(size=(D, D)) * 1e-31 for _ in range(2))
        w[2][:D] = 1e10  # V and gO of a token of 1e30 overflow, its Q and K do not
        w[3][:D] = 1e10
        p = np.concatenate([m.ravel() for m in w])
        x = np.abs(rng.normal(size=(2, T, D))).astype(np.float32) * 1e-12
        g = x.copy()
        x[:, -1], g[:, -1] = 1e30, 1e30
        out, gr, _ = _mha(dev, 2, T, D, NH, 0, p, x.reshape(2, T * D), g.reshape(2, T * D))
        assert np.all(out == np.inf), (T, D)
        assert np.all(gr[3 * (D * D + D) - D:3 * (D * D + D)] == np.inf), (T, D)  # V's bias gradient


@pytest.mark.parametrize("T,D,NH,causal", [(486, 48, 3, 0), (112, 128, 1, 1), (38, 64, 1, 1), (300, 128, 2, 1), (197, 192, 3, 0)])
def test_attn_vanishing_sums(dev, T, D, NH, causal):
    """Without rotary embedding the key projection's bias gradient vanishes:
    every row of gradScore sums to zero.  What is left is the rounding of P, dP
    and their row sums, which must not exceed that of float32 arithmetic in the
    reference's order of operations (float64 exponential, d = sum P dP): here
    numpy's, with half as much again allowed for one draw of 4 samples."""
    B, hd = 4, D // NH
    log(f"attention vanishing sums T={T} D={D} heads={NH} causal={causal}")
    rng = np.random.default_rng(T + D)
    p = (rng.normal(size=4 * (D * D + D)) / np.sqrt(D)).astype(np.float32)
    x, g = (rng.normal(size=(B, T, D)).astype(np.float32) for _ in range(2))
    _, got, _ = _mha(dev, B, T, D, NH, causal, p, x.reshape(B, -1), g.reshape(B, -1))
    n1 = D * D + D
    w = [(p[i * n1:i * n1 + D * D].reshape(D, D), p[i * n1 + D * D:(i + 1) * n1]) for i in range(4)]
    q, k, v = (x @ w[i][0].T + w[i][1] for i in range(3))
    go = g @ w[3][0]
    left = np.zeros(D, np.float32)
    mask = np.triu(np.ones((T, T), bool), 1) if causal else np.zeros((T, T), bool)
    for b in range(B):
        for h in range(NH):
            qh, kh, vh, gh = (z[b, :, h * hd:(h + 1) * hd] for z in (q, k, v, go))
            s = np.where(mask, np.float32(-1e9), qh @ kh.T / np.float32(np.sqrt(hd)))
            e = np.exp((s - s.max(1, keepdims=True)).astype(np.float64)).astype(np.float32)
            pr = e / e.sum(1, keepdims=True)
            dp = gh @ vh.T
            ds = np.where(mask, np.float32(0), pr * (dp - (pr * dp).sum(1, keepdims=True))) / np.float32(np.sqrt(hd))
            left[h * hd:(h + 1) * hd] += (ds.T @ qh).sum(0)
    assert q.dtype == ds.dtype == np.float32
    a, r = np.linalg.norm(got[n1 + D * D:2 * n1]), np.linalg.norm(left / B)
    log(f"  left over: {a:.3e}, numpy {r:.3e}")
    assert a <= 1.5 * r


@pytest.mark.parametrize("T,D,NH", [(150, 64, 2), (70, 96, 1), (200, 24, 1), (40, 128, 1), (530, 16, 1)])
@pytest.mark.parametrize("rows", [1, 300])
def test_attn_masked_keys_with_weight(dev, oracle, T, D, NH, rows):
    """A masked key scores -1e9, which weighs nothing beside ordinary scores.
    Rows whose own keys all score lower (here by q_0 = 1e6, k_0 = -1e6 in each
    head) divide their weight among the masked keys, in every tile, and their
    value gradient too.  Column 0 of each head's query gradient is left out, and
    with it the input gradient of the column that sets it: rounding times 1e6."""
    B, hd = 150 if rows > 1 else 1, D // NH  # few and many workgroups
    log(f"attention masked weights T={T} D={D} heads={NH} B={B}")
    rng = np.random.default_rng(T + D)
    n1 = D * D + D
    w = [rng.normal(size=n1).astype(np.float32) / np.float32(np.sqrt(D)) for _ in range(4)]
    for i in range(2):
        W, b = w[i][:D * D].reshape(D, D), w[i][D * D:]
        W[:, 0] = 0
        W[::hd] = 0
        b[::hd] = 0 if i == 0 else -1e6
        if i == 0:
            W[::hd, 0] = 1e6
    p = np.concatenate(w)
    x, g = (rng.normal(size=(1, T, D)).astype(np.float32) for _ in range(2))
    x[:, :, 0] = 0
    x[:, [0, 3, T // 2, T - 2], 0] = 1
    net = oracle.Net([oracle.spec(oracle.LAYER_MHA, dim=D, num_heads=NH, seq_len=T, causal=1, use_rope=0)],
                     oracle.LOSS_MSE)
    net.params[:] = p
    out_r, gin_r = net.accumulate_grad(x.reshape(1, -1), g.reshape(1, -1), 1, T * D, T * D)
    gr = net.grads.copy()
    out, got, gin = _mha(dev, B, T, D, NH, 1, p, np.tile(x.reshape(1, -1), (B, 1)), np.tile(g.reshape(1, -1), (B, 1)))
    keep = np.ones(D, bool)
    keep[0] = False
    for r in (0, B - 1):
        assert max_rel(out[r], out_r[0]) <= TOL
        assert max_rel(gin[r].reshape(T, D)[:, keep], gin_r.reshape(T, D)[:, keep]) <= TOL
    rows_ = np.arange(D) % hd != 0
    for i, name in ((0, "wQ"), (2, "wV"), (3, "wOut")):
        a, b = (z[i * n1:i * n1 + D * D].reshape(D, D) for z in (got, gr))
        k = rows_ if i == 0 else slice(None)
        assert max_rel(a[k], b[k]) <= TOL, name


@pytest.mark.parametrize("T,D,NH,causal,shift", [(150, 64, 2, 1, 1), (70, 96, 1, 0, 3), (200, 24, 1, 1, 2), (33, 48, 1, 0, 1)])
def test_attn_workspace_at_any_float(dev, T, D, NH, causal, shift):
    """A workspace that starts at any float gives what an aligned one gives (the
    GEMMs around the attention sum in another order there)."""
    log(f"attention T={T} D={D} heads={NH} workspace {shift} floats past its start")
    rng = np.random.default_rng(T)
    p = (rng.normal(size=4 * (D * D + D)) / np.sqrt(D)).astype(np.float32)
    x, g = (rng.normal(size=(2, T * D)).astype(np.float32) for _ in range(2))
    a, b = _mha(dev, 2, T, D, NH, causal, p, x, g), _mha(dev, 2, T, D, NH, causal, p, x, g, shift)
    for u, v in zip(a, b):
        assert np.isfinite(v).all() and max_rel(v, u) <= TOL
