"""LayerNorm and RMSNorm rows held in registers, at the edges of their dispatch
(columns per lane 4 / 8 / 16 / 32, 16-byte or 4-byte accesses by row length and
by pointer, the forward's 512, the longest row of 2048 and the first beyond it)
and of the backward's grid (one row, one wave's remainder, more rows than the
grid walks at once), against float64 in numpy.  Tolerance: the per-tensor 1e-4
of the reference's largest magnitude that every operator is held to."""
import ctypes as C

import numpy as np
import pytest

from gpuutil import DBuf, TOL, log

pytestmark = pytest.mark.gpu


def _ref(kind, x, gam, bet, g, scale, eps):
    x, gam, bet, g = (a.astype(np.float64) for a in (x, gam, bet, g))
    n = x.shape[1]
    if kind == "ln":
        mean = x.mean(1, keepdims=True)
        std = np.sqrt(x.var(1, keepdims=True) + eps)
        d, gp = x - mean, g * gam
        dx = (gp - gp.sum(1, keepdims=True) / n) / std - d * (gp * d).sum(1, keepdims=True) / (n * std * std)
        return gam * d / std + bet, dx, scale * (g * d / std).sum(0), scale * g.sum(0)
    rms = np.sqrt((x * x).mean(1, keepdims=True) + eps)
    dx = gam / rms * (g - x * (g * gam * x).sum(1, keepdims=True) / (n * rms * rms))
    return x / rms * gam, dx, scale * (g * x / rms).sum(0), None


@pytest.mark.parametrize("kind", ["ln", "rms"])
@pytest.mark.parametrize("rows,N,shift", [
    (1, 1, 0), (1, 256, 0), (7, 257, 0), (9, 511, 0), (8, 512, 0), (17, 513, 0), (65, 516, 0), (33, 1024, 0),
    (33, 1024, 1), (12, 1025, 0), (40, 2044, 0), (5, 2047, 0), (9, 2048, 0), (4, 2049, 0), (4099, 36, 0),
    (4097, 33, 0), (6000, 520, 0)])
def test_norm_sizes(dev, kind, rows, N, shift):
    """shift: every buffer starts that many floats past its aligned start."""
    from goneuron_amd._lib import check, lib
    L = lib()
    log(f"{kind} rows={rows} N={N} shift={shift}")
    rng = np.random.default_rng(rows * 4099 + N)
    x = (rng.normal(size=(rows, N)) * 1.5 + 0.3).astype(np.float32)
    g = rng.normal(size=(rows, N)).astype(np.float32)
    gam = (1 + 0.3 * rng.normal(size=N)).astype(np.float32)
    bet = (0.3 * rng.normal(size=N)).astype(np.float32)

    def buf(a):
        return DBuf(dev, np.concatenate([np.full(shift, np.nan, np.float32), np.ravel(a)]))

    def at(b):
        return C.c_void_p(C.cast(b.p, C.c_void_p).value + 4 * shift)

    dx, dg, dgam, dbet = buf(x), buf(g), buf(gam), buf(bet)
    y, st, gin, gg, gb, wk = (buf(np.full(n, np.nan, np.float32)) for n in (rows * N, 2 * rows, rows * N, N, N, rows * N))
    scale, eps = np.float32(1) / np.float32(rows), C.c_float(1e-5)
    sc = C.c_float(scale)
    if kind == "ln":
        check(dev.h, L.gn_layernorm_forward(dev.h, at(dx), at(dgam), at(dbet), at(y), at(st), rows, N, eps))
        check(dev.h, L.gn_layernorm_backward(dev.h, at(dg), at(dx), at(dgam), at(st), at(gin), at(gg), at(gb), at(wk),
                                             rows, N, sc))
    else:
        check(dev.h, L.gn_rmsnorm_forward(dev.h, at(dx), at(dgam), at(y), at(st), rows, N, eps))
        check(dev.h, L.gn_rmsnorm_backward(dev.h, at(dg), at(dx), at(dgam), at(st), at(gin), at(gg), at(wk), rows, N, sc))
    want = _ref(kind, x, gam, bet, g, float(scale), 1e-5)
    for name, b, w in zip(("y", "dx", "dgamma", "dbeta"), (y, gin, gg, gb), want):
        if w is None:
            continue
        got = b.get().ravel()[shift:]
        assert got.size == w.size and np.isfinite(got).all(), name
        # a single column has x - mean = 0: the results are exact zeros or rounding
        r = np.abs(got - w.ravel()).max() / max(np.abs(w).max(), 1e-30) if np.abs(w).max() > 1e-6 else np.abs(got).max()
        assert r <= TOL, (name, r)


@pytest.mark.parametrize("kind", ["ln", "rms"])
@pytest.mark.parametrize("rows,N,shift", [(130, 63, 0), (5000, 64, 0), (130, 64, 3), (131, 65, 0), (129, 68, 0), (9, 2, 0)])
def test_norm_short_rows(dev, kind, rows, N, shift):
    """Both sides of the longest row that takes a column per lane."""
    test_norm_sizes(dev, kind, rows, N, shift)
