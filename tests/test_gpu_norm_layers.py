"""LayerNorm and RMSNorm of wide rows inside models, on both sides of the longest
row that the one-pass backward holds in registers (2048; beyond it the layers
and blocks keep a matrix for g * xhat) and of the model's own LayerNorm kernel
(512): two training steps against the oracle, every parameter tensor to 1e-4
(gpuutil.compare_step)."""
import numpy as np
import pytest

from gpuutil import compare_step, random_block

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["layernorm", "rmsnorm"])
@pytest.mark.parametrize("n,first", [(512, 0), (516, 0), (1024, 1), (2048, 0), (2052, 0), (2049, 1)])
def test_wide_norm_layers(gn, oracle, kind, n, first):
    """Dense -> norm -> Dense, or the norm first."""
    B, C = 24, 7
    rng = np.random.default_rng(n)
    norm = {"kind": kind, "n": n, "len": n} if kind == "layernorm" else {"kind": kind, "n": n}
    layers = [norm, {"kind": "dense", "in": n, "out": C, "act": "softmax", "ptr": True}]
    if not first:
        layers.insert(0, {"kind": "dense", "in": 20, "out": n, "act": "tanh", "ptr": False})
    cfg = dict(num=70, name=f"{kind}_{n}", B=B, loss="ce", lr=1e-3, x="normal", in_len=n if first else 20, classes=C,
               layers=layers)
    y = np.zeros((B, C), np.float32)
    y[np.arange(B), rng.integers(0, C, size=B)] = 1
    compare_step(gn, oracle, cfg, steps=2, xy=(rng.normal(size=(B, cfg["in_len"])).astype(np.float32), y))


@pytest.mark.parametrize("norm", ["ln", "rms"])
@pytest.mark.parametrize("dim,heads", [(576, 9), (2052, 27)])
def test_wide_blocks(gn, oracle, norm, dim, heads):
    """A transformer block of rows longer than 512 and longer than 2048."""
    from goneuron_amd import configs
    cfg = configs.gpt(B=3, T=5, vocab=13, dim=dim, heads=heads, ff=40, norm=norm)
    compare_step(gn, oracle, cfg, steps=1, perturb=random_block(cfg, scale=0.4 / np.sqrt(dim)))
