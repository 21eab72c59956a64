"""A Dense stack whose backward products all run on the split-bf16 GEMM, in tiles
that end inside the matrices (1600 = 12.5 x 128), with each activation
derivative in the dX epilogue: every layer's gradient against float64.  A ReLU
unit's branch is the GPU forward's (its pre-activation may lie within rounding
of 0).  Bound, in the 2-norm of a layer's gradient: a product of K = 1600 terms
errs by less than sqrt(K) 2^-24 of its norm, and the output layer's gradient
passes at most four products on its way down."""
import numpy as np
import pytest

from gpuutil import log

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("acts", [("tanh", "relu", "sigmoid"), ("relu", "relu", "relu")])
def test_dense_stack_all_layers_vs_float64(gn, acts):
    torch = pytest.importorskip("torch")
    from goneuron_amd import configs
    n, C = 1600, 320
    log(f"dense stack {acts} against float64")
    rng = np.random.default_rng(4)
    layers = [configs.dense(n, n, a) for a in acts] + [configs.dense(n, C, "logsoftmax", True)]
    cfg = dict(num=80, name="dense_split", B=n, loss="ce", lr=1e-3, x="normal", in_len=n, classes=C, layers=layers)
    x = rng.normal(size=(n, n)).astype(np.float32)
    y = np.zeros((n, C), np.float32)
    y[np.arange(n), rng.integers(0, C, size=n)] = 1
    model = configs.build(cfg)
    p0 = model.Params()
    model.TrainBatch(x, y)
    got = model.Gradients()
    dev = torch.device("cuda:0")
    P = torch.tensor(p0.astype(np.float64), device=dev, requires_grad=True)
    h, at, sl = torch.tensor(x.astype(np.float64), device=dev), 0, []
    for i, d in enumerate(layers):
        w = d["in"] * d["out"]
        z = h @ P[at:at + w].view(d["out"], d["in"]).T + P[at + w:at + w + d["out"]]
        sl.append(slice(at, at + w + d["out"]))
        at = sl[-1].stop
        if d["act"] == "relu":
            h = z * torch.tensor(model.LayerOutput(i, n * d["out"]).reshape(n, d["out"]) > 0, device=dev)
        else:
            h = {"tanh": torch.tanh, "sigmoid": torch.sigmoid, "logsoftmax": lambda v: torch.log_softmax(v, 1)}[d["act"]](z)
    h.backward(((h - torch.tensor(y.astype(np.float64), device=dev)) / n).detach())
    ref = P.grad.cpu().numpy()
    for i, s in enumerate(sl):
        err = np.linalg.norm(got[s] - ref[s]) / np.linalg.norm(ref[s])
        log(f"  layer {i}: {err:.2e}")
        assert err <= 4 * np.sqrt(n) * 2.0 ** -24, (i, err)
    model.Close()
