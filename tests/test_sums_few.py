"""Column sums of few 256-row chunks finished in their own launch: the bias
gradient (up to 8 chunks) and LayerNorm backward's dbeta and dgamma (one),
at the chunk counts where the plans change and past them, bit for bit against
the C oracle, with infinities, NaN and -0 among the values."""

import numpy as np
import pytest
import torch

import gpt2_model as G
from inputs import normal
from oracle import oracle
from test_gpt2 import _dev16, _load, _make, _tokens

pytestmark = pytest.mark.gpu


def _bits(t):
    a = t.cpu().numpy() if torch.is_tensor(t) else t
    return np.where(np.isnan(a), np.float32(np.nan), a).view(np.int32)   # any NaN as one NaN


@pytest.mark.parametrize("rows", [1, 7, 255, 256, 257, 512, 1000, 1024, 1025, 2048, 2049])
@pytest.mark.parametrize("cols", [8, 72, 200])
def test_bias_gradient(flint, cuda, rows, cols):
    dy = normal((rows, cols), rows, 1.0, torch.float16)
    dy[:, 1] = -0.0
    dy[rows // 2, 2] = float("inf")
    dy[0, 3], dy[rows - 1, 3] = float("inf"), float("-inf")
    dy[rows - 1, 4] = float("nan")
    old = normal((cols,), 7)
    old[1] = -0.0
    for accumulate in (False, True):
        out = old.clone().to(cuda)
        flint.bias_gradient(out, dy.to(cuda), rows, cols, accumulate=accumulate)
        torch.cuda.synchronize()
        ref = oracle.bias_gradient(dy.numpy(), old.numpy() if accumulate else None)
        assert np.array_equal(_bits(out), _bits(ref))


# Either side of each line of bias_gradient_one_launch.
@pytest.mark.parametrize("rows,cols", [(512, 8192), (512, 8200), (513, 6232), (513, 6240),
                                       (1024, 3120), (1024, 3128), (1536, 1608), (1536, 1616),
                                       (2048, 904), (2048, 912)])
def test_bias_gradient_where_the_plan_changes(flint, cuda, tune, rows, cols):
    dy = normal((rows, cols), rows, 1.0, torch.float16).to(cuda)

    def run():
        out = normal((cols,), 7).to(cuda)
        flint.bias_gradient(out, dy, rows, cols, accumulate=True)
        torch.cuda.synchronize()
        return out

    got = run()
    tune("sums_few", "0")
    assert np.array_equal(_bits(got), _bits(run()))


@pytest.mark.parametrize("rows", [1, 256, 257, 1000, 1024, 1025])
@pytest.mark.parametrize("cols", [8, 264, 768])
@pytest.mark.parametrize("accumulate", [False, True])
def test_layernorm_parameter_sums(flint, cuda, tune, rows, cols, accumulate):
    x = normal((rows, cols), 11)
    gamma, beta = 1 + normal((cols,), 12, 0.1), normal((cols,), 13, 0.1)
    dy = normal((rows, cols), 14, 1.0, torch.float16)
    dy[:, 1] = -0.0
    dy[rows // 2, 2] = float("inf")
    xg, gg, dyg = x.to(cuda), gamma.to(cuda), dy.to(cuda)
    mean, rstd = torch.empty(rows, device=cuda), torch.empty(rows, device=cuda)
    y = torch.empty((rows, cols), dtype=torch.float16, device=cuda)
    flint.layernorm_forward(y, mean, rstd, xg, gg, beta.to(cuda), rows, cols)

    def run():
        dx = torch.zeros((rows, cols), device=cuda)
        dgamma, dbeta = normal((cols,), 15).to(cuda), normal((cols,), 16).to(cuda)
        flint.layernorm_backward(dx, dgamma, dbeta, dyg, xg, mean, rstd, gg, rows, cols,
                                 accumulate_dx=True, accumulate_params=accumulate)
        torch.cuda.synchronize()
        return dx, dgamma, dbeta

    got = run()
    tune("sums_few", "0")
    for a, b in zip(got, run()):
        assert np.array_equal(_bits(a), _bits(b))
    ref = oracle.bias_gradient(dy.numpy(), normal((cols,), 16).numpy() if accumulate else None)
    assert np.array_equal(_bits(got[2]), _bits(ref))


@pytest.mark.parametrize("sequences,length", [(1, 8), (4, 64), (1, 264), (16, 72), (32, 64)])
def test_model_bias_gradients(flint, cuda, tune, sequences, length):
    """Two layers' bias gradients in one launch (widths 96 beside 384, 288
    beside 96: a part of a column block at either end) against two passes each,
    in a fresh and in an accumulating backward."""
    cfg = dict(layers=2, heads=3, width=96, block_size=272, vocab=997, padded_vocab=1000)
    shapes = G.parameter_shapes(cfg["layers"], cfg["width"], cfg["block_size"],
                                cfg["padded_vocab"])
    params = G.init_params(shapes, cfg["layers"], cfg["vocab"], seed=3, trained=True)
    idx, tgt = _tokens(cfg, sequences, length, 4)

    def run():
        with _make(flint, cfg, sequences, length) as model:
            _load(model, params)
            tok = _dev16(idx)
            model.forward(tok, _dev16(tgt), 0.5)
            model.backward(tok)
            model.backward(tok, accumulate=True)
            torch.cuda.synchronize()
            return {n: model.read(a, (r, c), torch.float32).cpu() for n, a, r, c in model.gradients()
                    if n.endswith("bias")}

    got = run()
    tune("sums_few", "0")
    for n, g in run().items():
        assert torch.equal(g.view(torch.int32), got[n].view(torch.int32)), n
