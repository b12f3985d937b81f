"""Token runs of the sort-free embedding backward at the lengths where its plan
changes: one wave up to 16 rows, the whole workgroup beyond, 16 rows a batch and
64 list entries a read; widths with one and two columns a thread and a partial
last group. The C oracle's order, bit for bit, rows that hold -0 and infinities
included."""

import numpy as np
import pytest
import torch

from inputs import normal
from oracle import oracle

pytestmark = pytest.mark.gpu

RUNS = [1, 4, 5, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 129]


@pytest.mark.parametrize("width", [8, 256, 264, 520, 768, 1000])
def test_runs_of_every_length(flint, cuda, width):
    _check(flint, cuda, RUNS, width)


@pytest.mark.parametrize("width", [8, 264, 768])
@pytest.mark.parametrize("rows", [2000, 2600, 8192])
def test_short_runs_over_many_workgroups(flint, cuda, width, rows):
    """Beside the long runs mostly pairs, whose rows lie blocks apart, and
    single rows; more positions than workgroups, up to the most tokens."""
    left = rows - sum(RUNS)
    _check(flint, cuda, RUNS + [2] * (left // 4) + [1] * (left - left // 4 * 2), width)


def _check(flint, cuda, runs, width):
    vocab = len(runs) + 3
    tok = torch.cat([torch.full((n,), v, dtype=torch.int64) for v, n in enumerate(runs)])
    tok = tok[torch.randperm(len(tok), generator=torch.Generator().manual_seed(width))]
    sequences, length = 1, len(tok)
    dx = normal((length, width), 21)
    dx[:, 1::7] *= 3000.0
    dx[:, 2] = -0.0
    dx[tok == 9, 3] = float("inf")
    wte, wpe = normal((vocab, width), 22), normal((length, width), 23)
    wte[:, 2] = -0.0
    dwte, dwpe = wte.clone().to(cuda), wpe.clone().to(cuda)
    flint.embedding_backward(dwte, dwpe, dx.to(cuda), tok.to(torch.int16).to(cuda), sequences,
                             length, vocab, width, accumulate_wte=True, accumulate_wpe=True)
    torch.cuda.synchronize()
    ewte, ewpe = oracle.embedding_backward(dx.numpy(), tok.numpy().astype(np.uint16), sequences,
                                           length, vocab, width, wte.numpy(), wpe.numpy())
    assert np.array_equal(dwte.cpu().numpy().view(np.int32), ewte.view(np.int32))
    assert np.array_equal(dwpe.cpu().numpy().view(np.int32), ewpe.view(np.int32))
