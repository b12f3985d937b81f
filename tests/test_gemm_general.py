"""gemm.hip's kernels, which by default only run what neither the pipeline nor
the few-tile kernels take: every layout, epilogue and tile with the other two
turned off, against float64. A value may miss it by the rounding of its sums
(2 k 2^-24 sum |x w|, and what the epilogue's slope of at most 1.2 makes of it),
its own (2^-11, 2^-24 where FP16 is subnormal) and GELU's 2^-19."""

import math

import pytest
import torch

from inputs import normal, uniform

pytestmark = pytest.mark.gpu

H, F = torch.float16, torch.float32
TILES = [None, "128,192,64,2,2", "256,192,64,2,2", "128,128,64,2,2", "64,128,64,2,1",
         "128,64,64,2,4", "128,256,64,2,2", "128,192,64,3,2"]
# Whole tiles and k-steps of every tile; edges of both, and k tails; less than one tile.
SHAPES = [(512, 768, 192), (300, 264, 200), (129, 72, 1000), (40, 8, 8)]


@pytest.fixture
def general(flint, tune, request):
    tune("gemm_pipe", "0")
    if request.param is not None:
        tune("gemm_config", request.param)
    return flint


def _near(what, got, ref, sums, slope=1.0):
    """sums: the sums' error bound. FP32 outputs have no rounding of FP16."""
    half = got.dtype == H
    bound = slope * sums + (2.0 ** -11 * ref.abs() + 2.0 ** -24 if half else 2.0 ** -23 * ref.abs())
    if slope != 1.0:
        bound = bound + 2.0 ** -19 * ref.abs()
    torch.cuda.synchronize()
    assert bool(((got.double() - ref).abs() <= bound).all()), what


def _sums(x, w, k):
    return 2 * k * 2.0 ** -24 * (x.double().abs() @ w.double().abs())


def _gelu(s):
    return 0.5 * s * (1 + torch.tanh(math.sqrt(2 / math.pi) * (s + 0.044715 * s ** 3)))


def _gelu_grad(s):
    u = math.sqrt(2 / math.pi) * (s + 0.044715 * s ** 3)
    t = torch.tanh(u)
    return 0.5 * (1 + t) + 0.5 * s * (1 - t * t) * math.sqrt(2 / math.pi) * (1 + 3 * 0.044715 * s * s)


@pytest.mark.parametrize("general", TILES, indirect=True)
@pytest.mark.parametrize("m,n,k", SHAPES + [(37, 53, 24), (200, 998, 136)])
def test_nt(general, cuda, m, n, k):
    x, w = uniform((m, k), 1).to(cuda), normal((n, k), 2, 0.1, H).to(cuda)
    b, r = normal((n,), 3).to(cuda), normal((m, n), 4).to(cuda)
    wt = w.t().contiguous()
    plain, sums = x.double() @ wt.double(), _sums(x, wt, k)
    biased = plain + b.double()
    sums_b = sums + 2.0 ** -23 * (plain.abs() + b.double().abs())
    y = torch.full((m, n), float("nan"), dtype=H, device=cuda)
    general.gemm_nt(y, x, w, m, n, k)
    _near("plain", y, plain, sums)
    general.gemm_nt_bias(y.fill_(float("nan")), x, w, b, m, n, k)
    _near("bias", y, biased, sums_b)
    pre = torch.full_like(y, float("nan"))
    general.gemm_nt_bias_gelu(y.fill_(float("nan")), pre, x, w, b, m, n, k)
    _near("pre", pre, biased, sums_b)
    _near("gelu", y, _gelu(biased), sums_b, 1.2)
    if n % 2 == 0:
        out = torch.full((m, n), float("nan"), device=cuda)
        general.gemm_nt_bias_residual(out, x, w, b, r, m, n, k)
        _near("residual", out, r.double() + biased, sums_b)


@pytest.mark.parametrize("general", TILES, indirect=True)
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_nn(general, cuda, m, n, k):
    x, w = uniform((m, k), 5).to(cuda), normal((k, n), 6, 0.1, H).to(cuda)
    pre = normal((m, n), 7, 2.0, H).to(cuda)
    plain, sums = x.double() @ w.double(), _sums(x, w, k)
    y = torch.full((m, n), float("nan"), dtype=H, device=cuda)
    general.gemm_nn(y, x, w, m, n, k)
    _near("plain", y, plain, sums)
    general.gemm_nn_dgelu(y.fill_(float("nan")), x, w, pre, m, n, k)
    # The derivative's own 2^-19 is of its terms, which cancel where it is small.
    _near("dgelu", y, plain * _gelu_grad(pre.double()), sums + 2.0 ** -19 * plain.abs(), 1.2)


@pytest.mark.parametrize("general", TILES, indirect=True)
@pytest.mark.parametrize("m,n,k", [(512, 768, 192), (304, 264, 200), (136, 72, 1000), (40, 8, 8),
                                   (72, 200, 1), (136, 120, 3001), (8, 8, 16384)])   # m in eights
@pytest.mark.parametrize("accumulate", [False, True])
def test_tn(general, cuda, m, n, k, accumulate):
    x, w = normal((k, m), 8, 0.1, H).to(cuda), uniform((k, n), 9).to(cuda)
    y0 = normal((m, n), 10).to(cuda)
    ws = torch.empty(max(general.gemm_tn_workspace(m, n, k), 16), dtype=torch.uint8, device=cuda)
    y = y0.clone()
    general.gemm_tn(y, x, w, m, n, k, accumulate=accumulate, workspace=ws)
    xt = x.t().contiguous()
    ref = xt.double() @ w.double()
    sums = _sums(xt, w, k)
    if accumulate:
        sums = sums + 2.0 ** -23 * (ref.abs() + y0.double().abs())
        ref = ref + y0.double()
    _near("tn", y, ref, sums)
    if k <= 1024:   # one piece: whole numbers come out exactly, so no product is missed or doubled
        xi, wi = (x * 20).round(), (w * 4).round()
        general.gemm_tn(y, xi, wi, m, n, k, workspace=ws)
        torch.cuda.synchronize()
        assert torch.equal(y.double(), xi.t().double() @ wi.double())


@pytest.mark.parametrize("general", TILES, indirect=True)
@pytest.mark.parametrize("batches,m,n,k", [(3, 512, 768, 192), (5, 200, 136, 72), (7, 40, 56, 24)])
def test_batched(general, cuda, batches, m, n, k):
    x, w = uniform((batches, m, k), 11).to(cuda), uniform((batches, n, k), 12).to(cuda)
    wt, xt = w.transpose(1, 2).contiguous(), x.transpose(1, 2).contiguous()
    ref = torch.stack([x[i].double() @ wt[i].double() for i in range(batches)])
    sums = torch.stack([_sums(x[i], wt[i], k) for i in range(batches)])
    y = torch.full((batches, m, n), float("nan"), dtype=H, device=cuda)
    general.gemm_nt_batched(y, x, w, batches, m, n, k, 0.125)
    _near("nt", y, 0.125 * ref, 0.125 * sums)
    general.gemm_nn_batched(y.fill_(float("nan")), x, wt, batches, m, n, k)
    _near("nn", y, ref, sums)
    general.gemm_tn_batched(y.fill_(float("nan")), xt, wt, batches, m, n, k)
    _near("tn", y, ref, sums)
