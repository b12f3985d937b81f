"""The few-tile GEMM kernels (gemm_small.hip), each configuration forced: every
layout and epilogue at edges of tiles, k tails and odd widths, bit for bit
against the other kernels (one MFMA chain over k either way), inside guard
bands. TN's FP32 output may split k elsewhere from k = 2048 on: below it is held
to the bits as well, and whole-number operands, whose sums are exact in any
order, show a missing or doubled product at every k. Beside that it stays within
2 k eps sum |x w| of float64."""

import pytest
import torch

from inputs import normal, uniform

pytestmark = pytest.mark.gpu

CONFIGS = ["32,32,5,8,2", "32,64,4,6,2", "64,64,8,6,2", "64,64,4,4,1", "128,64,8,3,1"]
H, F = torch.float16, torch.float32
GUARD = 1024


def _bits(t):
    return t.view(torch.int16 if t.dtype == H else torch.int32)


def _run(flint, call, outs, **plan):
    """The outputs of call(*outputs) under a plan, checked for stray stores."""
    bufs = []
    for shape, dtype in outs:
        count = 1
        for s in shape:
            count *= s
        buf = torch.full((count + 2 * GUARD,), float("nan"), dtype=dtype, device="cuda")
        buf[:GUARD] = 7.5
        buf[GUARD + count:] = 7.5
        bufs.append((buf, buf[GUARD:GUARD + count].view(shape), count))
    with flint.tuned(**plan):
        call(*(v for _, v, _ in bufs))
    torch.cuda.synchronize()
    for buf, _, count in bufs:
        assert bool((buf[:GUARD] == 7.5).all()), "wrote before an output"
        assert bool((buf[GUARD + count:] == 7.5).all()), "wrote past an output"
    return [v for _, v, _ in bufs]


def _same(flint, what, call, outs, cfg):
    ref = _run(flint, call, outs, gemm_small="0")
    got = _run(flint, call, outs, gemm_small=cfg)
    for a, b in zip(got, ref):
        assert torch.equal(_bits(a), _bits(b)), what


@pytest.mark.parametrize("cfg", CONFIGS)
@pytest.mark.parametrize("m,n,k", [(1, 8, 8), (33, 72, 24), (64, 64, 64), (200, 136, 72),
                                   (129, 264, 1000), (65, 64, 3072)])
def test_nt_and_nn(flint, cuda, cfg, m, n, k):
    x = uniform((m, k), 1).to(cuda)
    w = normal((n, k), 2, 0.05, H).to(cuda)
    b = normal((n,), 3).to(cuda)
    r = normal((m, n), 4).to(cuda)
    wn = w.t().contiguous()
    pre = normal((m, n), 5, 1.0, H).to(cuda)
    for what, call, outs in (
            ("nt", lambda y: flint.gemm_nt(y, x, w, m, n, k), [((m, n), H)]),
            ("bias", lambda y: flint.gemm_nt_bias(y, x, w, b, m, n, k), [((m, n), H)]),
            ("gelu", lambda y, p: flint.gemm_nt_bias_gelu(y, p, x, w, b, m, n, k),
             [((m, n), H), ((m, n), H)]),
            ("residual", lambda y: flint.gemm_nt_bias_residual(y, x, w, b, r, m, n, k),
             [((m, n), F)]),
            ("nn", lambda y: flint.gemm_nn(y, x, wn, m, n, k), [((m, n), H)]),
            ("dgelu", lambda y: flint.gemm_nn_dgelu(y, x, wn, pre, m, n, k), [((m, n), H)])):
        _same(flint, what, call, outs, cfg)


@pytest.mark.parametrize("cfg", CONFIGS)
@pytest.mark.parametrize("m,n,k", [(37, 53, 24), (1, 1, 8), (130, 998, 192)])
def test_nt_with_odd_widths(flint, cuda, cfg, m, n, k):
    x = uniform((m, k), 6).to(cuda)
    w = normal((n, k), 7, 0.05, H).to(cuda)
    b = normal((n,), 8).to(cuda)
    r = normal((m, n), 9).to(cuda)
    _same(flint, "nt", lambda y: flint.gemm_nt(y, x, w, m, n, k), [((m, n), H)], cfg)
    _same(flint, "gelu", lambda y, p: flint.gemm_nt_bias_gelu(y, p, x, w, b, m, n, k),
          [((m, n), H), ((m, n), H)], cfg)
    if n % 2 == 0:
        _same(flint, "residual", lambda y: flint.gemm_nt_bias_residual(y, x, w, b, r, m, n, k),
              [((m, n), F)], cfg)


@pytest.mark.parametrize("cfg", CONFIGS)
@pytest.mark.parametrize("m,n,k", [(8, 8, 1), (72, 200, 63), (64, 64, 64), (136, 120, 3000)])
@pytest.mark.parametrize("accumulate", [False, True])
def test_tn(flint, cuda, cfg, m, n, k, accumulate):
    x = normal((k, m), 10, 0.1, H).to(cuda)
    w = uniform((k, n), 11).to(cuda)
    y0 = normal((m, n), 12).to(cuda)
    ws = torch.empty(max(flint.gemm_tn_workspace(m, n, k), 16), dtype=torch.uint8, device=cuda)

    def call(y):
        y.copy_(y0)
        flint.gemm_tn(y, x, w, m, n, k, accumulate=accumulate, workspace=ws)

    got, = _run(flint, call, [((m, n), F)], gemm_small=cfg)
    ref = x.double().t() @ w.double() + (y0.double() if accumulate else 0)
    bound = 2 * k * 2.0 ** -24 * (x.double().abs().t() @ w.double().abs()) + 2.0 ** -22 * ref.abs()
    assert bool(((got.double() - ref).abs() <= bound).all())
    if k < 2048:
        _same(flint, "one piece", call, [((m, n), F)], cfg)
    x, w, y0 = (x * 20).round(), (w * 4).round(), (y0 * 4).round()
    got, = _run(flint, call, [((m, n), F)], gemm_small=cfg)
    assert torch.equal(got.double(), x.double().t() @ w.double() + (y0.double() if accumulate else 0))


@pytest.mark.parametrize("cfg", CONFIGS)
@pytest.mark.parametrize("batches,m,n,k", [(3, 40, 56, 24), (5, 264, 72, 96), (7, 200, 64, 200)])
def test_batched(flint, cuda, cfg, batches, m, n, k):
    x = uniform((batches, m, k), 13).to(cuda)
    w = uniform((batches, n, k), 14).to(cuda)
    wn = uniform((batches, k, n), 15).to(cuda)
    xt = uniform((batches, k, m), 16).to(cuda)
    outs = [((batches, m, n), H)]
    _same(flint, "nt", lambda y: flint.gemm_nt_batched(y, x, w, batches, m, n, k, 0.125), outs, cfg)
    _same(flint, "nn", lambda y: flint.gemm_nn_batched(y, x, wn, batches, m, n, k), outs, cfg)
    _same(flint, "tn", lambda y: flint.gemm_tn_batched(y, xt, wn, batches, m, n, k), outs, cfg)


@pytest.mark.parametrize("cfg", CONFIGS)
@pytest.mark.parametrize("length", [320, 32])
def test_the_models_causal_products_and_heads_views(flint, cuda, cfg, length):
    """The stored-probability model's attention products: k-ranges cut at the
    diagonal, operands and outputs as heads views. Logits, dlogits and losses
    bit for bit; gradients through TN's sums."""
    import test_gpt2 as model

    shape = dict(layers=1, heads=4, width=256, block_size=1024, vocab=1000, padded_vocab=1024)
    sizes = model.G.parameter_shapes(1, 256, 1024, 1024)
    params = model.G.init_params(sizes, 1, 1000, seed=17, trained=True)
    params = {name: t.half().float().cuda() for name, t in params.items()}
    idx, tgt = model._tokens(shape, 2, length, 18)
    tok, trg = model._dev16(idx), model._dev16(tgt)

    def passes(plan):
        with flint.tuned(gemm_small=plan):
            return model._model_passes(flint, shape, 2, length, params, tok, trg, 0.5, False)

    got, ref = passes(cfg), passes("0")
    for a, b in zip(got[:3], ref[:3]):
        assert torch.equal(_bits(a), _bits(b))
    for name in ref[3]:
        assert model._rel_l2(got[3][name], ref[3][name]) <= 1e-6, name


# The pipeline's k tails (NT and NN in whole 16-byte chunks, TN any k): the
# tile that takes them, forced, against the few-tile kernels' bits.
@pytest.mark.parametrize("m,n,k", [(129, 200, 72), (300, 136, 744), (257, 392, 8), (130, 200, 2056)])
def test_pipeline_k_tails(flint, cuda, m, n, k):
    x = uniform((m, k), 31).to(cuda)
    w = normal((n, k), 32, 0.05, H).to(cuda)
    x[:, -8:] *= 50.0          # the tail matters
    b = normal((n,), 33).to(cuda)
    r = normal((m, n), 34).to(cuda)
    wn = w.t().contiguous()
    pre = normal((m, n), 35, 1.0, H).to(cuda)
    for what, call, outs in (
            ("nt", lambda y: flint.gemm_nt(y, x, w, m, n, k), [((m, n), H)]),
            ("bias", lambda y: flint.gemm_nt_bias(y, x, w, b, m, n, k), [((m, n), H)]),
            ("gelu", lambda y, p: flint.gemm_nt_bias_gelu(y, p, x, w, b, m, n, k),
             [((m, n), H), ((m, n), H)]),
            ("residual", lambda y: flint.gemm_nt_bias_residual(y, x, w, b, r, m, n, k),
             [((m, n), F)]),
            ("nn", lambda y: flint.gemm_nn(y, x, wn, m, n, k), [((m, n), H)]),
            ("dgelu", lambda y: flint.gemm_nn_dgelu(y, x, wn, pre, m, n, k), [((m, n), H)])):
        ref = _run(flint, call, outs, gemm_small="64,64,4,4,1")
        got = _run(flint, call, outs, gemm_pipe="128,192,3,64", gemm_small="0")
        for a, c in zip(got, ref):
            assert torch.equal(_bits(a), _bits(c)), what


@pytest.mark.parametrize("cfg", ["128,192,3,64", "128,192,3,64,4,1", "256,256,3", "256,64,3,64"])
@pytest.mark.parametrize("m,n,k", [(136, 72, 1), (264, 200, 63), (136, 120, 3001)])
def test_pipeline_tn_takes_any_k(flint, cuda, cfg, m, n, k):
    x = normal((k, m), 36, 0.1, H).to(cuda)
    w = uniform((k, n), 37).to(cuda)
    ws = torch.empty(max(flint.gemm_tn_workspace(m, n, k), 16), dtype=torch.uint8, device=cuda)
    def call(y):
        flint.gemm_tn(y, x, w, m, n, k, workspace=ws)

    plan = dict(gemm_pipe=cfg, gemm_small="0")
    got, = _run(flint, call, [((m, n), F)], **plan)
    ref = x.double().t() @ w.double()
    bound = 2 * k * 2.0 ** -24 * (x.double().abs().t() @ w.double().abs()) + 2.0 ** -22 * ref.abs()
    assert bool(((got.double() - ref).abs() <= bound).all())
    if k < 2048:   # one piece
        few, = _run(flint, call, [((m, n), F)], gemm_small="64,64,4,4,1")
        assert torch.equal(_bits(got), _bits(few))
    x, w = (x * 20).round(), (w * 4).round()   # exact sums in any order
    got, = _run(flint, call, [((m, n), F)], **plan)
    assert torch.equal(got.double(), x.double().t() @ w.double())


def test_more_tiles_than_a_launch_holds(flint, cuda):
    """13.6 million 32 x 32 tiles of 320 threads are past the 2^32 threads of a
    launch: the forced configuration cannot run and the product runs as it
    would have, every value right (small whole numbers, exact in FP16)."""
    m, n, k = 8388480, 1664, 8
    x = (uniform((m, k), 41) * 4).round().to(cuda)
    w = (uniform((n, k), 42) * 4).round().to(cuda)
    y = torch.full((m, n), float("nan"), dtype=H, device=cuda)
    with flint.tuned(gemm_small="32,32,5,8,2"):
        flint.gemm_nt(y, x, w, m, n, k)
    torch.cuda.synchronize()
    wt = w.float().t().contiguous()
    for r in range(0, m, 262140):
        assert torch.equal(y[r:r + 262140].float(), x[r:r + 262140].float() @ wt), r


@pytest.mark.parametrize("plan", [{}, dict(gemm_small="0")], ids=["default", "general"])
@pytest.mark.parametrize("layout", ["nt", "nn", "tn"])
def test_an_operand_past_2_31_bytes(flint, cuda, layout, plan):
    """Where the pipeline's 32-bit offsets end: few tiles run the few-tile
    kernels, without them the general ones. Operands of -1, 0 and 1, so that
    every sum is a whole number below 2,048 (six of its standard deviations,
    171) and exact in FP32 and FP16 in any order."""
    big, few, k = 16416, 64, 65536
    g = torch.Generator(device=cuda).manual_seed(45)

    def signs(*shape):
        return torch.randint(-1, 2, shape, generator=g, device=cuda, dtype=H)

    if layout == "nt":
        x, w, m, n = signs(few, k), signs(big, k), few, big
        call, out = lambda y: flint.gemm_nt(y, x, w, m, n, k), H
    elif layout == "nn":
        x, w, m, n = signs(few, k), signs(k, big), few, big
        call, out = lambda y: flint.gemm_nn(y, x, w, m, n, k), H
    else:
        x, w, m, n = signs(k, big), signs(k, few), big, few
        ws = torch.empty(flint.gemm_tn_workspace(m, n, k), dtype=torch.uint8, device=cuda)
        call, out = lambda y: flint.gemm_tn(y, x, w, m, n, k, workspace=ws), F
    got, = _run(flint, call, [((m, n), out)], **plan)
    ref = torch.zeros(m, n, device=cuda)
    for c in range(0, k, 4096):
        xs = x[c:c + 4096].t() if layout == "tn" else x[:, c:c + 4096]
        ws_ = w[:, c:c + 4096].t() if layout == "nt" else w[c:c + 4096]
        ref += xs.float().contiguous() @ ws_.float().contiguous()
    assert float(ref.abs().max()) < 2048
    assert torch.equal(got.float(), ref)


def test_which_overrides_decide_the_kernel(flint, cuda):
    """TN 768 x 768 x 3000 shows its plan in its bits: by default the few-tile
    kernels sum k in one piece, the pipeline and the general kernel in two of
    1,536 and 1,464. A gemm_pipe value that names no tile, or one that cannot
    run TN, leaves the default; gemm_config, as k is not whole 32-deep steps,
    means the general kernel."""
    m, n, k = 768, 768, 3000
    x = normal((k, m), 43, 0.1, H).to(cuda)
    w = uniform((k, n), 44).to(cuda)
    ws = torch.empty(flint.gemm_tn_workspace(m, n, k), dtype=torch.uint8, device=cuda)

    def bits(**plan):
        got, = _run(flint, lambda y: flint.gemm_tn(y, x, w, m, n, k, workspace=ws), [((m, n), F)],
                    **plan)
        return _bits(got).clone()

    default, two = bits(), bits(gemm_small="0")
    assert not torch.equal(default, two)
    for value in ("", "default", "128,192", "96,96,3", "256,192,2,64,8"):
        assert torch.equal(bits(gemm_pipe=value), default), value
    assert torch.equal(bits(gemm_pipe="128,192,3,64"), two)
    assert torch.equal(bits(gemm_pipe="0"), two)
    assert torch.equal(bits(gemm_config="128,192,64,2,2,4"), two)
    assert torch.equal(bits(gemm_config="96,96,64,2,2,4"), default)
    assert torch.equal(bits(gemm_config="128,192,64,2,2,4", gemm_small="64,64,8,6,2"), default)
