"""What a user of this library has it do, as measurable cases.

A training or evaluation program calls libflint in two ways: it composes a
model from the public kernels block by block (embedding, attention layer, MLP,
output head, optimizer), or it hands whole passes to the assembled GPT-2
(flint_gpt2_*). Each case below is one such call sequence at one size, through
the ctypes binding, on torch's current stream, with every buffer and workspace
kept by the program:

  mlp        LayerNorm, up + bias + GELU, down + bias + residual; training adds
             the whole backward, gradients of every parameter and of the input
  attention  LayerNorm, the qkv projection, causal attention over the heads
             (fused, or with the scores and probabilities stored), projection +
             bias + residual; training adds the whole backward
  head       logits and softmax + cross-entropy (which writes dlogits);
             training adds the gradients of the table and of the input
  embedding  token + position rows; training adds both tables' gradients, the
             token rows adding onto the output head's gradient
  adamw      one clipped, loss-scaled AdamW step over a model's tensors
  model      flint_gpt2_forward, and flint_gpt2_backward when training

Sizes run from one short sequence through a small model to the GPT-2 124M
shapes at 8,192 tokens that the benchmark suite times.
"""

import math

import torch

from flint_amd.flint_lib import Flint, Gpt2

GPT2 = dict(layers=12, heads=12, width=768, block_size=1024, vocab=50257, padded_vocab=50304)


def listed():
    return [
        # One prompt of 64 tokens through a GPT-2 MLP: evaluation, where launch
        # latency and the few rows count.
        dict(name="mlp-eval-64", kind="mlp", tokens=64, width=768, train=False),
        # A small model's MLP on a batch that is no multiple of anything, its
        # width a multiple of 8 and not of 32.
        dict(name="mlp-train-1000x200", kind="mlp", tokens=1000, width=200, train=True),
        # The GPT-2 124M MLP at the benchmark's 8,192 tokens.
        dict(name="mlp-train-8192", kind="mlp", tokens=8192, width=768, train=True),
        # One odd-length sequence through the fused attention: evaluation.
        dict(name="attention-eval-1x200", kind="attention", sequences=1, length=200, heads=12,
             head_width=64, fused=True, train=False),
        # The GPT-2 124M attention layer at 8 x 1024, fused.
        dict(name="attention-train-8x1024", kind="attention", sequences=8, length=1024, heads=12,
             head_width=64, fused=True, train=True),
        # The same layer with stored probabilities, composed call by call as
        # the reference's sequence is, on a short batch.
        dict(name="attention-stored-2x256", kind="attention", sequences=2, length=256, heads=12,
             head_width=64, fused=False, train=True),
        # A character-sized vocabulary's output head, odd rows.
        dict(name="head-train-777x997", kind="head", tokens=777, width=192, vocab=997,
             padded_vocab=1000, train=True),
        # The GPT-2 124M output head.
        dict(name="head-train-8192", kind="head", tokens=8192, width=768, vocab=50257,
             padded_vocab=50304, train=True),
        # The GPT-2 124M embedding on text-like tokens (few words make up most
        # of it).
        dict(name="embedding-train-8x1024", kind="embedding", sequences=8, length=1024,
             vocab=50257, width=768, train=True),
        # The optimizer step of GPT-2 124M.
        dict(name="adamw-124m", kind="adamw", **GPT2),
        # A whole training micro-step of the default model on one short
        # sequence (fine-tuning, or a step of the tests' gate).
        dict(name="model-train-1x256", kind="model", sequences=1, length=256, fused=False,
             train=True, **GPT2),
        # The benchmark's training micro-step: 8 x 1024 tokens, fused attention.
        dict(name="model-train-8x1024", kind="model", sequences=8, length=1024, fused=True,
             train=True, **GPT2),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["mlp", "mlp", "attention", "attention", "head", "embedding", "adamw",
                       "model"])
    train = rng.random() < 0.7
    if kind == "mlp":
        # Half the widths are whole heads of 64, the others any multiple of 8.
        width = 64 * rng.randint(1, 12) if rng.random() < 0.5 else 8 * rng.randint(8, 96)
        return dict(kind=kind, tokens=_log_int(rng, 16, 8192), width=width, train=train)
    if kind == "attention":
        fused = rng.random() < 0.6
        sequences = _log_int(rng, 1, 8)
        length = _log_int(rng, 16, 1024)
        if not fused:
            length = max(16, length // 8 * 8)   # stored rows are 16-byte multiples
        head_width = 64 if fused or rng.random() < 0.7 else 32
        return dict(kind=kind, sequences=sequences, length=length, heads=rng.randint(1, 12),
                    head_width=head_width, fused=fused, train=train)
    if kind == "head":
        vocab = rng.choice([_log_int(rng, 100, 50257), 50257])
        pad = rng.choice([8, 64, 128])
        return dict(kind=kind, tokens=_log_int(rng, 16, 8192), width=64 * rng.randint(1, 12),
                    vocab=vocab, padded_vocab=(vocab + pad - 1) // pad * pad, train=train)
    if kind == "embedding":
        return dict(kind=kind, sequences=_log_int(rng, 1, 8), length=_log_int(rng, 16, 1024),
                    vocab=rng.choice([_log_int(rng, 100, 50257), 50257]),
                    width=8 * rng.randint(8, 96), train=train)
    shape = _model_shape(rng)
    if kind == "adamw":
        return dict(kind=kind, **shape)
    length = max(16, _log_int(rng, 16, shape["block_size"]) // 8 * 8)
    return dict(kind=kind, sequences=_log_int(rng, 1, 8), length=length,
                fused=rng.random() < 0.5, train=train, **shape)


def _model_shape(rng):
    heads = rng.randint(1, 12)
    vocab = rng.choice([1000, _log_int(rng, 100, 50257), 50257])
    return dict(layers=rng.randint(1, 12), heads=heads, width=64 * heads,
                block_size=1024, vocab=vocab, padded_vocab=(vocab + 63) // 64 * 64)


# ------------------------------------------------------------------ inputs
_library = None


def _flint():
    global _library
    if _library is None:
        _library = Flint()
    return _library


class _Make:
    """Seeded tensors on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, shape, std=1.0, mean=0.0, dtype=torch.float32):
        t = torch.randn(shape, generator=self.g, device="cuda", dtype=torch.float32)
        return (t * std + mean).to(dtype)

    def weight(self, rows, cols, std=0.02):
        return self.normal((rows, cols), std, dtype=torch.float16)

    def residual(self, rows, cols):
        """A residual stream: unit activations, a few outlier channels."""
        t = self.normal((rows, cols))
        t[:, ::97] *= 8.0
        return t

    def tokens(self, count, vocab):
        """Text-like ids: frequencies fall as 1 / (rank + 2.7), the frequent
        words anywhere in the vocabulary. uint16 values held in int16."""
        u = torch.rand(count, generator=self.g, device="cuda", dtype=torch.float64)
        rank = (2.7 * (((vocab + 2.7) / 2.7) ** u - 1.0)).long().clamp_(max=vocab - 1)
        order = torch.randperm(vocab, generator=self.g, device="cuda")
        return order[rank].to(torch.int32).to(torch.int16)


def _half(*shape):
    return torch.empty(shape, dtype=torch.float16, device="cuda")


def _single(*shape):
    return torch.empty(shape, dtype=torch.float32, device="cuda")


def _bytes(n):
    return torch.empty(max(int(n), 16), dtype=torch.uint8, device="cuda")


def _ids(tokens):
    return tokens.long() & 0xFFFF


class _Memory:
    """Model memory as torch sees it, without a copy; keeps the model alive."""

    def __init__(self, owner, address, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=shape, typestr=typestr, version=2,
                                             data=(address, False), strides=None)


class _Model(Gpt2):
    def __del__(self):
        self.close()

    def view(self, address, shape, typestr):
        return torch.as_tensor(_Memory(self, address, shape, typestr), device="cuda")


def prepare(case, seed):
    f = _flint()
    s = dict(case=case, f=f)
    s.update(_PREPARE[case["kind"]](f, case, _Make(seed)))
    return s


def run(state):
    return _RUN[state["case"]["kind"]](state["f"], state["case"], state)


# --------------------------------------------------------------------- mlp
def _norm_inputs(mk, width):
    return dict(gamma=mk.normal((width,), 0.1, 1.0), beta=mk.normal((width,), 0.1))


def _mlp_inputs(f, case, mk):
    rows, w = case["tokens"], case["width"]
    s = dict(x=mk.residual(rows, w), **_norm_inputs(mk, w))
    s.update(w_up=mk.weight(4 * w, w), b_up=mk.normal((4 * w,), 0.02),
             w_down=mk.weight(w, 4 * w), b_down=mk.normal((w,), 0.02))
    s.update(h=_half(rows, w), mean=_single(rows), rstd=_single(rows), gelu=_half(rows, 4 * w),
             pre=_half(rows, 4 * w), y=_single(rows, w))
    if case["train"]:
        s.update(dy=mk.normal((rows, w), 0.05), dx=_single(rows, w), g=_half(rows, w),
                 dpre=_half(rows, 4 * w), dh=_half(rows, w), dw_up=_single(4 * w, w),
                 db_up=_single(4 * w), dw_down=_single(w, 4 * w), db_down=_single(w),
                 dgamma=_single(w), dbeta=_single(w),
                 ws=_bytes(max(f.gemm_tn_workspace(4 * w, w, rows),
                               f.gemm_tn_workspace(w, 4 * w, rows),
                               f.bias_gradient_workspace(rows, 4 * w),
                               f.layernorm_backward_workspace(rows, w))))
    return s


def _mlp_run(f, case, s):
    rows, w = case["tokens"], case["width"]
    f.layernorm_forward(s["h"], s["mean"], s["rstd"], s["x"], s["gamma"], s["beta"], rows, w)
    f.gemm_nt_bias_gelu(s["gelu"], s["pre"], s["h"], s["w_up"], s["b_up"], rows, 4 * w, w)
    f.gemm_nt_bias_residual(s["y"], s["gelu"], s["w_down"], s["b_down"], s["x"], rows, w, 4 * w)
    if not case["train"]:
        return dict(y=s["y"])
    ws = s["ws"]
    f.copy(s["dx"], s["dy"], rows * w * 4)   # the residual branch; the block's adds to it
    f.fp32_to_fp16(s["g"], s["dy"], rows * w)
    f.gemm_tn(s["dw_down"], s["g"], s["gelu"], w, 4 * w, rows, workspace=ws)
    f.bias_gradient(s["db_down"], s["g"], rows, w, workspace=ws)
    f.gemm_nn_dgelu(s["dpre"], s["g"], s["w_down"], s["pre"], rows, 4 * w, w)
    f.gemm_tn(s["dw_up"], s["dpre"], s["h"], 4 * w, w, rows, workspace=ws)
    f.bias_gradient(s["db_up"], s["dpre"], rows, 4 * w, workspace=ws)
    f.gemm_nn(s["dh"], s["dpre"], s["w_up"], rows, w, 4 * w)
    f.layernorm_backward(s["dx"], s["dgamma"], s["dbeta"], s["dh"], s["x"], s["mean"], s["rstd"],
                         s["gamma"], rows, w, accumulate_dx=True, workspace=ws)
    return {k: s[k] for k in ("y", "dx", "dw_up", "db_up", "dw_down", "db_down", "dgamma",
                              "dbeta")}


def _leaf(t):
    return t.double().requires_grad_(True)


def _norm64(x, gamma, beta):
    return torch.nn.functional.layer_norm(x, (x.shape[-1],), gamma, beta, 1e-5)


def _gelu64(x):
    return torch.nn.functional.gelu(x, approximate="tanh")


def _mlp_exact(case, s):
    names = ("x", "gamma", "beta", "w_up", "b_up", "w_down", "b_down")
    p = {n: _leaf(s[n]) for n in names}
    h = _norm64(p["x"], p["gamma"], p["beta"])
    u = _gelu64(h @ p["w_up"].T + p["b_up"])
    y = p["x"] + (u @ p["w_down"].T + p["b_down"])
    out = dict(y=y.detach())
    if case["train"]:
        y.backward(s["dy"].double())
        out.update({"d" + n: p[n].grad for n in names if not n.startswith(("w_", "b_"))})
        out.update({"d" + n: p[n].grad for n in names if n.startswith(("w_", "b_"))})
    return out


def _mlp_work(case):
    m, w = case["tokens"], case["width"]
    gemm = 2 * m * w * 4 * w
    weights = 2 * 4 * w * w
    if not case["train"]:
        return dict(flops=2 * gemm, bytes=m * w * 8 + weights * 2)
    return dict(flops=6 * gemm, bytes=m * w * (4 + 4 + 4 + 4) + weights * (2 + 4))


# --------------------------------------------------------------- attention
def _attention_inputs(f, case, mk):
    S, T, H, hw = case["sequences"], case["length"], case["heads"], case["head_width"]
    rows, w, nb = S * T, H * hw, S * H
    s = dict(x=mk.residual(rows, w), **_norm_inputs(mk, w))
    s.update(w_qkv=mk.weight(3 * w, w, 0.05), b_qkv=mk.normal((3 * w,), 0.02),
             w_proj=mk.weight(w, w), b_proj=mk.normal((w,), 0.02))
    s.update(h=_half(rows, w), mean=_single(rows), rstd=_single(rows), qkv=_half(rows, 3 * w),
             q=_half(nb, T, hw), k=_half(nb, T, hw), v=_half(nb, T, hw), o=_half(nb, T, hw),
             attn=_half(rows, w), y=_single(rows, w))
    if case["fused"]:
        s.update(lse=_single(nb, T))
    else:
        s.update(scores=_half(nb, T, T), p=_half(nb, T, T))
    if case["train"]:
        s.update(dy=mk.normal((rows, w), 0.05), dx=_single(rows, w), g=_half(rows, w),
                 dattn=_half(rows, w), do=_half(nb, T, hw), dq=_half(nb, T, hw),
                 dk=_half(nb, T, hw), dv=_half(nb, T, hw), dqkv=_half(rows, 3 * w),
                 dh=_half(rows, w), dw_qkv=_single(3 * w, w), db_qkv=_single(3 * w),
                 dw_proj=_single(w, w), db_proj=_single(w), dgamma=_single(w), dbeta=_single(w))
        need = [f.gemm_tn_workspace(3 * w, w, rows), f.gemm_tn_workspace(w, w, rows),
                f.bias_gradient_workspace(rows, 3 * w), f.layernorm_backward_workspace(rows, w)]
        if case["fused"]:
            need.append(f.attention_backward_workspace(nb, T, hw))
        else:
            s.update(ds=_half(nb, T, T))
        s.update(ws=_bytes(max(need)))
    return s


def _attention_run(f, case, s):
    S, T, H, hw = case["sequences"], case["length"], case["heads"], case["head_width"]
    rows, w, nb = S * T, H * hw, S * H
    scale = 1.0 / math.sqrt(hw)
    f.layernorm_forward(s["h"], s["mean"], s["rstd"], s["x"], s["gamma"], s["beta"], rows, w)
    f.gemm_nt_bias(s["qkv"], s["h"], s["w_qkv"], s["b_qkv"], rows, 3 * w, w)
    for j, part in enumerate("qkv"):
        f.heads_split(s[part], s["qkv"], S, T, H, hw, 3 * w, j * w)
    if case["fused"]:
        f.attention_forward(s["o"], s["lse"], s["q"], s["k"], s["v"], nb, T, hw, scale)
    else:
        f.gemm_nt_batched(s["scores"], s["q"], s["k"], nb, T, T, hw, scale)
        f.causal_softmax_forward(s["p"], s["scores"], nb, T)
        f.gemm_nn_batched(s["o"], s["p"], s["v"], nb, T, hw, T)
    f.heads_merge(s["attn"], s["o"], S, T, H, hw, w, 0)
    f.gemm_nt_bias_residual(s["y"], s["attn"], s["w_proj"], s["b_proj"], s["x"], rows, w, w)
    if not case["train"]:
        return dict(y=s["y"])
    ws = s["ws"]
    f.copy(s["dx"], s["dy"], rows * w * 4)
    f.fp32_to_fp16(s["g"], s["dy"], rows * w)
    f.gemm_tn(s["dw_proj"], s["g"], s["attn"], w, w, rows, workspace=ws)
    f.bias_gradient(s["db_proj"], s["g"], rows, w, workspace=ws)
    f.gemm_nn(s["dattn"], s["g"], s["w_proj"], rows, w, w)
    f.heads_split(s["do"], s["dattn"], S, T, H, hw, w, 0)
    if case["fused"]:
        f.attention_backward(s["dq"], s["dk"], s["dv"], s["do"], s["q"], s["k"], s["v"], s["o"],
                             s["lse"], nb, T, hw, scale, workspace=ws)
    else:
        f.gemm_tn_batched(s["dv"], s["p"], s["do"], nb, T, hw, T)
        f.gemm_nt_batched(s["ds"], s["do"], s["v"], nb, T, T, hw, 1.0)
        f.causal_softmax_backward(s["ds"], s["p"], s["ds"], nb, T, scale)
        f.gemm_nn_batched(s["dq"], s["ds"], s["k"], nb, T, hw, T)
        f.gemm_tn_batched(s["dk"], s["ds"], s["q"], nb, T, hw, T)
    for j, part in enumerate(("dq", "dk", "dv")):
        f.heads_merge(s["dqkv"], s[part], S, T, H, hw, 3 * w, j * w)
    f.gemm_tn(s["dw_qkv"], s["dqkv"], s["h"], 3 * w, w, rows, workspace=ws)
    f.bias_gradient(s["db_qkv"], s["dqkv"], rows, 3 * w, workspace=ws)
    f.gemm_nn(s["dh"], s["dqkv"], s["w_qkv"], rows, w, 3 * w)
    f.layernorm_backward(s["dx"], s["dgamma"], s["dbeta"], s["dh"], s["x"], s["mean"], s["rstd"],
                         s["gamma"], rows, w, accumulate_dx=True, workspace=ws)
    return {k: s[k] for k in ("y", "dx", "dw_qkv", "db_qkv", "dw_proj", "db_proj", "dgamma",
                              "dbeta")}


def _causal64(q, k, v):
    """Causal attention of [..., length, head width] in float64."""
    T = q.shape[-2]
    s = torch.matmul(q, k.transpose(-1, -2).contiguous()) / math.sqrt(q.shape[-1])
    mask = torch.triu(torch.ones(T, T, dtype=torch.bool, device=q.device), 1)
    return torch.matmul(torch.softmax(s.masked_fill(mask, float("-inf")), -1), v)


def _attention64(x, gamma, beta, w_qkv, b_qkv, w_proj, b_proj, S, T, H):
    rows, w = x.shape
    qkv = _norm64(x, gamma, beta) @ w_qkv.T + b_qkv
    q, k, v = (t.reshape(S, T, H, w // H).transpose(1, 2).contiguous()
               for t in qkv.split(w, dim=-1))
    o = _causal64(q, k, v).transpose(1, 2).reshape(rows, w)
    return x + (o @ w_proj.T + b_proj)


def _attention_exact(case, s):
    names = ("x", "gamma", "beta", "w_qkv", "b_qkv", "w_proj", "b_proj")
    p = {n: _leaf(s[n]) for n in names}
    y = _attention64(*(p[n] for n in names), case["sequences"], case["length"], case["heads"])
    out = dict(y=y.detach())
    if case["train"]:
        y.backward(s["dy"].double())
        out.update({"d" + n: p[n].grad for n in names})
    return out


def _attention_work(case):
    S, T, H, hw = case["sequences"], case["length"], case["heads"], case["head_width"]
    m, w = S * T, H * hw
    gemm = 2 * m * w * 4 * w                           # qkv and projection
    core = 2 * S * H * hw * T * (T + 1) // 2           # one causal product
    if not case["train"]:
        return dict(flops=gemm + 2 * core, bytes=m * w * 8 + 4 * w * w * 2)
    return dict(flops=3 * gemm + 6 * core, bytes=m * w * 16 + 4 * w * w * (2 + 4))


# -------------------------------------------------------------------- head
def _loss_scale(rows):
    return 1024.0 / rows


def _head_inputs(f, case, mk):
    rows, w, V, PV = case["tokens"], case["width"], case["vocab"], case["padded_vocab"]
    s = dict(h=mk.normal((rows, w), dtype=torch.float16), wte=mk.weight(PV, w, 0.05),
             targets=mk.tokens(rows, V))
    s["wte"][V:] = 0
    s.update(logits=_half(rows, PV), dlogits=_half(rows, PV), loss=_single(rows))
    if case["train"]:
        s.update(dwte=_single(PV, w), dh=_half(rows, w), ws=_bytes(f.gemm_tn_workspace(PV, w, rows)))
    return s


def _head_run(f, case, s):
    rows, w, V, PV = case["tokens"], case["width"], case["vocab"], case["padded_vocab"]
    f.gemm_nt(s["logits"], s["h"], s["wte"], rows, PV, w)
    f.softmax_cross_entropy(s["dlogits"], s["loss"], s["logits"], s["targets"], _loss_scale(rows),
                            rows, V, PV)
    out = {k: s[k] for k in ("logits", "dlogits", "loss")}
    if case["train"]:
        f.gemm_tn(s["dwte"], s["dlogits"], s["h"], PV, w, rows, workspace=s["ws"])
        f.gemm_nn(s["dh"], s["dlogits"], s["wte"], rows, w, PV)
        out.update(dwte=s["dwte"], dh=s["dh"])
    return out


def _cross_entropy64(logits, targets, vocab, scale):
    """(row losses, dlogits over every column) in float64."""
    ls = torch.log_softmax(logits[:, :vocab], -1)
    rows = torch.arange(len(targets), device=logits.device)
    loss = -ls[rows, targets]
    d = torch.zeros_like(logits)
    d[:, :vocab] = ls.exp_()
    d[rows, targets] -= 1.0
    return loss, d.mul_(scale)


def _head_exact(case, s):
    h, wte = s["h"].double(), s["wte"].double()
    logits = h @ wte.T
    loss, d = _cross_entropy64(logits, _ids(s["targets"]), case["vocab"],
                               _loss_scale(case["tokens"]))
    out = dict(logits=logits, dlogits=d, loss=loss)
    if case["train"]:
        out.update(dwte=d.T.contiguous() @ h, dh=d @ wte)
    return out


def _head_work(case):
    m, w, PV = case["tokens"], case["width"], case["padded_vocab"]
    gemm = 2 * m * w * PV
    b = m * w * 2 + PV * w * 2 + m * PV * 4
    if not case["train"]:
        return dict(flops=gemm, bytes=b)
    return dict(flops=3 * gemm, bytes=b + PV * w * 4 + m * w * 2)


# --------------------------------------------------------------- embedding
def _embedding_inputs(f, case, mk):
    S, T, V, w = case["sequences"], case["length"], case["vocab"], case["width"]
    s = dict(tokens=mk.tokens(S * T, V), wte=mk.normal((V, w), 0.05), wpe=mk.normal((T, w), 0.02),
             x=_single(S * T, w))
    if case["train"]:
        s.update(dx=mk.normal((S * T, w), 0.05), dwte=mk.normal((V, w), 0.05), dwpe=_single(T, w),
                 ws=_bytes(f.embedding_backward_workspace(S, T, V, w)))
    return s


def _embedding_run(f, case, s):
    S, T, V, w = case["sequences"], case["length"], case["vocab"], case["width"]
    f.embedding_forward(s["x"], s["tokens"], s["wte"], s["wpe"], S, T, V, w)
    if not case["train"]:
        return dict(x=s["x"])
    f.embedding_backward(s["dwte"], s["dwpe"], s["dx"], s["tokens"], S, T, V, w,
                         accumulate_wte=True, workspace=s["ws"])
    return {k: s[k] for k in ("x", "dwte", "dwpe")}


def _embedding_exact(case, s):
    S, T, w = case["sequences"], case["length"], case["width"]
    ids = _ids(s["tokens"])
    x = s["wte"].double()[ids] + s["wpe"].double().repeat(S, 1)
    if not case["train"]:
        return dict(x=x)
    dx = s["dx"].double()
    return dict(x=x, dwte=s["dwte"].double().index_add_(0, ids, dx),
                dwpe=dx.reshape(S, T, w).sum(0))


def _embedding_work(case):
    S, T, w = case["sequences"], case["length"], case["width"]
    b = S * T * w * 8 + T * w * 4 + S * T * 2
    if case["train"]:
        # Each distinct token's row is read and written once; text-like tokens
        # repeat, about one row in three is distinct at these sizes.
        b += S * T * w * 4 + T * w * 4 + min(case["vocab"], S * T // 3 + 1) * w * 8
    return dict(flops=0, bytes=b)


# ------------------------------------------------------------------- adamw
ADAMW_TENSORS_RETURNED = ("param", "exp_avg", "exp_avg_sq", "param_half")


def _parameter_sizes(case):
    """(values, has two dimensions) of a model's tensors, in its order."""
    w = case["width"]
    out = [(case["padded_vocab"] * w, True), (case["block_size"] * w, True)]
    for _ in range(case["layers"]):
        out += [(w, False), (w, False), (3 * w * w, True), (3 * w, False), (w * w, True), (w, False),
                (w, False), (w, False), (4 * w * w, True), (4 * w, False), (4 * w * w, True),
                (w, False)]
    return out + [(w, False), (w, False)]


def _adamw_inputs(f, case, mk):
    sizes = _parameter_sizes(case)
    total = sum(n for n, _ in sizes)
    # A trainer keeps each kind of state in one flat buffer, tensors in order.
    flat = dict(param=mk.normal((total,), 0.02), grad=mk.normal((total,), 0.3),
                exp_avg=mk.normal((total,), 1e-4), exp_avg_sq=mk.normal((total,), 1e-4).square_(),
                param_half=_half(total))
    tensors, at = [], 0
    for n, matrix in sizes:
        tensors.append(dict({k: t[at:at + n] for k, t in flat.items()}, count=n,
                            weight_decay=0.1 if matrix else 0.0))
        at += n
    state = torch.zeros(8, dtype=torch.int32, device="cuda")
    f.train_state_init(state, 1024.0)
    state[2] = 100          # steps taken: mid-training bias corrections
    return dict(flat, tensors=tensors, sizes=sizes, state=state, options=f.adamw_defaults(),
                ws=_bytes(f.adamw_workspace(tensors)))


def _adamw_run(f, case, s):
    f.adamw_step(s["tensors"], s["state"], s["options"], s["ws"])
    return {k: s[k] for k in ADAMW_TENSORS_RETURNED}


def _adamw_exact(case, s):
    o = s["options"]
    lr, b1, b2 = float(o.lr), float(o.beta1), float(o.beta2)
    step = int(s["state"][2]) + 1
    g = s["grad"].double() / 1024.0
    g *= min(1.0, float(o.max_grad_norm) / (float(torch.linalg.vector_norm(g)) + 1e-6))
    decay = torch.cat([torch.full((n,), 0.1 if matrix else 0.0, dtype=torch.float32, device="cuda")
                       for n, matrix in s["sizes"]])
    p = s["param"].double() * (1.0 - lr * decay.double())
    m = s["exp_avg"].double()
    m += (1.0 - b1) * (g - m)
    v = b2 * s["exp_avg_sq"].double() + (1.0 - b2) * g * g
    denom = v.sqrt() / math.sqrt(1.0 - b2 ** step) + float(o.eps)
    p -= (lr / (1.0 - b1 ** step)) * m / denom
    return dict(param=p, exp_avg=m, exp_avg_sq=v, param_half=p)


def _adamw_work(case):
    n = sum(size for size, _ in _parameter_sizes(case))
    # Gradient, weight and both moments read; weight, moments and FP16 copy
    # written.
    return dict(flops=0, bytes=n * (4 * 4 + 3 * 4 + 2))


# ------------------------------------------------------------------- model
def _model_inputs(f, case, mk):
    S, T, w = case["sequences"], case["length"], case["width"]
    m = _Model(f, case["layers"], case["heads"], w, case["block_size"], case["vocab"],
               case["padded_vocab"], S, T, backward=case["train"], fused=case["fused"])
    params = []
    for name, address, rows, cols in m.parameters():
        if "ln_" in name and name.endswith("weight"):
            t = mk.normal((rows, cols), 0.1, 1.0)
        elif rows == 1:
            t = mk.normal((rows, cols), 0.02)
        else:
            std = 0.02 / math.sqrt(2 * case["layers"]) if name.endswith("c_proj.weight") else 0.02
            t = mk.normal((rows, cols), std).half().float()   # the FP16 copies hold the same
            if name == "wte.weight":
                t[case["vocab"]:] = 0
        view = m.view(address, (rows, cols), "<f4")
        view.copy_(t)
        params.append((name, view))
    m.sync_weights()
    s = dict(model=m, params=params, tokens=mk.tokens(S * T, case["vocab"]),
             targets=mk.tokens(S * T, case["vocab"]))
    logits, dlogits, loss = m.outputs()
    out = dict(logits=m.view(logits, (S * T, case["padded_vocab"]), "<f2"),
               dlogits=m.view(dlogits, (S * T, case["padded_vocab"]), "<f2"),
               loss=m.view(loss, (S * T,), "<f4"))
    if case["train"]:
        for name, (address, count) in _gradient_blocks(m).items():
            out["d" + name] = m.view(address, (count,), "<f4")
    s["out"] = out
    return s


def _block_of(name):
    """A tensor's block: its layer, or its own name outside the layers."""
    return ".".join(name.split(".")[:2]) if name.startswith("blocks.") else name


def _gradient_blocks(m):
    """block -> (address, values): a layer's gradients lie one after the other."""
    blocks = {}
    for name, address, rows, cols in m.gradients():
        block = _block_of(name)
        first, count = blocks.get(block, (address, 0))
        if address != first + 4 * count:
            raise RuntimeError(f"{name} does not follow the gradient before it")
        blocks[block] = (first, count + rows * cols)
    return blocks


def _model_run(f, case, s):
    m = s["model"]
    m.forward(s["tokens"], s["targets"], _loss_scale(case["sequences"] * case["length"]))
    if case["train"]:
        m.backward(s["tokens"])
    return s["out"]


def _model_exact(case, s):
    S, T, H, V = case["sequences"], case["length"], case["heads"], case["vocab"]
    p = {name: t.double().requires_grad_(case["train"]) for name, t in s["params"]}
    ids, targets = _ids(s["tokens"]), _ids(s["targets"])

    def vec(name):
        return p[name].reshape(-1)

    with torch.set_grad_enabled(case["train"]):
        x = p["wte.weight"][ids] + p["wpe.weight"][:T].repeat(S, 1)
        for i in range(case["layers"]):
            b = f"blocks.{i}."
            x = _attention64(x, vec(b + "ln_1.weight"), vec(b + "ln_1.bias"),
                             p[b + "attn.c_attn.weight"], vec(b + "attn.c_attn.bias"),
                             p[b + "attn.c_proj.weight"], vec(b + "attn.c_proj.bias"), S, T, H)
            h = _norm64(x, vec(b + "ln_2.weight"), vec(b + "ln_2.bias"))
            u = _gelu64(h @ p[b + "mlp.c_fc.weight"].T + vec(b + "mlp.c_fc.bias"))
            x = x + (u @ p[b + "mlp.c_proj.weight"].T + vec(b + "mlp.c_proj.bias"))
        h = _norm64(x, vec("ln_f.weight"), vec("ln_f.bias"))
        logits = h @ p["wte.weight"].T
    loss, d = _cross_entropy64(logits.detach(), targets, V, _loss_scale(S * T))
    out = dict(logits=logits.detach(), dlogits=d, loss=loss)
    if case["train"]:
        logits.backward(d)
        blocks = {}
        for name, _ in s["params"]:
            blocks.setdefault("d" + _block_of(name), []).append(p[name].grad.reshape(-1))
        out.update({n: torch.cat(t) for n, t in blocks.items()})
    return out


def _model_work(case):
    L, S, T, H, w = (case[k] for k in ("layers", "sequences", "length", "heads", "width"))
    m, PV = S * T, case["padded_vocab"]
    gemm = L * 2 * m * 12 * w * w + 2 * m * w * PV
    core = L * 2 * S * H * (w // H) * T * (T + 1) // 2
    n = sum(size for size, _ in _parameter_sizes(case))
    b = n * 2 + m * PV * 4
    if not case["train"]:
        return dict(flops=gemm + 2 * core, bytes=b)
    return dict(flops=3 * gemm + 6 * core, bytes=b + n * 4)


_PREPARE = dict(mlp=_mlp_inputs, attention=_attention_inputs, head=_head_inputs,
                embedding=_embedding_inputs, adamw=_adamw_inputs, model=_model_inputs)
_RUN = dict(mlp=_mlp_run, attention=_attention_run, head=_head_run, embedding=_embedding_run,
            adamw=_adamw_run, model=_model_run)
_EXACT = dict(mlp=_mlp_exact, attention=_attention_exact, head=_head_exact,
              embedding=_embedding_exact, adamw=_adamw_exact, model=_model_exact)
_WORK = dict(mlp=_mlp_work, attention=_attention_work, head=_head_work,
             embedding=_embedding_work, adamw=_adamw_work, model=_model_work)


def work(case):
    return _WORK[case["kind"]](case)


def exact(case, seed):
    return _EXACT[case["kind"]](case, prepare(case, seed))


# Relative errors (2-norm) between correct implementations. Sums in another
# order move an FP16-storing block's outputs by up to 4e-7 where no FP16 value
# flips; against 64 bits the FP16 intermediates leave up to 4.7e-4 (mlp, head)
# and 1.0e-3 (attention, through P and dS), and the fused and the stored
# attention differ by 8.5e-4 through a 12-layer model. The embedding's and the
# optimizer's FP32 results are within 4e-8 of 64 bits; the optimizer's FP16
# copies of them differ where a last-bit change crosses a rounding boundary.
_TOLERANCE = dict(mlp=1e-3, head=1e-3, attention=2e-3, model=3e-3, embedding=1e-6, adamw=2e-5)


def tolerance(case):
    return {"rel": _TOLERANCE[case["kind"]]}
