"""The work a program has this framework do, as cases that can be timed and checked: compiled functions over
the layers of a decoder (projections, norms, attention, MLP, vocabulary head) in inference and in training, a
whole decoder block with its gradients and a whole training step, over their range of sizes.

A case is compiled once per shape by ``lumen_amd.compile`` (as a program keeps its compiled functions), takes
device tensors and returns the outputs as torch views of the memory the compiled function wrote.
"""

import functools
import math

import torch

import lumen_amd as L
import lumen_amd.functional as F
from lumen_amd import native
from lumen_amd import workloads as W

DTYPES = {"float32": torch.float32, "bfloat16": torch.bfloat16, "float16": torch.float16, "int64": torch.int64}
NAMES = {v: k for k, v in DTYPES.items()}
LEARNING_RATE = 1.0  # of the training step: large enough for a step to move bfloat16 weights
INTERFACE = {"float32": "<f4", "bfloat16": "<i2", "float16": "<f2"}


def listed():
    return [
        # a small float32 dense layer (relu(x w), the float32 fold): the smallest call, latency and launches
        dict(name="linear_f32", kind="linear_f32", m=256, k=512, n=1024),
        # scale and shift, GELU, layer norm and softmax of activations: one fused elementwise/row chain
        dict(name="chain", kind="chain", rows=8192, cols=4096),
        # an RMS norm in training at the 12-layer step's size: forward, input and weight gradients
        dict(name="norm_train", kind="norm_train", rows=16384, cols=2048),
        # causal attention in training: forward and the three gradients
        dict(name="attn_train", kind="attn_train", b=8, sq=2048, sk=2048, n=16, nkv=16, d=128, causal=True,
             dtype="bfloat16"),
        # attention over a prompt of odd length with grouped key/value heads, head dim 64, float16 (prefill)
        dict(name="attn_prefill", kind="attn_fwd", b=2, sq=1777, sk=1777, n=16, nkv=4, d=64, causal=True,
             dtype="float16"),
        # one new token a sequence against a key/value cache (decode)
        dict(name="attn_decode", kind="attn_fwd", b=16, sq=1, sk=4096, n=16, nkv=16, d=128, causal=True,
             dtype="bfloat16"),
        # the 12-layer model's MLP over a whole batch of prompts (prefill)
        dict(name="mlp_prefill", kind="mlp", tokens=16384, dim=2048, ffn=8192),
        # the same MLP for one new token of each of 16 sequences (decode)
        dict(name="mlp_decode", kind="mlp", tokens=16, dim=2048, ffn=8192),
        # evaluation loss of the vocabulary head over the 12-layer model's batch: a loss a token, no gradients
        dict(name="head_loss", kind="head_loss", tokens=16384, dim=2048, vocab=32000),
        # the vocabulary head in training on a ragged batch: the mean loss and both gradients
        dict(name="head_train", kind="head_train", tokens=3000, dim=1024, vocab=32000),
        # one block of the 12-layer model in training, one sequence: output, input and weight gradients
        dict(name="block_train", kind="block_train", batch=1, seq=4096, dim=2048, heads=16, ffn=8192),
        # a whole training step of the 2-layer model: forward, backward and SGD, the loss and new weights
        dict(name="step", kind="step", batch=16, seq=512, dim=512, heads=8, ffn=2048, layers=2, vocab=32000),
    ]


# ---- drawn cases


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mult(rng, lo, hi, q):
    return max(q, _log(rng, lo, hi) // q * q)


def _draw(rng):
    kind = rng.choice(["linear_f32", "chain", "norm_train", "attn_train", "attn_prefill", "attn_decode", "mlp", "mlp",
                       "head_loss", "head_train", "block_train", "step"])
    if kind == "linear_f32":
        return dict(kind=kind, m=_log(rng, 1, 1024), k=_log(rng, 32, 2048), n=_log(rng, 32, 2048))
    if kind == "chain":
        cols = _log(rng, 128, 8192)
        return dict(kind=kind, rows=_log(rng, 1, 16384), cols=cols // 8 * 8 if rng.random() < 0.7 else cols)
    if kind == "norm_train":
        return dict(kind=kind, rows=_log(rng, 16, 16384), cols=_mult(rng, 256, 8192, 8))
    if kind.startswith("attn"):
        d = rng.choice([64, 64, 128, 128, 32, 96])
        n = rng.choice([4, 8, 16, 32])
        c = dict(kind="attn_train" if kind == "attn_train" else "attn_fwd", b=_log(rng, 1, 32), n=n,
                 nkv=n // rng.choice([1, 1, 4]), d=d, causal=True, dtype=rng.choice(["bfloat16", "float16"]))
        if kind == "attn_decode":
            c.update(sq=rng.choice([1, 1, 1, 4]), sk=_log(rng, 128, 32768))
        else:
            s = _log(rng, 33, 8192)
            c.update(sq=s, sk=s, causal=rng.random() < 0.75)
        return c
    if kind == "mlp":
        dim = _mult(rng, 256, 4096, 64)
        ffn = 4 * dim if rng.random() < 0.6 else _mult(rng, 512, 16384, 8)
        return dict(kind=kind, tokens=_log(rng, 1, 16384), dim=dim, ffn=ffn)
    if kind in ("head_loss", "head_train"):
        vocab = _log(rng, 1000, 64000)
        return dict(kind=kind, tokens=_log(rng, 16, 16384), dim=_mult(rng, 256, 2048, 64),
                    vocab=vocab // 64 * 64 if rng.random() < 0.7 else vocab)
    heads, hd = rng.choice([4, 8, 16]), rng.choice([64, 64, 128])
    c = dict(kind=kind, batch=_log(rng, 1, 8), seq=_log(rng, 65, 4096), dim=heads * hd, heads=heads, ffn=4 * heads * hd)
    if kind == "step":
        c.update(layers=rng.choice([1, 2, 3]), vocab=_mult(rng, 1000, 32000, 8))
    return c


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 300)


def draw(rng):
    """A case of the same kinds and ranges that costs no more than the largest listed one."""
    most = max(_cost(c) for c in listed())
    while True:
        c = _draw(rng)
        if _cost(c) <= most:
            return c


# ---- the programs


def _linear_f32(x, w):
    return [F.relu(F.matmul(x, w, "float32", "float32"))]


def _chain(x, a, b):
    t = F.layer_norm(F.gelu((x * a + b).float()), x.shape[-1])
    return [F.softmax(t, -1).bfloat16()]


def _norm(x, w):
    return F.rms_norm(x.float(), x.size(-1), w.float()).bfloat16()


def _norm_train(x, w, dy):
    y, pullback = L.vjp(_norm, x, w)
    return [y, *pullback(dy)]


def _attn_fwd(q, k, v, causal):
    return [F.flash_attention(q, k, v, is_causal=causal)]


def _attn_train(q, k, v, do, causal):
    o, pullback = L.vjp(lambda q, k, v: F.flash_attention(q, k, v, is_causal=causal), q, k, v)
    return [o, *pullback(do)]


def _mlp(x, w1, w2):
    h = F.gelu(F.matmul(x, w1.t(), "float32", "float32")).bfloat16()
    return [F.matmul(h, w2.t(), "float32", "bfloat16")]


def _head_loss(h, w, target):
    return [F.cross_entropy(F.matmul(h, w.t(), "float32", "float32"), target)]


def _head_train(h, w, target):
    def loss(h, w):
        return F.mean(F.cross_entropy(F.matmul(h, w.t(), "float32", "float32"), target))

    value, grads = L.value_and_grad(loss, (0, 1))(h, w)
    return [value, *grads]


def _block_train(block, x, dy, batch, heads):
    y = block(x, batch, heads)
    y.backward(dy)
    return [y, x.grad, *(p.grad for p in block.parameters())]


PROGRAMS = {"linear_f32": _linear_f32, "chain": _chain, "norm_train": _norm_train, "attn_fwd": _attn_fwd,
            "attn_train": _attn_train, "mlp": _mlp, "head_loss": _head_loss, "head_train": _head_train,
            "block_train": _block_train, "step": W.train_step}


@functools.lru_cache(maxsize=None)
def _program(kind):
    return L.compile(PROGRAMS[kind], device="hip")


def _config(case):
    return W.TransformerConfig(vocab=case.get("vocab", 8), dim=case["dim"], heads=case["heads"], ffn=case["ffn"],
                               seq=case["seq"], batch=case["batch"], layers=case.get("layers", 1))


@functools.lru_cache(maxsize=None)
def _model(cfg):
    return W.build(cfg, lr=LEARNING_RATE)


# ---- inputs


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, shape, dtype, std=1.0, mean=0.0):
    return (torch.randn(shape, generator=g, device="cuda") * std + mean).to(DTYPES[dtype])


def _inputs(case, seed):
    """The case's inputs as torch tensors on the GPU, from the seed alone."""
    g, kind = _generator(seed), case["kind"]
    bf = functools.partial(_normal, g, dtype="bfloat16")
    if kind == "linear_f32":
        return [_normal(g, (case["m"], case["k"]), "float32"), _normal(g, (case["k"], case["n"]), "float32")]
    if kind == "chain":
        c = case["cols"]
        return [bf((case["rows"], c)), bf((c,), std=0.1, mean=1.0), bf((c,), std=0.1)]
    if kind == "norm_train":
        r, c = case["rows"], case["cols"]
        return [bf((r, c)), bf((c,), std=0.1, mean=1.0), bf((r, c))]
    if kind in ("attn_fwd", "attn_train"):
        b, n, nkv, d, dt = case["b"], case["n"], case["nkv"], case["d"], case["dtype"]
        q = _normal(g, (b, case["sq"], n, d), dt)
        k, v = (_normal(g, (b, case["sk"], nkv, d), dt) for _ in range(2))
        return [q, k, v] + ([_normal(g, q.shape, dt)] if kind == "attn_train" else [])
    if kind == "mlp":
        t, d, f = case["tokens"], case["dim"], case["ffn"]
        return [bf((t, d)), bf((f, d), std=0.02), bf((d, f), std=0.02)]
    if kind in ("head_loss", "head_train"):
        t, d, v = case["tokens"], case["dim"], case["vocab"]
        target = torch.randint(0, v, (t,), generator=g, device="cuda")
        return [bf((t, d)), bf((v, d), std=0.02), target]
    tokens = case["batch"] * case["seq"]
    if kind == "block_train":
        return [bf((tokens, case["dim"])), bf((tokens, case["dim"]))]
    ids = torch.randint(0, case["vocab"], (case["batch"], case["seq"]), generator=g, device="cuda")
    return [ids, torch.roll(ids, -1, 1)]


def _weights(case):
    """The weights of a block or model (torch, by parameter path): the same for every seed, as the checkpoint
    that a program starts from; norm scales 1, the others N(0, 0.02)."""
    g = _generator(7)
    model = _modules(case)[0]
    return {path: torch.ones(p.shape, device="cuda", dtype=torch.bfloat16) if len(p.shape) == 1
            else _normal(g, p.shape, "bfloat16", std=0.02) for path, p in model.named_parameters()}


def _modules(case):
    model, opt = _model(_config(case))
    return (model.layers[0], None) if case["kind"] == "block_train" else (model, opt)


def _device(t):
    """A device tensor of the framework's with ``t``'s values."""
    out = L.empty(tuple(t.shape), NAMES[t.dtype], "hip")
    native.d2d(out.data_ptr(), t.data_ptr(), out.nbytes)
    return out


def _load(module, weights):
    """The weights into the module, from host memory as from a file."""
    host = {path: w.cpu().view(torch.int16).numpy().view("uint16") for path, w in weights.items()}
    module.load_state_dict({path: L.Tensor("bfloat16", a.shape, "cpu", host=a) for path, a in host.items()})


def prepare(case, seed):
    inputs = _inputs(case, seed)
    torch.cuda.synchronize()
    native.set_device(0)
    args = [_device(t) for t in inputs]
    native.sync()
    kind, weights = case["kind"], []
    if kind in ("attn_fwd", "attn_train"):
        args.append(case["causal"])
    if kind in ("block_train", "step"):
        module, opt = _modules(case)
        _load(module, _weights(case))
        if kind == "block_train":
            args = [module, *args, case["batch"], case["heads"]]
        else:
            args = [module, opt, *args]
            weights = module.parameters()
    return {"program": _program(kind), "args": args, "weights": weights, "views": {}}


class _Memory:
    """A device tensor's memory for torch, which keeps this object (and so the memory) as long as its view."""

    def __init__(self, t):
        self.tensor = t
        self.__cuda_array_interface__ = {"shape": tuple(t.shape), "typestr": INTERFACE[t.dtype],
                                         "data": (t.data_ptr(), False), "version": 2}


def _view(views, t):
    """``t`` as a torch tensor over the same memory (made once for each place an output is written)."""
    key = (t.data_ptr(), t.dtype, t.shape)
    v = views.get(key)
    if v is None:
        v = views[key] = torch.as_tensor(_Memory(t), device="cuda").view(DTYPES[t.dtype])
    return v


def run(state):
    out = state["program"](*state["args"])
    views = state["views"]
    if state["weights"]:  # a training step: its loss and the weights it updated
        return [_view(views, out)] + [_view(views, w._placed("hip:0")) for w in state["weights"]]
    return [_view(views, t) for t in out]


# ---- what a pass cannot do without


def _attn_flops(case, backward):
    sq, sk = case["sq"], case["sk"]
    pairs = sum(max(0, min(sk, i + 1 + sk - sq)) for i in range(sq)) if case["causal"] else sq * sk
    return case["b"] * case["n"] * pairs * case["d"] * (14 if backward else 4)


def _matrices(case):
    d, f = case["dim"], case["ffn"]
    return 4 * d * d + 2 * d * f


def work(case):
    kind = case["kind"]
    if kind == "linear_f32":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": 4 * (m * k + k * n + m * n), "flops": 2 * m * n * k}
    if kind == "chain":
        return {"bytes": 4 * case["rows"] * case["cols"] + 4 * case["cols"], "flops": 0}
    if kind == "norm_train":
        return {"bytes": 8 * case["rows"] * case["cols"] + 4 * case["cols"], "flops": 0}
    if kind in ("attn_fwd", "attn_train"):
        q = 2 * case["b"] * case["sq"] * case["n"] * case["d"]
        kv = 2 * case["b"] * case["sk"] * case["nkv"] * case["d"]
        train = kind == "attn_train"
        return {"bytes": 4 * q + 4 * kv if train else 2 * q + 2 * kv, "flops": _attn_flops(case, train)}
    if kind == "mlp":
        t, d, f = case["tokens"], case["dim"], case["ffn"]
        return {"bytes": 4 * t * d + 4 * d * f, "flops": 4 * t * d * f}
    if kind in ("head_loss", "head_train"):
        t, d, v = case["tokens"], case["dim"], case["vocab"]
        train = kind == "head_train"
        once = 2 * (t + v) * d
        return {"bytes": (2 * once if train else once) + 8 * t + (4 if train else 4 * t),
                "flops": (6 if train else 2) * t * d * v}
    tokens, layers = case["batch"] * case["seq"], case.get("layers", 1)
    attn = _attn_flops(dict(b=case["batch"], n=case["heads"], sq=case["seq"], sk=case["seq"],
                            d=case["dim"] // case["heads"], causal=True), True)
    flops = layers * (6 * tokens * _matrices(case) + attn)
    params = layers * _matrices(case)
    if kind == "block_train":
        return {"bytes": 4 * params + 8 * tokens * case["dim"], "flops": flops}
    table = case["vocab"] * case["dim"]
    return {"bytes": 4 * (params + 2 * table + case["seq"] * case["dim"]) + 16 * tokens,
            "flops": flops + 6 * tokens * table}


# ---- how far another correct implementation may be off


def tolerance(case):
    kind = case["kind"]
    if kind == "linear_f32":  # 32-bit sums of up to 2048 products: 4e-7 from 64 bits at 512
        return {"rel": 2e-6}
    if kind == "head_loss":  # float32 losses near 10 from 32-bit logits: 4e-8 from 64 bits
        return {"rel": 2e-6}
    if kind == "step":  # a weight's update rounds to another bfloat16 neighbour for about one value in a hundred
        return {"rel": 2e-3}
    if case.get("dtype") == "float16":  # 3e-4 from 64 bits
        return {"rel": 2e-3}
    return {"rel": 1e-2}  # bfloat16 results of bfloat16 intermediates: 2e-3 to 6e-3 from 64 bits


# ---- the same in 64 bits


def _gelu64(x):
    return 0.5 * x * (1 + torch.tanh(0.7978845608 * (x + 0.044715 * x * x * x)))


def _rms64(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 2.0**-23) * w


def _attn64(q, k, v, causal):
    """Attention of [B, S, N, H] float64 operands, a sequence and a group of heads at a time."""
    b, sq, n, d = q.shape
    sk, nkv = k.shape[1], k.shape[2]
    hidden = None
    if causal:
        hidden = torch.ones(sq, sk, dtype=torch.bool, device=q.device).triu(1 + sk - sq)
    outs = []
    for i in range(b):
        heads = []
        for h in range(nkv):
            g = n // nkv
            qs = q[i, :, h * g:(h + 1) * g].permute(1, 0, 2).reshape(g * sq, d)
            s = (qs @ k[i, :, h].t().contiguous()).reshape(g, sq, sk) / math.sqrt(d)
            if hidden is not None:
                s = s.masked_fill(hidden, -math.inf)
            p = torch.softmax(s, -1).reshape(g * sq, sk)
            heads.append((p @ v[i, :, h].contiguous()).reshape(g, sq, v.shape[3]).permute(1, 0, 2))
        outs.append(torch.cat(heads, 1))
    return torch.stack(outs)


def _block64(x, w, batch, heads):
    t, d = x.shape
    h = _rms64(x, w["attn.norm"])
    q, k, v = ((h @ w[f"attn.{m}"].t()).reshape(batch, t // batch, heads, d // heads) for m in ("wq", "wk", "wv"))
    x = x + _attn64(q, k, v, True).reshape(t, d) @ w["attn.wo"].t()
    h = _rms64(x, w["mlp.norm"])
    return x + _gelu64(h @ w["mlp.w1"].t()) @ w["mlp.w2"].t()


def _nll64(logits, target):
    return torch.logsumexp(logits, -1) - logits.gather(1, target.reshape(-1, 1)).reshape(-1)


def exact(case, seed):
    w = work(case)
    if w["flops"] > 4e12:
        return None
    kind = case["kind"]
    x = [t.double() if t.is_floating_point() else t for t in _inputs(case, seed)]
    if kind == "linear_f32":
        return [torch.relu(x[0] @ x[1])]
    if kind == "chain":
        t = _gelu64(x[0] * x[1] + x[2])
        t = t - t.mean(-1, keepdim=True)
        return [torch.softmax(t / torch.sqrt((t * t).mean(-1, keepdim=True) + 1e-5), -1)]
    if kind == "attn_fwd":
        return [_attn64(*x, case["causal"])]
    if kind == "mlp":
        return [_gelu64(x[0] @ x[1].t()) @ x[2].t()]
    if kind == "head_loss":
        return [_nll64(x[0] @ x[1].t(), x[2])]
    if kind in ("norm_train", "attn_train"):
        leaves = [t.requires_grad_() for t in (x[:2] if kind == "norm_train" else x[:3])]
        y = _rms64(*leaves) if kind == "norm_train" else _attn64(*leaves, case["causal"])
        return [y.detach(), *torch.autograd.grad(y, leaves, x[-1])]
    if kind == "head_train":
        leaves = [t.requires_grad_() for t in x[:2]]
        loss = _nll64(leaves[0] @ leaves[1].t(), x[2]).mean()
        return [loss.detach(), *torch.autograd.grad(loss, leaves)]
    weights = {path: t.double().requires_grad_() for path, t in _weights(case).items()}
    if kind == "block_train":
        leaves = [x[0].requires_grad_(), *weights.values()]
        y = _block64(x[0], weights, case["batch"], case["heads"])
        return [y.detach(), *torch.autograd.grad(y, leaves, x[1])]
    ids, target = x
    h = (weights["embed.tokens"][ids] + weights["embed.positions"]).reshape(-1, case["dim"])
    for i in range(case["layers"]):
        own = {path.split(".", 2)[2]: t for path, t in weights.items() if path.startswith(f"layers.{i}.")}
        h = _block64(h, own, case["batch"], case["heads"])
    loss = _nll64(_rms64(h, weights["norm"]) @ weights["head"].t(), target.reshape(-1)).mean()
    grads = torch.autograd.grad(loss, list(weights.values()))
    return [loss.detach(), *(t.detach() - LEARNING_RATE * g for t, g in zip(weights.values(), grads))]
