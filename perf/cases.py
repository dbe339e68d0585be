"""What the speed of this framework is measured on: whole ``optimizer.step()`` calls.

A case is one optimizer class on the parameter list of one network, in the middle of a training run: parameters
and gradients of real magnitudes on the GPU, accumulators that several steps have filled.  One pass is one
``step()``, which is all that a training loop calls.  The networks are those of this repository's benchmark and
tests (a small MLP classifier, GPT-2-small, ViT-B/16, ResNet-50, Llama-1.1B, three thousand odd tensors next to
one embedding); ``draw`` varies their widths, depths, vocabularies, storage types and options.

Parameters, gradients and every kind of accumulator each lie in one flat buffer with 512-byte aligned slots (what
separate allocations would give them), so that a pass returns everything it has updated as a handful of tensors.
"""

import math
import random

import torch

from pylo_amd import CELO2_CUDA, ELO_CELO2_CUDA, ELO_CUDA, AdafacLO_CUDA, VeLO_CUDA
from pylo_amd.models import CELO2MLP, MetaMLP, VeLOMLP, VeLORNN

_ALIGN = 128          # elements between slot boundaries of a flat buffer: 512 bytes of fp32


# ---------------------------------------------------------------------------------------------- networks
def _mlp(case):
    """Linear layers of ``width`` hidden units with biases, (out, in) as torch.nn.Linear keeps them."""
    dims = [case["inputs"]] + [case["width"]] * (case["layers"] - 1) + [case["outputs"]]
    out = []
    for a, b in zip(dims[:-1], dims[1:]):
        out += [(b, a), (b,)]
    return out, []


def _gpt(case):
    """Decoder: token and position embedding, per layer two norms of two vectors, qkv, proj and the two ffn matrices."""
    d, f = case["width"], case["ffn"]
    shapes = [(case["vocab"], d), (case["context"], d)]
    for _ in range(case["layers"]):
        shapes += [(d,), (d,), (d, 3 * d), (d, d), (d,), (d,), (d, f), (f, d)]
    return shapes, [0, 1]


def _vit(case):
    """Image transformer: patch embedding (a 16 x 16 convolution), class token, positions, layers as above, head."""
    d, f = case["width"], case["ffn"]
    shapes = [(d, 3, 16, 16), (1, 1, d), (case["context"], d)]
    for _ in range(case["layers"]):
        shapes += [(d,), (d,), (d, 3 * d), (d, d), (d,), (d,), (d, f), (f, d)]
    return shapes + [(d, case["outputs"])], []


def _llama(case):
    """Decoder with grouped-query attention and a gated ffn: q, k, v, o, gate, up, down, one vector per norm."""
    d, f, kv = case["width"], case["ffn"], case["kv"]
    shapes = [(case["vocab"], d)]
    for _ in range(case["layers"]):
        shapes += [(d,), (d, d), (d, kv), (d, kv), (d, d), (d,), (d, f), (d, f), (f, d)]
    return shapes + [(case["vocab"], d)], [0, len(shapes)]


def _resnet(case):
    """Bottleneck residual network: 7 x 7 stem, stages of 1 x 1, 3 x 3, 1 x 1 kernels with norms, one matrix at the end."""
    w = case["width"]
    shapes, inp = [(w, 3, 7, 7), (w,), (w,)], w
    for k, blocks in enumerate((3, 4, 6, 3) if case["layers"] == 50 else (case["layers"],) * 4):
        p = w << k
        for b in range(blocks):
            shapes += [(p, inp, 1, 1), (p,), (p,), (p, p, 3, 3), (p,), (p,), (4 * p, p, 1, 1), (4 * p,), (4 * p,)]
            if b == 0:
                shapes += [(4 * p, inp, 1, 1), (4 * p,), (4 * p,)]
            inp = 4 * p
    return shapes + [(case["outputs"], inp), (case["outputs"],)], []


def _many(case):
    """``count`` tensors of 1 .. ``most`` elements, drawn over the logarithm, vectors and odd matrices mixed, and one
    embedding (rows x width)."""
    rng = random.Random(case["shapes_seed"])
    shapes = [(37, case["most"] // 16 + 3), (case["most"] // 16 + 3, 37)]
    while len(shapes) < case["count"]:
        n = max(1, int(math.exp(rng.random() * math.log(case["most"]))))
        if rng.random() < 0.4:
            shapes.append((n,))
        else:
            r = max(1, int(math.exp(rng.random() * math.log(n))))
            shapes.append((r, max(1, n // r)))
    return shapes + [(case["vocab"], case["width"])], [len(shapes)]


_NETS = {"mlp": _mlp, "gpt": _gpt, "vit": _vit, "llama": _llama, "resnet": _resnet, "many": _many}
_TYPES = {"float32": torch.float32, "bfloat16": torch.bfloat16, "float16": torch.float16}


def _shapes(case):
    return _NETS[case["net"]](case)


def _is_celo2(case):
    return case["optimizer"] in ("ELO_CELO2", "CELO2")


# ------------------------------------------------------------------------------------------------- cases
_GPT2S = {"net": "gpt", "layers": 12, "width": 768, "ffn": 3072, "vocab": 50257, "context": 1024}
_VITB16 = {"net": "vit", "layers": 12, "width": 768, "ffn": 3072, "context": 197, "outputs": 1000}
_RESNET50 = {"net": "resnet", "layers": 50, "width": 64, "outputs": 1000}
_LLAMA = {"net": "llama", "layers": 22, "width": 2048, "kv": 256, "ffn": 5632, "vocab": 32000}
_MLP = {"net": "mlp", "layers": 3, "inputs": 784, "width": 128, "outputs": 10}
_MANY = {"net": "many", "count": 3000, "most": 65536, "shapes_seed": 11, "vocab": 32000, "width": 4096}


def _case(name, optimizer, net, dtype="float32", clip=0.0, weight_decay=0.0, embedding_adamw=False):
    c = {"name": name, "optimizer": optimizer, **net, "dtype": dtype, "clip": clip, "weight_decay": weight_decay,
         "embedding_adamw": embedding_adamw}
    if name is None:
        del c["name"]
    return c


def listed():
    return [
        # a small classifier, as in a first experiment or a meta-training inner loop: latency and launches
        _case("elo_celo2_mlp", "ELO_CELO2", _MLP, clip=1.0, weight_decay=0.1),
        # the headline configuration: every matrix orthogonalised, global-norm clipping, weight decay
        _case("elo_celo2_gpt2s", "ELO_CELO2", _GPT2S, clip=1.0, weight_decay=0.1),
        # the same network trained with parameters and gradients stored in bfloat16
        _case("elo_celo2_gpt2s_bf16", "ELO_CELO2", _GPT2S, dtype="bfloat16", clip=1.0, weight_decay=0.1),
        # a convolutional network: kernels finished slice by slice, with CELO2's own AdamW and no clipping
        _case("celo2_resnet50", "CELO2", _RESNET50),
        # three thousand small odd tensors, the embedding on AdamW as a user would route it
        _case("elo_celo2_many", "ELO_CELO2", _MANY, clip=1.0, weight_decay=0.1, embedding_adamw=True),
        # the small classifier under VeLO: the LSTM and a chain of small launches
        _case("velo_mlp", "VeLO", _MLP),
        # VeLO's configuration, stored in fp32 and in bfloat16
        _case("velo_vitb16", "VeLO", _VITB16),
        _case("velo_vitb16_bf16", "VeLO", _VITB16, dtype="bfloat16"),
        # VeLO over many tensors: an LSTM row and a mixed network for each of them
        _case("velo_many", "VeLO", _MANY),
        # the small classifier under ELO with clipping and weight decay
        _case("elo_mlp", "ELO", _MLP, clip=1.0, weight_decay=0.01),
        # AdafacLO's configuration, the largest parameter set, and a convolutional network
        _case("adafac_llama1b", "AdafacLO", _LLAMA),
        _case("adafac_resnet50", "AdafacLO", _RESNET50),
    ]


def _logint(rng, lo, hi, multiple=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(multiple, int(round(v / multiple)) * multiple)


def draw(rng):
    """A network of one of the families above with its width, depth and the rest drawn over the range from the small
    classifier to Llama-1.1B, under one of the five classes."""
    while True:
        kind = rng.choice(("mlp", "gpt", "vit", "llama", "resnet", "many"))
        optimizer = rng.choice(("ELO_CELO2", "ELO_CELO2", "CELO2", "VeLO", "VeLO", "AdafacLO", "AdafacLO", "ELO"))
        # widths in earnest are multiples of the head size, mostly; a fifth of the draws are not
        step = rng.choice((64, 64, 64, 16, 1))
        width = _logint(rng, 64, 2048, step)
        layers = _logint(rng, 1, 24)
        if kind == "mlp":
            net = {"net": kind, "layers": rng.randint(2, 6), "inputs": _logint(rng, 2, 4096), "width": _logint(rng, 8, 4096),
                   "outputs": _logint(rng, 1, 1000)}
        elif kind == "gpt":
            net = {"net": kind, "layers": layers, "width": width, "ffn": 4 * width, "vocab": _logint(rng, 256, 50304),
                   "context": _logint(rng, 128, 4096, 128)}
        elif kind == "vit":
            net = {"net": kind, "layers": layers, "width": width, "ffn": 4 * width, "context": rng.choice((50, 197, 257)),
                   "outputs": _logint(rng, 10, 1000)}
        elif kind == "llama":
            net = {"net": kind, "layers": layers, "width": width, "kv": max(1, width // rng.choice((1, 4, 8))),
                   "ffn": _logint(rng, 2.5 * width, 3 * width, 16), "vocab": _logint(rng, 1000, 50304)}
        elif kind == "resnet":
            net = {"net": kind, "layers": rng.choice((1, 2, 3, 50)), "width": rng.choice((16, 24, 32, 48, 64, 96)),
                   "outputs": rng.choice((10, 100, 365, 1000))}
        else:
            net = {"net": kind, "count": _logint(rng, 50, 3000), "most": _logint(rng, 256, 65536),
                   "shapes_seed": rng.randint(0, 10 ** 6), "vocab": _logint(rng, 1000, 32000),
                   "width": _logint(rng, 64, 2048)}
        clip = rng.choice((0.0, 1.0)) if optimizer != "VeLO" else 0.0
        c = _case(None, optimizer, net, dtype=rng.choice(("float32",) * 7 + ("bfloat16", "bfloat16", "float16")), clip=clip,
                  weight_decay=rng.choice((0.0, 0.01, 0.1)), embedding_adamw=optimizer in ("ELO_CELO2", "CELO2") and rng.random() < 0.5)
        n = sum(math.prod(s) for s in _shapes(c)[0])
        most = 1.1e9 if optimizer in ("AdafacLO", "ELO") else 4e8
        if n <= most and work(c)["flops"] <= (4e12 if not _is_celo2(c) else 2e12):
            return c


# ---------------------------------------------------------------------------------------------- one pass
def _flat(shapes):
    """Slot offsets in a flat buffer and its length."""
    offs, at = [], 0
    for s in shapes:
        offs.append(at)
        at += -(-max(1, math.prod(s)) // _ALIGN) * _ALIGN
    return offs, at


def _optimizer(case, params, embeddings):
    wd, clip = case["weight_decay"], case["clip"]
    torch.manual_seed(1)           # the meta-networks' weights: the same for every seed of the inputs
    if _is_celo2(case):
        groups = [{"params": params}]
        if case["embedding_adamw"] and embeddings:
            groups = [{"params": [p for i, p in enumerate(params) if i not in embeddings]},
                      {"params": [params[i] for i in embeddings], "is_embedding": True}]
        cls = ELO_CELO2_CUDA if case["optimizer"] == "ELO_CELO2" else CELO2_CUDA
        return cls(groups, lr=3.16e-4, weight_decay=wd, clip_grad=clip > 0, clip_norm=clip or 1.0,
                   network=CELO2MLP(), hf_key=None)
    if case["optimizer"] == "VeLO":
        return VeLO_CUDA(params, lr=1.0, num_steps=10000, weight_decay=wd, rnn=VeLORNN(), mlp=VeLOMLP())
    if case["optimizer"] == "ELO":
        return ELO_CUDA(params, lr=1e-3, weight_decay=wd, clip_grad=clip > 0, clip_norm=clip or 1.0,
                        network=MetaMLP(39, 32, 1), hf_key=None)
    return AdafacLO_CUDA(params, lr=1.0, weight_decay=wd, max_grad_norm=clip or None, network=MetaMLP(39, 32, 1))


def prepare(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    dtype = _TYPES[case["dtype"]]
    shapes, embeddings = _shapes(case)
    offs, total = _flat(shapes)
    gen = torch.Generator(device=dev).manual_seed(seed)
    rng = random.Random(seed)
    # parameters N(0, 0.02); gradients Gaussian, or heavy-tailed (Student's t with three degrees of freedom) on the
    # many-tensor sets, with a scale per tensor that is log-uniform in [1e-5, 1e-2]
    flat_p = torch.empty(total, device=dev).normal_(0.0, 0.02, generator=gen).to(dtype)
    slots = torch.tensor([b - a for a, b in zip(offs, offs[1:] + [total])], device=dev)
    scales = torch.tensor([10.0 ** rng.uniform(-5.0, -2.0) for _ in shapes], device=dev)
    flat_g = torch.empty(total, dtype=dtype, device=dev)

    def new_gradients():
        g = torch.randn(total, device=dev, generator=gen)
        if case["net"] == "many":
            chi = torch.zeros(total, device=dev)
            for _ in range(3):
                chi.addcmul_(*(torch.randn(total, device=dev, generator=gen),) * 2)
            g.mul_(chi.div_(3.0).rsqrt_())
        flat_g.copy_(g.mul_(torch.repeat_interleave(scales, slots, output_size=total)))

    def views(flat, lead=()):
        out = []
        for o, s in zip(offs, shapes):
            out.append(flat[o:o + math.prod(s)].view(tuple(lead) + tuple(s)))
        return out

    params = [torch.nn.Parameter(v) for v in views(flat_p)]
    for p, g in zip(params, views(flat_g)):
        p.grad = g
    opt = _optimizer(case, params, embeddings)
    state = {"opt": opt, "args": (torch.tensor(2.0, device=dev),) if case["optimizer"] == "VeLO" else ()}
    new_gradients()
    opt.step(*state["args"])       # the first step makes the accumulators
    out = {"params": flat_p}
    keys = sorted({k for p in params for k, t in opt.state[p].items() if torch.is_tensor(t) and t.is_cuda and t.numel()})
    for key in keys:
        rows = [(p, opt.state[p][key]) for p in params if torch.is_tensor(opt.state[p].get(key)) and opt.state[p][key].numel()]
        rows = [(p, t) for p, t in rows if not any(t is opt.state[p].get(k) for k in keys if k < key)]
        o, n = _flat([tuple(t.shape) for _, t in rows])
        flat = torch.zeros(n, device=dev, dtype=rows[0][1].dtype)
        for (p, t), at in zip(rows, o):
            v = flat[at:at + t.numel()].view(t.shape)
            v.copy_(t)
            for k in [k for k, u in opt.state[p].items() if u is t]:
                opt.state[p][k] = v
        out[key] = flat
    if case["optimizer"] == "VeLO":
        out["lstm_h"], out["lstm_c"] = opt.lstm_hidden_state
        out["loss_means"] = opt.loss_buffer["means"]
    for _ in range(2):             # two more steps on other gradients, then the gradients of the pass
        new_gradients()
        opt.step(*state["args"])
    new_gradients()
    state["out"] = out
    return state


def run(state):
    state["opt"].step(*state["args"])
    return state["out"]


# -------------------------------------------------------------------------------------- bytes, tolerances
def work(case):
    """Bytes: gradient, parameter and the four accumulators of an element (seven for a vector that keeps its own second
    moments) read once, parameter and accumulators written once, the row and column factors likewise.  Flops, in fp32:
    the per-element network, and Newton-Schulz as five iterations that take the symmetric products by halves and
    share the two products over the long dim between two iterations (3 Gram products, 3 updates, 11 m x m products)."""
    shapes, embeddings = _shapes(case)
    e = 4 if case["dtype"] == "float32" else 2
    nbytes = flops = 0.0
    celo2 = _is_celo2(case)
    per_elem = 2.0 * (252 if celo2 else 106 if case["optimizer"] == "VeLO" else 1600)
    for i, s in enumerate(shapes):
        n = math.prod(s)
        if celo2 and (len(s) < 2 or (case["embedding_adamw"] and i in embeddings)):
            nbytes += n * (3 * e + (32 if case["optimizer"] == "ELO_CELO2" else 16))
            flops += 20.0 * n
            continue
        flops += n * per_elem
        if len(s) < 2:
            nbytes += n * (3 * e + 56)
            continue
        a, b = sorted(s)[-2:]
        nbytes += n * (3 * e + 32) + 24.0 * (n // a + n // b)
        if celo2:
            m, k = sorted(s[-2:])
            flops += (n // (m * k)) * (9.0 * m * m * k + 11.0 * m ** 3)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Four times what was seen between implementations at the same precision after two passes: the default kernels
    against the fp32 matrix instructions with separate statistics passes, and against vector-pipe networks with one
    Gram product per iteration, over the listed cases and eight drawn ones.  Orthogonalised steps differed by 1.5e-7 of the
    parameters (9e-6 of a single one), the other classes by 5e-8 (5e-7); parameters stored in 16 bits by roundings that
    fall to the other side (two spacings of a single value, 3e-5 and 5e-6 over a set)."""
    if case["dtype"] == "bfloat16":
        return {"rel": 1.2e-4, "max": 6e-2}
    if case["dtype"] == "float16":
        return {"rel": 3e-5, "max": 6e-3}
    return {"rel": 6e-7, "max": 4e-5} if _is_celo2(case) else {"rel": 4e-7, "max": 4e-6}
