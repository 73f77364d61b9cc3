"""Performance cases: what a program that uses this plugin has it do, over the range of sizes it is used for.

Every case is compiled and executed through the PJRT entry points of `jax_mps_amd.pjrt`, as a jitted program is:
the five programs of `jax_mps_amd.programs.configs` (MLP, embedding, ResNet18, DistilBERT-shaped encoder, LSTM) and
the fused elementwise / reduce operators that such programs are made of.  `prepare` uploads the inputs and compiles the
module once per shape; `run` is one execution (for the MLP a few train steps in a row) and hands the results out as
tensors that share the device buffers' memory.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from jax_mps_amd import pjrt, runner
from jax_mps_amd.programs import configs
from jax_mps_amd.programs.configs import Program
from jax_mps_amd.shlo.builder import Builder, gelu_tanh, layer_norm, softmax


def listed():
    return [
        # a small classifier trained step by step: a few launches per step, bound by their latency
        {"name": "mlp_train_b256", "family": "mlp", "batch": 256, "d_in": 784, "d_hidden": 512, "steps": 10},
        # token embedding of a language model, forward and dense gradient, frequencies as in text
        {"name": "embedding_50000x768", "family": "embedding", "vocab": 50000, "dim": 768, "n_idx": 8192},
        # a smaller table of odd width, as for categorical features
        {"name": "embedding_12345x300", "family": "embedding", "vocab": 12345, "dim": 300, "n_idx": 1500},
        # image classifier training at its usual batch size: forward, backward and optimizer, float32
        {"name": "resnet18_train_b128", "family": "resnet18", "batch": 128, "image": 32, "width": 64, "train": True},
        # the same network on a small batch of odd-sized images with channel counts that are no powers of two
        {"name": "resnet18_train_b24_odd", "family": "resnet18", "batch": 24, "image": 28, "width": 48, "train": True},
        # evaluation of a few images: the forward pass alone
        {"name": "resnet18_forward_b16", "family": "resnet18", "batch": 16, "image": 32, "width": 64, "train": False},
        # encoder inference on a full batch, bfloat16
        {"name": "encoder_bf16_b32_s128", "family": "distilbert", "batch": 32, "seq": 128, "layers": 6, "heads": 12, "head_dim": 64,
         "d_ff": 3072, "vocab": 30522, "dtype": "bf16"},
        # one request of a serving program: a single short sentence
        {"name": "encoder_bf16_b1_s37", "family": "distilbert", "batch": 1, "seq": 37, "layers": 6, "heads": 12, "head_dim": 64,
         "d_ff": 3072, "vocab": 30522, "dtype": "bf16"},
        # the same encoder in float32, as it is run where bfloat16 is not wanted
        {"name": "encoder_f32_b8_s128", "family": "distilbert", "batch": 8, "seq": 128, "layers": 6, "heads": 12, "head_dim": 64,
         "d_ff": 3072, "vocab": 30522, "dtype": "f32"},
        # recurrent network trained through a scan: 2 x 100 dependent loop iterations
        {"name": "lstm_train_s100_b64", "family": "lstm", "seq": 100, "batch": 64, "d_in": 128, "hidden": 256},
        # a shorter sequence with sizes that are no multiples of a tile
        {"name": "lstm_train_s45_b20_odd", "family": "lstm", "seq": 45, "batch": 20, "d_in": 50, "hidden": 200},
        # one bandwidth-bound operator by itself: a large softmax
        {"name": "softmax_10000x1000", "family": "op", "op": "softmax", "rows": 10000, "cols": 1000},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["mlp", "embedding", "resnet18", "distilbert", "distilbert", "lstm", "op"])
    if family == "mlp":
        return {"family": family, "batch": _log_int(rng, 8, 512), "d_in": _log_int(rng, 12, 1024), "d_hidden": _log_int(rng, 16, 1024), "steps": 10}
    if family == "embedding":
        return {"family": family, "vocab": _log_int(rng, 500, 50000), "dim": _log_int(rng, 8, 768), "n_idx": _log_int(rng, 32, 8192)}
    if family == "resnet18":
        return {"family": family, "batch": _log_int(rng, 8, 100), "image": rng.randint(16, 32), "width": rng.choice([8, 16, 24, 32, 48, 64]),
                "train": rng.random() < 0.7}
    if family == "distilbert":
        heads, head_dim = rng.randint(2, 12), rng.choice([32, 64])
        return {"family": family, "batch": _log_int(rng, 1, 32), "seq": rng.randint(8, 128), "layers": rng.randint(1, 6), "heads": heads,
                "head_dim": head_dim, "d_ff": heads * head_dim * rng.choice([2, 4]), "vocab": _log_int(rng, 300, 30522),
                "dtype": rng.choice(["bf16", "bf16", "f32"])}
    if family == "lstm":
        return {"family": family, "seq": rng.randint(10, 100), "batch": _log_int(rng, 4, 64), "d_in": _log_int(rng, 6, 128),
                "hidden": _log_int(rng, 16, 256)}
    return {"family": "op", "op": rng.choice(sorted(_OPS)), "rows": _log_int(rng, 100, 10000), "cols": _log_int(rng, 64, 1000)}


# ---------------------------------------------------------------------------------------------------------------------
# programs
# ---------------------------------------------------------------------------------------------------------------------
def _op_sum(b, rows, cols):
    return [b.reduce_sum(b.arg((rows * cols,), "f32"), [0])]


def _op_column_stats(b, rows, cols):
    x = b.arg((rows, cols), "f32")
    return [b.reduce_sum(x, [0]), b.reduce_sum(b.mul(x, x), [0])]


def _op_layernorm_bf16(b, rows, cols):
    return [layer_norm(b, b.arg((rows, cols), "bf16"), b.arg((cols,), "bf16"), b.arg((cols,), "bf16"), 1e-12)]


def _op_bias_gelu_bf16(b, rows, cols):
    x, t = b.arg((rows, cols), "bf16"), b.arg((cols,), "bf16")
    return [gelu_tanh(b, b.add(x, b.broadcast_in_dim(t, (rows, cols), [1])))]


_OPS = {
    "softmax": lambda b, rows, cols: [softmax(b, b.arg((rows, cols), "f32"), -1)],
    "exp": lambda b, rows, cols: [b.exp(b.arg((rows * cols,), "f32"))],
    "add": lambda b, rows, cols: [b.add(b.arg((rows * cols,), "f32"), b.arg((rows * cols,), "f32"))],
    "sum": _op_sum,
    "column_stats": _op_column_stats,
    "layernorm_bf16": _op_layernorm_bf16,
    "bias_gelu_bf16": _op_bias_gelu_bf16,
}


def _op_program(case, seed):
    b = Builder("jit_" + case["op"])
    b.ret(*_OPS[case["op"]](b, case["rows"], case["cols"]))
    rng = np.random.default_rng(seed)
    inputs = [rng.standard_normal(shape, dtype=np.float32) for shape, _ in b.arg_types]
    return Program(case["op"], b.text(), inputs, [], [], [d for _, d in b.arg_types], list(b.result_types))


def _key(case):
    return tuple(sorted((k, v) for k, v in case.items() if k != "name"))


@functools.lru_cache(maxsize=4)
def _embedding_module(key):
    c = dict(key)
    return configs.build_embedding(vocab=c["vocab"], dim=c["dim"], n_idx=c["n_idx"])


def _program(case, seed):
    """The case's module and its inputs: those of the repository's own builders, at the case's sizes."""
    f = case["family"]
    if f == "mlp":
        return configs.build_mlp(batch=case["batch"], d_in=case["d_in"], d_hidden=case["d_hidden"], seed=seed)
    if f == "embedding":
        p = _embedding_module(_key(case))
        rng = np.random.default_rng(seed)
        table = rng.standard_normal((case["vocab"], case["dim"]), dtype=np.float32) * np.float32(0.02)
        inputs = [table, configs.zipf_indices(rng, case["n_idx"], case["vocab"]),
                  rng.standard_normal((case["n_idx"], case["dim"]), dtype=np.float32)]
        return Program(p.name, p.text, inputs, p.input_names, p.output_names, p.input_dtypes, p.output_types, p.feedback, p.meta)
    if f == "resnet18":
        return configs.build_resnet18(batch=case["batch"], image=case["image"], width=case["width"], train=case["train"], seed=seed)
    if f == "distilbert":
        p = configs.build_distilbert(batch=case["batch"], seq=case["seq"], layers=case["layers"], d_model=case["heads"] * case["head_dim"],
                                     heads=case["heads"], d_ff=case["d_ff"], vocab=case["vocab"], seed=seed, dtype=case["dtype"])
        # sentences of different length, padded to the longest
        lengths = np.random.default_rng(seed + 1).integers(case["seq"] // 2, case["seq"] + 1, case["batch"])
        lengths[0] = case["seq"]
        p.inputs[-1] = (np.arange(case["seq"])[None, :] < lengths[:, None]).astype(np.int32)
        return p
    if f == "lstm":
        return configs.build_lstm(seq=case["seq"], batch=case["batch"], d_in=case["d_in"], hidden=case["hidden"], seed=seed)
    return _op_program(case, seed)


# ---------------------------------------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------------------------------------
_EXECUTABLES = {}      # a program compiles a module once and keeps it


def _executable(text):
    if text not in _EXECUTABLES:
        if len(_EXECUTABLES) >= 4:
            _EXECUTABLES.pop(next(iter(_EXECUTABLES)))
        _EXECUTABLES[text] = pjrt.get_client().compile_and_load(text)
    return _EXECUTABLES[text]


def prepare(case, seed):
    p = _program(case, seed)
    exe = _executable(p.text)
    names = p.output_names
    # a train step's new momenta are its gradients (the first step's exactly) and its loss; 64 results at most leave the program here
    wanted = [i for i, n in enumerate(names) if n.startswith("mom.") or n == "loss"] if p.name == "resnet18_train" else range(len(p.output_types))
    return {"exe": exe, "buffers": runner.upload(pjrt.get_client(), p.inputs, p.input_dtypes), "feedback": p.feedback,
            "results": [(i,) + tuple(p.output_types[i]) for i in wanted], "steps": case.get("steps", 1)}


_TYPESTR = {"f32": "<f4", "bf16": "<i2", "i32": "<i4"}


class _DeviceArray:
    """A device buffer's memory under the array interface torch reads; keeps the buffer alive."""

    def __init__(self, buf, shape, dtype):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": shape, "typestr": _TYPESTR[dtype], "data": (buf.device_pointer(), False), "version": 2}


def _tensor(buf, shape, dtype):
    t = torch.as_tensor(_DeviceArray(buf, shape, dtype), device="cuda")
    return t.view(torch.bfloat16) if dtype == "bf16" else t


def run(state):
    exe, buffers, feedback = state["exe"], state["buffers"], state["feedback"]
    for _ in range(state["steps"]):
        outs = exe.execute(buffers, donate=True)      # the train state is donated and replaced by its successor
        for k, i in feedback.items():
            buffers[i] = outs[k]
    return [_tensor(outs[i], shape, dtype) for i, shape, dtype in state["results"]]


# ---------------------------------------------------------------------------------------------------------------------
# what a pass cannot do without, and how exactly its results are determined
# ---------------------------------------------------------------------------------------------------------------------
_SIZE = {"f32": 4, "bf16": 2, "i32": 4}


def work(case):
    f = case["family"]
    if f == "embedding":
        rows = case["n_idx"] * case["dim"] * 4
        # gather: indices, rows read, rows written; gradient: upstream rows and indices read, the dense result written
        return {"bytes": 2 * case["n_idx"] * 4 + 3 * rows + case["vocab"] * case["dim"] * 4, "flops": case["n_idx"] * case["dim"]}
    if f == "op":
        n = case["rows"] * case["cols"]
        b, per = {"softmax": (8, 5), "exp": (8, 1), "add": (12, 1), "sum": (4, 1), "column_stats": (4, 3), "layernorm_bf16": (4, 8),
                  "bias_gelu_bf16": (4, 10)}[case["op"]]
        return {"bytes": n * b, "flops": n * per}
    if f == "mlp":
        batch, d_in, d_hidden, n_cls = case["batch"], case["d_in"], case["d_hidden"], 10
        params = d_in * d_hidden + d_hidden + d_hidden * n_cls + n_cls
        # every step reads the batch and the parameters and writes the parameters; no gradient of the input
        return {"bytes": case["steps"] * 4 * (2 * params + batch * d_in + batch + 1),
                "flops": case["steps"] * 2 * batch * (2 * d_in * d_hidden + 3 * d_hidden * n_cls)}
    p = _shape_of(_key(case))
    return dict(p)


@functools.lru_cache(maxsize=64)
def _shape_of(key):
    case = dict(key)
    p = _program(case, 0)
    size = lambda shape, dtype: math.prod(shape) * _SIZE[dtype]   # noqa: E731
    nbytes = sum(size(a.shape, d) for a, d in zip(p.inputs, p.input_dtypes)) + sum(size(s, d) for s, d in p.output_types)
    if case["family"] == "distilbert":       # of the two embedding tables only the rows that are looked up
        d_model, item = case["heads"] * case["head_dim"], _SIZE[case["dtype"]]
        nbytes += ((case["batch"] * case["seq"] - case["vocab"]) + (case["seq"] - 512)) * d_model * item
        flops = p.meta["flops"]
    elif case["family"] == "lstm":
        flops = p.meta["flops"]
    else:
        flops = p.meta["step_flops"] if case["train"] else _resnet_forward_flops(key)
    return (("bytes", nbytes), ("flops", flops))


def _resnet_forward_flops(key):
    c = dict(key)
    return configs.build_resnet18(batch=c["batch"], image=c["image"], width=c["width"]).meta["fwd_flops"]


def tolerance(case):
    """About four times what the path shows against itself with its sums in another order (or, for the encoder, MLP and LSTM
    in float32, against 64-bit sums)."""
    f = case["family"]
    if f == "resnet18" and case["train"]:
        # one step differs by 1e-6; a second one by up to 1.5e-3 (0.11 at the worst element): among millions of activations a few lie so
        # close to zero that the last bit decides their ReLU, and each carries a whole element of its layer's gradient
        return {"rel": 6e-3, "max": 0.45}
    if f == "distilbert" and case["dtype"] == "bf16":
        return {"rel": 2e-2, "max": 0.25}      # 1.1e-2 and 0.066 between rounding after every operator and after every kernel
    if f == "op" and case["op"].endswith("bf16"):
        return {"rel": 1e-2}
    if f == "lstm":
        return {"rel": 1e-5, "max": 1e-3}      # 7e-7 and 2e-4 (small second moments) after three steps
    return {"rel": 1e-5}


# ---------------------------------------------------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------------------------------------------------
def _double(a, dtype="f32", grad=False):
    t = torch.from_numpy(np.ascontiguousarray(a))
    if dtype == "bf16":
        t = t.bfloat16()
    return t.double().requires_grad_(grad) if t.is_floating_point() else t.long()


def _layer_norm64(x, scale, bias, eps):
    return torch.nn.functional.layer_norm(x, x.shape[-1:], scale, bias, eps)


def _gelu64(x):
    return torch.nn.functional.gelu(x, approximate="tanh")


def _exact_mlp(p, steps):
    w1, b1, w2, b2, x, y = [_double(a) for a in p.inputs]
    for _ in range(steps):
        params = [t.detach().requires_grad_(True) for t in (w1, b1, w2, b2)]
        loss = torch.nn.functional.cross_entropy(torch.relu(x @ params[0] + params[1]) @ params[2] + params[3], y)
        w1, b1, w2, b2 = [(t - 0.01 * g).detach() for t, g in zip(params, torch.autograd.grad(loss, params))]
    return [w1, b1, w2, b2, loss.detach()]


def _exact_embedding(p):
    table, idx, upstream = [_double(a) for a in p.inputs]
    return [table[idx], torch.zeros_like(table).index_add_(0, idx, upstream)]


def _exact_resnet18(p, train):
    A = {n: _double(a, grad=train and n not in ("x", "y") and not n.startswith("mom.")) for n, a in zip(p.input_names, p.inputs)}

    def conv(name, h, stride):
        w = A[name + ".kernel"].permute(3, 2, 0, 1)
        total = max((-(-h.shape[2] // stride) - 1) * stride + w.shape[2] - h.shape[2], 0)
        return torch.nn.functional.conv2d(torch.nn.functional.pad(h, (total // 2, total - total // 2) * 2), w, stride=stride)

    def norm(name, h):
        return torch.nn.functional.batch_norm(h, None, None, A[name + ".scale"], A[name + ".bias"], training=True, eps=1e-5)

    h = torch.relu(norm("bn_init", conv("conv_init", A["x"].permute(0, 3, 1, 2), 1)))
    for stage in range(1, 5):
        for block in (1, 2):
            q, stride = "stage%d_block%d" % (stage, block), 2 if stage > 1 and block == 1 else 1
            y = torch.relu(norm(q + ".bn1", conv(q + ".conv1", h, stride)))
            y = norm(q + ".bn2", conv(q + ".conv2", y, 1))
            if q + ".conv_proj.kernel" in A:
                h = norm(q + ".bn_proj", conv(q + ".conv_proj", h, stride))
            h = torch.relu(h + y)
    logits = h.mean((2, 3)) @ A["dense.kernel"] + A["dense.bias"]
    loss = torch.nn.functional.cross_entropy(logits, A["y"])
    if not train:
        return [logits, loss]
    names = [n[4:] for n in p.output_names if n.startswith("mom.")]
    return list(torch.autograd.grad(loss, [A[n] for n in names])) + [loss.detach()]


def _exact_encoder(p, case):
    A = {n: _double(a, d) for n, a, d in zip(p.input_names, p.inputs, p.input_dtypes)}
    batch, seq, heads, dim = case["batch"], case["seq"], case["heads"], case["head_dim"]
    x = _layer_norm64(A["word_emb"][A["input_ids"]] + A["pos_emb"][:seq], A["emb_ln.scale"], A["emb_ln.bias"], 1e-12)
    masked = (A["attention_mask"] == 0)[:, None, None, :]
    for n in range(case["layers"]):
        def linear(t, name):
            return t @ A["layer%d.%s.kernel" % (n, name)] + A["layer%d.%s.bias" % (n, name)]

        def norm(t, name):
            return _layer_norm64(t, A["layer%d.%s.scale" % (n, name)], A["layer%d.%s.bias" % (n, name)], 1e-12)

        q, k, v = linear(x, "qkv").reshape(batch, seq, 3, heads, dim).permute(2, 0, 3, 1, 4).contiguous()
        probs = torch.softmax((q @ k.transpose(2, 3).contiguous() / math.sqrt(dim)).masked_fill(masked, -math.inf), -1)
        x = norm(x + linear((probs @ v).transpose(1, 2).reshape(batch, seq, heads * dim), "out"), "sa_ln")
        x = norm(x + linear(_gelu64(linear(x, "ffn1")), "ffn2"), "out_ln")
    return [x]


def _exact_lstm(p, case):
    params = [_double(a, grad=True) for a in p.inputs[:5]]
    xs, y = _double(p.inputs[-2]), _double(p.inputs[-1])
    wi, wh, bias, wo, bo = params
    h = c = torch.zeros(case["batch"], case["hidden"], dtype=torch.float64)
    for x in xs:
        i, f, g, o = (x @ wi + h @ wh + bias).chunk(4, 1)
        c = torch.sigmoid(f) * c + torch.sigmoid(i) * torch.tanh(g)
        h = torch.sigmoid(o) * torch.tanh(c)
    loss = torch.nn.functional.cross_entropy(h @ wo + bo, y)
    grads = torch.autograd.grad(loss, params)
    # Adam's first step: its moments start at zero
    mu, nu = [0.1 * g for g in grads], [0.001 * g * g for g in grads]
    new = [(t - 1e-3 * (m / 0.1) / (torch.sqrt(v / 0.001) + 1e-8)).detach() for t, m, v in zip(params, mu, nu)]
    return new + mu + nu + [None, loss.detach()]


_EXACT_OPS = {
    "softmax": lambda x: [torch.softmax(x, -1)],
    "exp": lambda x: [torch.exp(x)],
    "add": lambda x, y: [x + y],
    "sum": lambda x: [x.sum()],
    "column_stats": lambda x: [x.sum(0), (x * x).sum(0)],
    "layernorm_bf16": lambda x, scale, bias: [_layer_norm64(x, scale, bias, 1e-12)],
    "bias_gelu_bf16": lambda x, bias: [_gelu64(x + bias)],
}


def exact(case, seed):
    p = _program(case, seed)
    f = case["family"]
    if f == "mlp":
        return _exact_mlp(p, case["steps"])
    if f == "embedding":
        return _exact_embedding(p)
    if f == "resnet18":
        return _exact_resnet18(p, case["train"])
    if f == "distilbert":
        return _exact_encoder(p, case)
    if f == "lstm":
        return _exact_lstm(p, case)
    return _EXACT_OPS[case["op"]](*[_double(a, d) for a, d in zip(p.inputs, p.input_dtypes)])
