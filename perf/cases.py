"""The work a program has this framework do, as cases that can be timed and compared.

Each case is one pass through the public entry points of `hpfp8`: a linear layer or a SwiGLU MLP block in inference
(decode and prefill), their training steps (forward and backward, every recipe and the options that training programs
switch on), the MoE grouped linear (inference, and forward and input gradient with frozen experts), and the gradient
bucket's round trip.  Layer sizes are those of the repository's own configurations (hidden 7168, MLP width 18432, o_proj
16384 -> 7168, experts [4096, 7168], the per-tensor 2048 x 1024 x 1024 problem, the 72-gradient bucket) or multiples of
128 in the same ranges.

`listed()` names the cases, `draw(rng)` gives further ones of the ranges they stand for, `prepare` makes what a program
holds before the call, `run` is the pass.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "hyper-parallel_amd"))      # imported from the repository's root

import hpfp8  # noqa: E402


# ------------------------------------------------------------------------------------------------
# the cases
# ------------------------------------------------------------------------------------------------
def listed():
    return [
        # one decode step of a served layer: a handful of sequences against the attention output projection, whose
        # FP8 form was made when the model was loaded
        dict(name="decode_linear", kind="linear_infer", tokens=8, inp=16384, out=7168, recipe="blockwise", bias=False),
        # the same step of the dense MLP block, at a larger serving batch that is no multiple of anything
        dict(name="decode_mlp", kind="mlp_infer", tokens=37, hidden=7168, inter=18432),
        # the MoE layer of a decode step: 64 tokens, each routed to 8 of 32 experts
        dict(name="decode_moe", kind="moe_infer", rows=512, experts=32, inp=7168, out=4096),
        # a chunk of prefill: an ordinary linear, ragged token count, bias
        dict(name="prefill_linear", kind="linear_infer", tokens=1000, inp=7168, out=7168, recipe="blockwise", bias=True),
        # a full prefill of the dense MLP block
        dict(name="prefill_mlp", kind="mlp_infer", tokens=4096, hidden=7168, inter=18432),
        # training of a small linear with one scale per tensor, weight quantized in the step: launches count
        dict(name="train_small_per_tensor", kind="linear_train", tokens=2048, inp=1024, out=1024, recipe="per_tensor",
             bias=True, cached=False, main_grad=False),
        # training of the attention output projection, the default recipe, weight quantized in the step
        dict(name="train_o_proj", kind="linear_train", tokens=4096, inp=16384, out=7168, recipe="blockwise", bias=True,
             cached=False, main_grad=False),
        # a packed batch of variable-length sequences: the token count is no multiple of the scaling groups
        dict(name="train_ragged", kind="linear_train", tokens=1531, inp=7168, out=2048, recipe="blockwise", bias=True,
             cached=False, main_grad=False),
        # one micro-batch of several: the weight's FP8 form is that of the step, its gradient is added onto the fp32
        # main gradient; power-of-two scales
        dict(name="train_accumulate_pow2", kind="linear_train", tokens=2048, inp=4096, out=7168, recipe="blockwise_pow2",
             bias=False, cached=True, main_grad=True),
        # training of the dense MLP block, weights quantized in the step
        dict(name="train_mlp", kind="mlp_train", tokens=4096, hidden=7168, inter=18432, cached=False),
        # fine-tuning through an MoE layer whose experts are frozen (what lies below it is trained): 16384 tokens to 8
        # of 32 experts, unevenly, forward and input gradient; the experts' FP8 form was made once
        dict(name="train_through_moe", kind="moe_train", rows=131072, experts=32, inp=7168, out=4096),
        # the gradient bucket around a reduce-scatter over 8 ranks: 72 gradients, weights and vectors, packed and
        # quantized; this rank's reduced row dequantized, scaled and unpacked
        dict(name="bucket", kind="bucket", elements=1 << 28, gradients=72, shards=8, odd=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A feature count: a multiple of 128, spread over the logarithm of the range."""
    return max(lo, min(hi, 128 * max(1, round(_log_int(rng, lo, hi) / 128))))


def _tokens(rng, lo, hi):
    """A token count: half of the time a multiple of 128 (a padded batch), otherwise anything."""
    n = _log_int(rng, lo, hi)
    return max(128, n // 128 * 128) if rng.random() < 0.5 and n >= 128 else n


def draw(rng):
    kind = rng.choice(["linear_infer", "linear_infer", "mlp_infer", "moe_infer", "linear_train", "linear_train",
                       "linear_train", "mlp_train", "moe_train", "bucket"])
    most = max(_seconds(c) for c in listed())
    while True:
        if kind == "linear_infer":
            case = dict(kind=kind, tokens=_tokens(rng, 1, 8192), inp=_width(rng, 1024, 16384), out=_width(rng, 1024, 16384),
                        recipe=rng.choice(["blockwise", "blockwise", "blockwise_pow2", "per_tensor"]), bias=rng.random() < 0.5)
        elif kind == "mlp_infer":
            case = dict(kind=kind, tokens=_tokens(rng, 1, 8192), hidden=_width(rng, 1024, 7168), inter=_width(rng, 1024, 18432))
        elif kind == "moe_infer":
            case = dict(kind=kind, rows=_log_int(rng, 64, 65536), experts=rng.choice([8, 16, 32, 64]),
                        inp=_width(rng, 1024, 7168), out=_width(rng, 1024, 4096))
        elif kind == "linear_train":
            recipe = rng.choice(["blockwise", "blockwise", "blockwise_pow2", "per_tensor"])
            case = dict(kind=kind, tokens=_tokens(rng, 256, 8192), inp=_width(rng, 1024, 16384), out=_width(rng, 1024, 16384),
                        recipe=recipe, bias=rng.random() < 0.5, cached=rng.random() < 0.5,
                        main_grad=recipe != "per_tensor" and rng.random() < 0.3)
        elif kind == "mlp_train":
            case = dict(kind=kind, tokens=_tokens(rng, 256, 8192), hidden=_width(rng, 1024, 7168),
                        inter=_width(rng, 1024, 18432), cached=rng.random() < 0.5)
        elif kind == "moe_train":
            case = dict(kind=kind, rows=_log_int(rng, 1024, 131072), experts=rng.choice([8, 16, 32, 64]),
                        inp=_width(rng, 1024, 7168), out=_width(rng, 1024, 4096))
        else:
            case = dict(kind=kind, elements=_log_int(rng, 1 << 20, 1 << 28), gradients=_log_int(rng, 4, 200),
                        shards=rng.choice([1, 2, 4, 8]), odd=rng.random() < 0.5)
        if _seconds(case) <= most:
            return case


def _seconds(case):
    """A rough time of a pass, to keep drawn cases below the largest listed one."""
    w = work(case)
    return w["bytes"] / 5e12 + w["flops"] / 2e15


# ------------------------------------------------------------------------------------------------
# what a program has in hand
# ------------------------------------------------------------------------------------------------
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _normal(g, shape, std=1.0):
    return torch.empty(shape, dtype=torch.bfloat16, device="cuda").normal_(0.0, std, generator=g)


def _activations(g, rows, cols):
    """Normal values, 0.1 % of them fifty times larger: the outliers of a transformer's activations."""
    x = _normal(g, (rows, cols))
    n = max(1, round(0.001 * rows * cols))
    x.view(-1)[torch.randint(0, rows * cols, (n,), device="cuda", generator=g)] *= 50.0
    return x


def _gradients(g, rows, cols):
    """Laplace-distributed values of the size of an output gradient."""
    u = torch.empty((rows, cols), dtype=torch.float32, device="cuda").uniform_(-0.4999, 0.4999, generator=g)
    return (u.sign() * torch.log1p(u.abs_().mul_(-2.0)).mul_(-0.0007)).to(torch.bfloat16)


def _expert_rows(case, seed):
    """Rows per expert: a Zipf(1.1) law over the experts in random order, two of them without any."""
    r = np.random.RandomState(int(seed) % (1 << 32))
    e, rows = case["experts"], case["rows"]
    p = 1.0 / np.arange(1, e + 1) ** 1.1
    p[-2:] = 0.0
    return r.multinomial(rows, r.permutation(p / p.sum()))


def _expert_weights(g, case):
    """The experts' bf16 weights, drawn expert by expert (no fp32 copy of the stack)."""
    return _normal(g, (case["experts"], case["out"], case["inp"]), 0.02)


def _bucket_sizes(case):
    """Elements each gradient owns in one row of the bucket: large matrices and a third of vectors, adding up to about
    `elements` over all shards.  `odd`: sizes that are no multiple of a vector (a vocabulary or a head count that does
    not divide), so chunks of the gradients start anywhere."""
    count, per_row = case["gradients"], case["elements"] // case["shards"]
    small = max(1, count // 3)
    vector = max(16, min(7168 // case["shards"], per_row // (8 * count)))
    matrix = max(16, (per_row - small * vector) // max(1, count - small))
    sizes = []
    for i in range(count):
        n = vector if i % 3 == 2 and i // 3 < small else matrix
        sizes.append(n - n % 16 + (i * 37 % 15 + 1 if case["odd"] else 0))
    return sizes


def prepare(case, seed):
    g = _generator(seed)
    kind = case["kind"]
    s = dict(case=case)
    if kind in ("linear_infer", "linear_train"):
        s["x"] = _activations(g, case["tokens"], case["inp"])
        s["w"] = _normal(g, (case["out"], case["inp"]), 0.02)
        s["b"] = _normal(g, (case["out"],), 0.1) if case["bias"] else None
        s["f8"] = None
        if kind == "linear_infer" or case["cached"]:
            s["f8"] = hpfp8.quantize_weight(s["w"], with_transpose=kind == "linear_train", pow2=case["recipe"] == "blockwise_pow2",
                                            per_tensor=case["recipe"] == "per_tensor")
    elif kind in ("mlp_infer", "mlp_train"):
        s["x"] = _activations(g, case["tokens"], case["hidden"])
        s["gu"] = _normal(g, (2 * case["inter"], case["hidden"]), 0.006)
        s["dn"] = _normal(g, (case["hidden"], case["inter"]), 0.006)
        s["gu8"] = s["dn8"] = None
        if kind == "mlp_infer" or case["cached"]:
            s["gu8"] = hpfp8.quantize_weight(s["gu"], with_transpose=kind == "mlp_train")
            s["dn8"] = hpfp8.quantize_weight(s["dn"], with_transpose=kind == "mlp_train")
        if kind == "mlp_infer":
            s["gu"] = s["dn"] = None               # a served model keeps the FP8 form alone
    elif kind in ("moe_infer", "moe_train"):
        s["x"] = _activations(g, case["rows"], case["inp"])
        s["w"] = _expert_weights(g, case)
        s["offs"] = torch.from_numpy(np.cumsum(_expert_rows(case, seed)).astype(np.int32)).cuda()
        s["f8"] = hpfp8.quantize_grouped_weight(s["w"], with_transpose=kind == "moe_train")
    else:
        sizes = _bucket_sizes(case)
        s["bucket"] = hpfp8.Fp8GradBucket(sizes, shard_size=case["shards"], grad_scale=0.125)
        s["grads"] = []
        for n in sizes:
            t = _normal(g, (n * case["shards"],), 1e-4)
            t[torch.randint(0, t.numel(), (1 + t.numel() // 10000,), device="cuda", generator=g)] *= 1e3
            s["grads"].append(t)
        s["flat"] = torch.zeros(s["bucket"].row_elems, dtype=torch.bfloat16, device="cuda")
        s["outs"] = [s["flat"][o:o + n] for o, n in zip(s["bucket"].offsets, sizes)]
    if kind.endswith("_train"):
        width = case["hidden"] if kind == "mlp_train" else case["out"]
        s["go"] = _gradients(g, s["x"].shape[0], width)
        s["x"].requires_grad_(True)
        for name in ("w", "b", "gu", "dn"):
            if s.get(name) is not None:
                s[name] = torch.nn.Parameter(s[name], requires_grad=kind != "moe_train")
        if case.get("main_grad"):
            s["w"].main_grad = torch.zeros(s["w"].shape, dtype=torch.float32, device="cuda")
    return s


# ------------------------------------------------------------------------------------------------
# one pass
# ------------------------------------------------------------------------------------------------
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "linear_infer":
        with torch.no_grad():
            return hpfp8.fp8_linear(s["x"], s["w"], s["b"], recipe=case["recipe"], weight_fp8=s["f8"])
    if kind == "mlp_infer":
        with torch.no_grad():
            return hpfp8.fp8_swiglu_mlp(s["x"], s["gu8"], s["dn8"])
    if kind == "moe_infer":
        with torch.no_grad():
            return hpfp8.fp8_grouped_linear(s["x"], s["w"], s["offs"], weight_fp8=s["f8"])
    if kind == "linear_train":
        y = hpfp8.fp8_linear(s["x"], s["w"], s["b"], recipe=case["recipe"], weight_fp8=s["f8"],
                             apply_grad_on_fp32_main_grad=case["main_grad"])
        wanted = [s["x"]] + ([] if case["main_grad"] else [s["w"]]) + ([s["b"]] if case["bias"] else [])
        grads = torch.autograd.grad(y, wanted, s["go"])
        return [y.detach(), *grads] + ([s["w"].main_grad] if case["main_grad"] else [])
    if kind == "mlp_train":
        y = hpfp8.fp8_swiglu_mlp(s["x"], s["gu"], s["dn"], gate_up_fp8=s["gu8"], down_fp8=s["dn8"])
        return [y.detach(), *torch.autograd.grad(y, (s["x"], s["gu"], s["dn"]), s["go"])]
    if kind == "moe_train":
        y = hpfp8.fp8_grouped_linear(s["x"], s["w"], s["offs"], weight_fp8=s["f8"])
        return [y.detach(), *torch.autograd.grad(y, (s["x"],), s["go"])]
    codes, scale_inv = s["bucket"].pack(s["grads"])
    s["bucket"].unpack(codes[0], scale_inv[0], s["outs"])
    return [codes.view(torch.uint8), scale_inv, s["flat"]]


# ------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ------------------------------------------------------------------------------------------------
def work(case):
    """Bytes: every input read once, every output written once.  A weight whose FP8 form was made before is read as
    codes (1 byte, once in each direction: the two directions contract over different dimensions)."""
    kind = case["kind"]
    if kind in ("linear_infer", "linear_train"):
        m, k, n = case["tokens"], case["inp"], case["out"]
        if kind == "linear_infer":
            return {"bytes": 2 * m * k + n * k + 2 * m * n, "flops": 2 * m * n * k}
        weight = 2 * n * k
        return {"bytes": 2 * (2 * m * k + 2 * m * n) + weight + (8 if case["main_grad"] else 2) * n * k, "flops": 6 * m * n * k}
    if kind in ("mlp_infer", "mlp_train"):
        m, h, i = case["tokens"], case["hidden"], case["inter"]
        if kind == "mlp_infer":
            return {"bytes": 4 * m * h + 3 * h * i, "flops": 6 * m * h * i}
        return {"bytes": 8 * m * h + 12 * h * i, "flops": 18 * m * h * i}
    if kind in ("moe_infer", "moe_train"):
        r, e, k, n = case["rows"], case["experts"], case["inp"], case["out"]
        used = min(e - 2, r)                      # two experts get no rows
        if kind == "moe_infer":
            return {"bytes": 2 * r * (k + n) + used * n * k, "flops": 2 * r * n * k}
        return {"bytes": 4 * r * (k + n) + 2 * used * n * k, "flops": 4 * r * n * k}
    row = sum(_bucket_sizes(case))
    return {"bytes": int(row * case["shards"] * (3 + 4 / 128) + row * (3 + 4 / 128)), "flops": 0}


def tolerance(case):
    """Four times what the path differs by from itself with every matrix product in 64 bits.  One GEMM: the bf16
    rounding of a result that an order of summation moves (rel 2.6e-4 to 4.7e-4, one bf16 step of 2^-7 at most).  In an
    MLP block such a result is quantized again, which turns a step into an E4M3 code and shows in everything behind it
    (rel 2.4e-3 to 3.4e-3; single elements of the gate/up weight gradient by more than their own size)."""
    kind = case["kind"]
    if kind == "bucket":
        return "exact"
    if kind == "mlp_infer":
        return {"rel": 1.4e-2, "max": 0.16}
    if kind == "mlp_train":
        return {"rel": 1.4e-2, "max": 0.99}
    return {"rel": 2e-3, "max": 3.2e-2}
