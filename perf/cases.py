"""The work a user of this package has it do, as cases that can be timed: sizes, types and options in, one pass through
the public entry points out.

A case is a dict of plain values:

  what       "train": loss and both gradients, as a training step takes them; "eval": the loss alone, under no_grad
  N, H, V    token rows, hidden size, vocabulary
  dtype      of the activations and the weight ("bf16", "f16", "f32")
  master     True: the weight (and its gradient) is a float32 master copy under 16-bit activations
  tied       True: the weight is an embedding stored (V, H), handed over as ``weight.t()``; else a
             ``LinearCrossEntropyLoss`` module, stored (H, V)
  ignore     share of the labels that are ignore_index
  zipf       True: labels drawn from a Zipf distribution, as words are; else uniform
  trained    True: hidden states that point at their labels' columns by between nothing and certainty, as those of a
             model that has learned something do; else those of a model at its initialisation
  z_reg, scale, monitoring, n_chunk     the loss options
"""
from __future__ import annotations

import math

import torch

from linear_cross_entropy_loss_amd import LinearCrossEntropyLoss, linear_cross_entropy

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
IGNORE = -100
# float16 training multiplies the loss by such a factor before the backward, so that small gradients survive
LOSS_SCALE = 4096.0


def _case(what, N, H, V, dtype, **options):
    case = dict(what=what, N=N, H=H, V=V, dtype=dtype, master=False, tied=False, ignore=0.0, zipf=False, trained=False,
                z_reg=0.0, scale=1.0, monitoring=False, n_chunk=4096)
    case.update(options)
    return case


def listed():
    cases = {
        # one short sequence through a toy model: launches and host work are all there is
        "train_tiny": _case("train", 256, 256, 4096, "bf16", ignore=0.05),
        # a small model whose sizes are multiples of nothing, as a character or byte-pair vocabulary gives them
        "train_ragged": _case("train", 1999, 500, 10007, "bf16", ignore=0.1, trained=True),
        # classification of many items into few classes
        "train_classes": _case("train", 16384, 1024, 1000, "bf16"),
        # a model with a tied embedding on one device batch
        "train_tied": _case("train", 4096, 1024, 32000, "bf16", tied=True, ignore=0.05, zipf=True, trained=True, z_reg=1e-4),
        # the output layer of a small GPT-2 (its vocabulary is odd)
        "train_gpt2": _case("train", 8192, 768, 50257, "bf16", zipf=True, trained=True),
        # float32 throughout: a small model, or a check against a 16-bit run
        "train_f32": _case("train", 2048, 2048, 16384, "f32"),
        # automatic mixed precision: bf16 activations, float32 master weight and weight gradient
        "train_master": _case("train", 8192, 2048, 65536, "bf16", master=True, ignore=0.05),
        # the headline workload of the benchmark
        "train_headline": _case("train", 16384, 2048, 131072, "bf16", ignore=0.05),
        # float16 with every loss option on
        "train_f16_options": _case("train", 16384, 4096, 131072, "f16", ignore=0.1, zipf=True, trained=True, z_reg=1e-4, scale=0.5,
                                   monitoring=True),
        # a long batch against a very large vocabulary, mixed precision in float16
        "train_long": _case("train", 32768, 4096, 262144, "f16", master=True, ignore=0.1, zipf=True, n_chunk=8192),
        # validation loss and its metrics over a batch
        "eval_batch": _case("eval", 8192, 4096, 128256, "bf16", trained=True, zipf=True, monitoring=True, ignore=0.05),
        # the likelihood of one short answer
        "eval_answer": _case("eval", 48, 2048, 50304, "bf16", trained=True, zipf=True),
    }
    return [dict(case, name=name) for name, case in cases.items()]


def _flops(case):
    contractions = 3 if case["what"] == "train" else 1
    return 2.0 * contractions * case["N"] * (1.0 - case["ignore"]) * case["H"] * case["V"]


def draw(rng):
    """One more case: sizes spread over their logarithms, about a third of them odd, options as users set them."""
    most = max(_flops(c) for c in listed())

    def size(low, high, multiple):
        v = math.exp(rng.uniform(math.log(low), math.log(high)))
        if rng.random() < 0.35:
            return max(low, min(high, int(v) | 1))
        return max(multiple, min(high, int(round(v / multiple)) * multiple))

    while True:
        what = "eval" if rng.random() < 0.25 else "train"
        dtype = rng.choice(["bf16", "bf16", "bf16", "f16", "f16", "f32"])
        master = dtype != "f32" and rng.random() < 0.25
        tied = dtype != "f32" and rng.random() < 0.35
        case = _case(
            what, size(16 if what == "eval" else 128, 32768, 64), size(64, 8192, 64), size(256, 262144, 128), dtype,
            master=master, tied=tied, ignore=rng.choice([0.0, 0.05, 0.1, 0.3]), zipf=rng.random() < 0.5,
            trained=rng.random() < 0.5, z_reg=rng.choice([0.0, 0.0, 1e-4]), scale=rng.choice([1.0, 1.0, 0.5]),
            monitoring=rng.random() < 0.3, n_chunk=rng.choice([2048, 4096, 4096, 8192]))
        # (float32 products cost several times a 16-bit one)
        if _flops(case) * (6.0 if dtype == "f32" else 1.0) <= most and case["H"] * case["V"] <= 1 << 30:
            return case


def prepare(case, seed):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    N, H, V = case["N"], case["H"], case["V"]
    dtype = DTYPES[case["dtype"]]
    w_dtype = torch.float32 if case["master"] else dtype
    std = 1.0 / math.sqrt(H)

    def init(t):
        with torch.no_grad():
            t.copy_(torch.nn.init.trunc_normal_(torch.empty(t.shape, device=dev), mean=0.0, std=std, a=-3 * std, b=3 * std,
                                                generator=gen))

    if case["zipf"]:
        p = torch.arange(1, V + 1, dtype=torch.float64, device=dev) ** -1.1
        cdf = torch.cumsum(p, 0) / p.sum()
        y = torch.searchsorted(cdf, torch.rand(N, generator=gen, dtype=torch.float64, device=dev)).clamp_(max=V - 1)
    else:
        y = torch.randint(0, V, (N,), generator=gen, device=dev)

    state = {"case": case}
    if case["tied"]:
        weight = torch.nn.Parameter(torch.empty((V, H), device=dev, dtype=w_dtype))
        init(weight)
        columns = weight.detach()[y]
    else:
        module = LinearCrossEntropyLoss(
            H, V, device=dev, dtype=w_dtype, ignore_index=IGNORE, logit_scale=case["scale"], z_regularization=case["z_reg"],
            N_chunk_size=case["n_chunk"], init_method=init)
        module.monitoring = case["monitoring"]
        state["module"] = module
        weight = module.weight
        columns = weight.detach()[:, y].t()
    x = torch.randn((N, H), generator=gen, device=dev)
    if case["trained"]:
        # the label's logit stands 0 ... 20 above the others' middle
        x += columns.float() * (torch.rand((N, 1), generator=gen, device=dev) * (20.0 / case["scale"]))
    if case["ignore"] > 0:
        drop = torch.rand(N, generator=gen, device=dev) < case["ignore"]
        drop[0] = False  # (some label is always there: the mean over none is not a number)
        y[drop] = IGNORE
    state.update(x=x.to(dtype).requires_grad_(case["what"] == "train"), y=y, weight=weight)
    return state


def run(state):
    case, x, y, weight = state["case"], state["x"], state["y"], state["weight"]
    with torch.set_grad_enabled(case["what"] == "train"):
        if case["tied"]:
            loss, z_value, logit_max, logit_entropy, logit_norm = linear_cross_entropy(
                x, y, weight.t(), IGNORE, case["z_reg"], case["scale"], case["n_chunk"], case["monitoring"])
            metrics = {"z_value": z_value, "logit_max": logit_max, "logit_entropy": logit_entropy, "logit_norm": logit_norm}
        else:
            loss = state["module"](x, y)
            metrics = state["module"].latest_metrics
    out = {"loss": loss.detach()}
    if case["monitoring"]:
        out.update({k: v.detach() for k, v in metrics.items()})
    if case["what"] == "train":
        scaled = loss * LOSS_SCALE if case["dtype"] == "f16" else loss
        out["dx"], out["dw"] = torch.autograd.grad(scaled, (x, weight))
    return out


def work(case):
    N, H, V = case["N"], case["H"], case["V"]
    es = 4 if case["dtype"] == "f32" else 2
    ws = 4 if case["master"] else es
    inputs = N * H * es + H * V * ws + N * 8
    outputs = N * H * es + H * V * ws if case["what"] == "train" else 0
    return {"bytes": float(inputs + outputs + 4), "flops": _flops(case)}


def tolerance(case):
    """Four times what the path shows against the same in 64 bits (2-norm)."""
    if case["what"] == "eval":
        return {"rel": 1e-5}  # (scalars, from sums of 32-bit terms)
    # the gradients pass through one or two roundings to the compute type and one to their own: measured up to 2.1e-3 in
    # bf16, 2.5e-4 in f16, 2.6e-6 in f32 (bf16 pairs: 16 bits of mantissa)
    return {"rel": {"bf16": 8e-3, "f16": 1e-3, "f32": 1.1e-5}[case["dtype"]]}
