"""The work that users have the fused loss do, as cases that can be prepared, run and timed one by one.

A case is one call of ``linear_cross_entropy`` -- forward alone, or forward and backward -- on inputs that are resident
on the GPU, as a training step or an evaluation makes it.  ``listed`` names fixed cases, ``draw`` makes more of the same
ranges, ``prepare`` builds the inputs, ``run`` is one pass, ``work`` counts what the pass cannot do without, and
``tolerance`` says how far two correct implementations of the same precision lie apart.

The keys of a case:

    batch, steps   rows of E are batch x steps tokens
    width, classes E is [batch, steps, width], C is [classes, width]
    dtype          "bf16", "fp16", "fp32": the type of E, C and the bias; "autocast": E is bf16, C and the bias are
                   fp32 parameters, and the call runs inside torch.autocast(bf16)
    impl, softcap (0: none), reduction, shift, bias     as the operator takes them
    z_loss         weight of the squared log-sum-exp in the loss (0: none)
    ignored        ignored labels: a share of the rows, at random ("random"), at the start of each sequence as a prompt
    ignored_at     is ("prompt"), or at its end as padding is ("padding")
    data           "flat": E ~ N(0, 1), C ~ N(0, 0.02), uniform labels: a head that has not learnt yet
                   "zipf": the same with labels of frequency 1 / rank^1.1, as those of text are
                   "peaked": E = 4 C[label] + N(0, 0.5): few classes matter to a row
                   "trained": E = g C[label] + h C[other] + N(0, 0.5), g and h of each row uniform in 2 .. 12: sure of
                   most labels, unsure of some, wrong about a few
    shard          C holds the first ``classes`` of this many classes (0: all of them)
    backward       whether the pass takes gradients
"""

import os
import sys

import torch

_PACKAGE = os.path.abspath("ml-cross-entropy_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from cut_cross_entropy import VocabParallelOptions, linear_cross_entropy  # noqa: E402
from cut_cross_entropy.utils import compute_z_loss  # noqa: E402

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32, "autocast": torch.bfloat16}
_UNFILTERED_E = ("cce_exact", "cce_kahan_full", "cce_kahan_full_c_full_e", "cce_kahan_full_e")
_UNFILTERED_C = ("cce_exact", "cce_kahan_full", "cce_kahan_full_c_full_e", "cce_kahan_full_c")


def _case(name, batch, steps, width, classes, **more):
    case = dict(name=name, batch=batch, steps=steps, width=width, classes=classes, dtype="bf16", impl="cce", softcap=0.0,
                reduction="mean", shift=0, bias=False, z_loss=0.0, ignored=0.0, ignored_at="random", data="flat",
                shard=0, backward=True)
    case.update(more)
    return case


def listed():
    return [
        # A unit-test-sized head: what a small model, a test suite or the first step of a notebook calls.  Launches and
        # host work are all of it.
        _case("small", 1, 256, 128, 512),
        # A GPT-2-sized vocabulary under a width that is no multiple of the kernels' stage, with everything else odd as
        # well: fp16, a bias, padded sequences, next-token labels, one loss and one log-sum-exp per token.
        _case("ragged", 4, 251, 1000, 50257, dtype="fp16", bias=True, softcap=50.0, shift=1, reduction="none", z_loss=1e-4,
              ignored=0.1, ignored_at="padding"),
        # Scoring a few continuations with the Gemma-2-2B-shaped head: forward alone, losses per token; reading C is
        # most of the work.
        _case("score", 4, 16, 2304, 256000, softcap=30.0, reduction="none", data="trained", backward=False),
        # One micro-batch of supervised fine-tuning on the Mistral-Nemo-shaped head: a short sequence, its prompt
        # ignored, a model that knows most answers.
        _case("finetune", 1, 512, 5120, 131072, shift=1, ignored=0.4, ignored_at="prompt", data="trained"),
        # The small reference workload of the benchmark (c1).
        _case("c1", 1, 4096, 1024, 32000, ignored=0.05),
        # The Phi-3.5-shaped head in the usual mixed-precision recipe: fp32 master weights under bf16 autocast, and the
        # preset for pre-training that filters dE alone.
        _case("mixed", 8, 1024, 3072, 32064, dtype="autocast", impl="cce_kahan_full_c", shift=1, data="zipf"),
        # Full fp32: the same head as a user who checks a recipe, or fine-tunes in fp32, runs it.
        _case("fp32", 2, 1024, 3072, 32064, dtype="fp32", shift=1, data="trained"),
        # The headline workload (c2): the Gemma-2-2B-shaped head.
        _case("c2", 1, 8192, 2304, 256000, softcap=30.0),
        # The Llama-3-8B-shaped head over long padded sequences (c3).
        _case("c3", 4, 4096, 4096, 128256, shift=1, ignored=0.0625, ignored_at="padding"),
        # Pre-training precision: no filter, z-loss, labels of text, one loss per token (c4).
        _case("c4", 1, 8192, 2048, 256000, impl="cce_kahan_full_c_full_e", reduction="none", z_loss=1e-4, data="zipf"),
        # Long sequences whose soft-max is peaked (c5), and one vocabulary shard of the same.
        _case("c5", 1, 65536, 3584, 152064, data="peaked"),
        _case("c5shard", 1, 65536, 3584, 19008, data="peaked", shard=152064),
    ]


_LARGEST = 2.0 * 65536 * 3584 * 152064  # multiply-adds x 2 of the largest listed case


def _spread(rng, low, high):
    """A whole number, its logarithm uniform."""
    return int(round(low * (high / low) ** rng.random()))


def draw(rng):
    while True:
        rows = _spread(rng, 16, 65536)
        batch = rng.choice([1, 1, 1, 2, 4, 8])
        steps = max(4, rows // batch)
        width = _spread(rng, 64, 5120)
        multiple = rng.choice([256, 128, 128, 128, 64, 8, 8, 1])
        width = max(64, width // multiple * multiple)
        classes = _spread(rng, 512, 256000)
        if rng.random() < 0.5:
            classes = max(512, classes // 64 * 64)
        dtype = rng.choice(["bf16"] * 5 + ["autocast", "autocast", "fp16", "fp32", "fp32"])
        backward = rng.random() < 0.8
        impl = rng.choice(["cce"] * 5 + ["cce_exact", "cce_kahan", "cce_kahan_full_c", "cce_kahan_full_e",
                                         "cce_kahan_full_c_full_e"])
        cost = 2.0 * batch * steps * width * classes * (4 if backward else 1) * (6 if dtype == "fp32" else 1)
        if cost > _LARGEST:
            continue
        reduction = rng.choice(["mean", "mean", "mean", "sum", "none"])
        z_loss = rng.choice([0.0, 0.0, 1e-4])
        return dict(batch=batch, steps=steps, width=width, classes=classes, dtype=dtype, impl=impl,
                    softcap=rng.choice([0.0, 0.0, 30.0, 50.0]), reduction=reduction, shift=rng.choice([0, 1, 1]),
                    bias=rng.random() < 0.2, z_loss=z_loss, ignored=rng.choice([0.0, 0.05, round(rng.random() * 0.6, 3)]),
                    ignored_at=rng.choice(["random", "prompt", "padding"]),
                    data=rng.choice(["flat", "zipf", "peaked", "trained", "trained"]),
                    shard=rng.choice([0, 0, 0, 0, classes * 4]), backward=backward)


def _ignored_steps(case):
    return int(case["ignored"] * case["steps"])


def _valid_rows(case):
    """Rows whose (shifted) label is not ignored.  Every sequence has the same number of ignored labels; the labels
    before ``shift`` are no row's label, and a prompt covers them."""
    labels = case["steps"] - case["shift"]
    hidden = _ignored_steps(case)
    if case["ignored_at"] == "prompt":
        hidden = max(0, hidden - case["shift"])
    return case["batch"] * (labels - min(hidden, labels))


def _labels(case, count, total, gen):
    if case["data"] != "zipf":
        return torch.randint(0, total, (count,), generator=gen, device="cuda")
    cdf = torch.arange(1, total + 1, dtype=torch.float64, device="cuda").pow_(-1.1).cumsum_(0)
    cdf /= cdf[-1].clone()
    u = torch.rand((count,), dtype=torch.float64, generator=gen, device="cuda")
    return torch.searchsorted(cdf, u).clamp_(max=total - 1)


def _randn(rows, cols, std, dtype, gen):
    out = torch.empty((rows, cols), dtype=dtype, device="cuda")
    step = max(1, (1 << 27) // cols)
    for s in range(0, rows, step):
        n = min(step, rows - s)
        out[s : s + n] = torch.randn((n, cols), generator=gen, device="cuda").mul_(std)
    return out


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    batch, steps, width, held = case["batch"], case["steps"], case["width"], case["classes"]
    total = case["shard"] or held
    e_type = _DTYPES[case["dtype"]]
    c_type = torch.float32 if case["dtype"] == "autocast" else e_type
    rows = batch * steps
    c = _randn(total, width, 0.02, c_type, gen)
    t = _labels(case, rows, total, gen)
    if case["data"] in ("flat", "zipf"):
        e = _randn(rows, width, 1.0, e_type, gen)
    else:
        e = torch.empty((rows, width), dtype=e_type, device="cuda")
        # row i predicts the label ``shift`` steps on
        said = t.roll(-case["shift"]) if case["shift"] else t
        other = torch.randint(0, total, (rows,), generator=gen, device="cuda")
        peaked = case["data"] == "peaked"
        sure = torch.rand((rows, 2), generator=gen, device="cuda").mul_(10.0).add_(2.0)
        for s in range(0, rows, 8192):
            part = slice(s, min(rows, s + 8192))
            noise = torch.randn((said[part].numel(), width), generator=gen, device="cuda").mul_(0.5)
            if peaked:
                e[part] = noise.add_(c[said[part]].float(), alpha=4.0)
            else:
                e[part] = noise + sure[part, :1] * c[said[part]].float() + sure[part, 1:] * c[other[part]].float()
    t = t.view(batch, steps)
    hidden = _ignored_steps(case)
    if hidden and case["ignored_at"] == "prompt":
        t[:, :hidden] = -100
    elif hidden and case["ignored_at"] == "padding":
        t[:, steps - hidden :] = -100
    elif hidden:
        shift = case["shift"]
        order = torch.rand((batch, steps - shift), generator=gen, device="cuda").argsort(dim=1)
        t[:, shift:].scatter_(1, order[:, : min(hidden, steps - shift)], -100)
    c = c[:held].clone() if held != total else c
    bias = _randn(1, held, 0.5, c_type, gen).view(-1) if case["bias"] else None
    state = dict(case=case, e=e.view(batch, steps, width), c=c, t=t, bias=bias, upstream=None)
    if case["backward"]:
        for x in (state["e"], c, bias):
            if x is not None:
                x.requires_grad_(True)
        if case["reduction"] == "none":
            # what the caller's own weighting of its tokens sends back
            out = (batch, steps - case["shift"])
            state["upstream"] = torch.rand(out, generator=gen, device="cuda").mul_(1.5).add_(0.5)
    state["shard"] = VocabParallelOptions(0, held) if held != total else None
    return state


def _loss(state):
    case = state["case"]
    out = linear_cross_entropy(
        state["e"], state["c"], state["t"], bias=state["bias"], softcap=case["softcap"] or None, reduction=case["reduction"],
        shift=case["shift"], return_lse=case["z_loss"] > 0, impl=case["impl"], vocab_parallel_options=state["shard"])
    if not case["z_loss"]:
        return out, None
    loss, lse = out
    extra = compute_z_loss(lse, state["t"], shift=case["shift"], reduction=case["reduction"])
    return loss + case["z_loss"] * extra, lse


def run(state):
    case = state["case"]
    with torch.set_grad_enabled(case["backward"]):
        if case["dtype"] == "autocast":
            with torch.autocast("cuda", dtype=torch.bfloat16):
                loss, lse = _loss(state)
        else:
            loss, lse = _loss(state)
    out = {"loss": loss.detach()}
    if lse is not None:
        out["lse"] = lse.detach()
    if case["backward"]:
        leaves = {"d_e": state["e"], "d_c": state["c"]}
        if state["bias"] is not None:
            leaves["d_bias"] = state["bias"]
        for x in leaves.values():
            x.grad = None
        loss.backward(state["upstream"])
        out.update({name: x.grad for name, x in leaves.items()})
    return out


def work(case):
    """Each input read once and each output written once.  The products: 2 B V D for the logits; an unfiltered gradient
    takes one product of the same size more, and the logits again, since the operator's point is that they are
    never kept.  A filtered gradient has to hold the entries of the labels; how many others pass the filter depends on the
    data, and they are not counted."""
    rows = case["batch"] * case["steps"]
    width, classes = case["width"], case["classes"]
    valid = _valid_rows(case)
    e_bytes = 4 if case["dtype"] == "fp32" else 2
    c_bytes = 4 if case["dtype"] in ("fp32", "autocast") else 2
    bias = classes * c_bytes if case["bias"] else 0
    outputs = (rows if case["reduction"] == "none" else 1) * 4 + (rows * 4 if case["z_loss"] else 0)
    moved = valid * width * e_bytes + classes * width * c_bytes + bias + rows * 8 + outputs
    plane = 2.0 * valid * width * classes
    flops = plane
    if case["backward"]:
        moved += rows * width * e_bytes + classes * width * c_bytes + bias
        # fp32's filter threshold lies below what a soft-max produces: its gradients are whole
        whole_e = case["impl"] in _UNFILTERED_E or case["dtype"] == "fp32"
        whole_c = case["impl"] in _UNFILTERED_C or case["dtype"] == "fp32"
        flops += plane * (whole_e + whole_c + (whole_e or whole_c))
        flops += 2.0 * valid * width * ((not whole_e) + (not whole_c))
    return {"bytes": float(moved), "flops": float(flops)}


def tolerance(case):
    """Measured against the same formulas in 64 bits over the listed cases and a dozen drawn ones, 2-norm of each output.

    16-bit inputs, whole gradients: 1e-3 .. 3.6e-3 (dz is rounded to the type of the inputs, as are the results); single
    elements of d_c, where the rows of a frequent class cancel, up to 0.64 of the root mean square.
    Filtered gradients: what lies below the threshold is dropped or kept by tile, up to 2.2e-2 of d_e between an
    implementation that drops all it may and one that drops nothing.
    fp32: up to 1.9e-6, single elements 7e-5.
    """
    if case["dtype"] == "fp32":
        return {"rel": 1e-5, "max": 1e-3}
    if not case["backward"]:
        return {"rel": 1e-5, "max": 1e-3}  # the sums of the log-sum-exp are fp32 whatever the inputs: 5e-7 measured
    filtered = case["impl"] not in _UNFILTERED_E or case["impl"] not in _UNFILTERED_C
    return {"rel": 0.025 if filtered else 0.01, "max": 0.99}
