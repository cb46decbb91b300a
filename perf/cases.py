"""Performance cases: the work that users of this library have it do, through its public entry points.

Four kinds of program call the library:

* generation: one token per call and row, the state updated in place (``FastWeightState``);
* a prompt, or scoring: a sequence without gradients (``LFWFunction`` under ``no_grad``);
* training: forward and backward of the decay rule (``LFWFunction``, ``LFWHeadsFunction`` on gate logits);
* training with the delta rule (``DFWFunction``).

Gates are sigmoid(N(mean, 1)) ("normal") as a model's projections give them, or constant per channel with
uniformly distributed values ("uniform"), the construction of the reference's own test.
"""
import math

import torch

from t2fw_amd import FastWeightState, LFWFunction, LFWHeadsFunction
from t2fw_amd.functional_dfw import DFWFunction

DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}


def _case(name, kind, dtype, rows, steps, value=64, key=64, heads=1, gates="normal", gate_mean=2.0):
    return {"name": name, "kind": kind, "dtype": dtype, "rows": rows, "steps": steps, "value": value, "key": key,
            "heads": heads, "gates": gates, "gate_mean": gate_mean}


def listed():
    return [
        # one sequence per head of a GPT-2-small batch of 8, a token per call: launch and host latency
        _case("step_small", "step", "float16", 96, 1),
        # the same at serving scale, 4096 sequences of 12 heads: the state streams through memory once per token
        _case("step_serving", "step", "float16", 4096 * 12, 1),
        # prompts of a batch of 8 at GPT-2-small's head shape
        _case("prefill", "prefill", "float16", 96, 1024),
        # the prompt of a single request: few rows, a length that is no multiple of anything
        _case("prefill_request", "prefill", "bfloat16", 12, 333),
        # the headline training step
        _case("train", "train", "float16", 96, 1024),
        # long-context training, slow decay
        _case("train_long", "train", "bfloat16", 128, 8192, gate_mean=3.0),
        # training a layer on [batch, time, heads, channels] projections with gate logits, a ragged length
        _case("train_heads", "train_heads", "bfloat16", 8, 1000, heads=12),
        # full-precision training
        _case("train_float32", "train", "float32", 96, 1024),
        # the largest shape of the reference's test grid: odd widths, gates from 1/64 to 63/64
        _case("train_odd", "train", "float16", 13, 385, value=33, key=17, gates="uniform"),
        # wide heads
        _case("train_wide", "train", "float16", 24, 1024, value=128, key=128),
        # the delta rule in the type that the reference tests it in
        _case("delta_float32", "delta", "float32", 96, 1024),
        # ... and in bf16 with values wider than keys, a ragged length
        _case("delta_wide", "delta", "bfloat16", 48, 777, value=128),
    ]


def _between(rng, lo, hi):
    """A whole number of [lo, hi], uniform in its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    what = rng.choice(["step", "prefill", "train", "train_heads", "train_float32", "train_odd", "train_wide", "delta",
                       "delta_wide"])
    half = rng.choice(["float16", "bfloat16"])
    mean = rng.choice([2.0, 3.0])
    if what == "step":
        c = _case("", "step", half, _between(rng, 12, 49152), 1)
    elif what == "prefill":
        c = _case("", "prefill", half, _between(rng, 4, 128), _between(rng, 16, 4096), gate_mean=mean)
    elif what == "train":
        c = _case("", "train", half, _between(rng, 8, 128), _between(rng, 64, 8192), gate_mean=mean)
    elif what == "train_heads":
        c = _case("", "train_heads", half, rng.randint(1, 8), _between(rng, 64, 1024), heads=rng.choice([4, 8, 12, 16]))
    elif what == "train_float32":
        c = _case("", "train", "float32", _between(rng, 8, 96), _between(rng, 64, 1024), gate_mean=mean)
    elif what == "train_odd":
        width = rng.randint(2, 63)
        c = _case("", "train", rng.choice(["float16", "float32"]), rng.randint(1, 16), _between(rng, 16, 1024), value=width,
                  key=(width + 1) // 2, gates="uniform")
    elif what == "train_wide":
        c = _case("", "train", half, _between(rng, 6, 24), _between(rng, 64, 1024), value=128, key=rng.choice([64, 128]))
    elif what == "delta":
        c = _case("", "delta", rng.choice(["float32", "float16", "bfloat16"]), _between(rng, 8, 96), _between(rng, 64, 1024))
    else:
        c = _case("", "delta", rng.choice(["float32", half]), _between(rng, 6, 24), _between(rng, 64, 1024),
                  value=rng.choice([128, 256]))
    del c["name"]
    return c


def _normal(gen, shape, scale, dtype):
    return torch.randn(shape, generator=gen, device="cuda").mul_(scale).to(dtype)


def _gates(gen, shape, case, dtype, logits=False):
    if case["gates"] == "uniform":
        n = shape[-1]
        g = torch.rand(n, generator=gen, device="cuda") * (1 - 2.0 / n) + 1.0 / n
        return g.expand(shape).to(dtype).contiguous()
    z = torch.randn(shape, generator=gen, device="cuda").add_(case["gate_mean"])
    return (z if logits else torch.sigmoid(z)).to(dtype)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype, kind = DTYPES[case["dtype"]], case["kind"]
    B, T, D, K, H = (case[n] for n in ("rows", "steps", "value", "key", "heads"))
    scale = 1.0 if case["gates"] == "uniform" else 0.125
    state = {"kind": kind}
    if kind == "delta":
        # keys are a distribution over channels times a write strength, as in the reference's test
        k = torch.randn((B, T, K), generator=gen, device="cuda")
        k = torch.softmax(k, dim=-1) * torch.sigmoid(k.mean(dim=-1, keepdim=True))
        ins = (_normal(gen, (B, T, K), 1.0, dtype), k.to(dtype), _normal(gen, (B, T, D), 1.0, dtype),
               _normal(gen, (B, D, K), 1.0, dtype))
        grads = (_normal(gen, (B, T, D), 1.0, dtype), _normal(gen, (B, D, K), 1.0, dtype))
    else:
        lead = (B,) if kind == "step" else (B, T, H) if kind == "train_heads" else (B, T)
        logits = kind == "train_heads"
        x = _normal(gen, lead + (D,), scale, dtype)
        f = _gates(gen, lead + (D,), case, dtype, logits)
        q = _normal(gen, lead + (K,), scale, dtype)
        k = _normal(gen, lead + (K,), scale, dtype)
        fk = _gates(gen, lead + (K,), case, dtype, logits)
        st = (B, H, D, K) if kind == "train_heads" else (B, D, K)
        ins = (x, f, q, k, fk, _normal(gen, st, 1.0 if case["gates"] == "uniform" else 0.1, dtype))
        grads = (_normal(gen, lead + (D,), 1.0, dtype), _normal(gen, st, 0.1, dtype))
    if kind == "step":
        state["layer"] = FastWeightState(D, K).reset(ins[5])
        state["token"] = ins[:5]
    elif kind == "prefill":
        state["inputs"] = ins
    else:
        state["inputs"] = [t.requires_grad_(True) for t in ins]
        state["grads"] = grads
    return state


def run(state):
    kind = state["kind"]
    if kind == "step":
        with torch.no_grad():
            out = state["layer"](*state["token"])
        return out, state["layer"].state
    if kind == "prefill":
        with torch.no_grad():
            return LFWFunction.apply(*state["inputs"])
    ins = state["inputs"]
    if kind == "train":
        out, last = LFWFunction.apply(*ins)
    elif kind == "train_heads":
        out, last = LFWHeadsFunction.apply(*ins, True)
    else:
        out, last = DFWFunction.apply(*ins)
    return (out, last) + torch.autograd.grad((out, last), ins, state["grads"])


def work(case):
    """Bytes: inputs, gradients coming in, results and gradients going out, once each.  Operations per state element
    and step: forward 6 (gate, update, output; delta rule: two products with the state and the update), backward 16
    (adjoint and state recurrences and the reductions of the gradients; delta rule 14)."""
    es = torch.empty(0, dtype=DTYPES[case["dtype"]]).element_size()
    kind, D, K = case["kind"], case["value"], case["key"]
    rows = case["rows"] * case["heads"]
    tokens = rows * case["steps"]
    states = rows * D * K
    if kind in ("step", "prefill"):
        return {"bytes": (tokens * (3 * D + 3 * K) + 2 * states) * es, "flops": 6.0 * tokens * D * K}
    if kind == "delta":
        return {"bytes": (tokens * (4 * D + 4 * K) + 4 * states) * es, "flops": 20.0 * tokens * D * K}
    return {"bytes": (tokens * (6 * D + 6 * K) + 4 * states) * es, "flops": 22.0 * tokens * D * K}


# Largest 2-norm relative error per kind and type, about four times what the present kernels show against the same
# call on float64 tensors.  Measured: one step and odd widths 2.1e-4 (float16), 1.7e-3 (bfloat16), i.e. the rounding of
# what is stored; 64-wide blocks with bf16 operands 4.1e-3 (both types), 8.2e-3 for gate-logit gradients of bfloat16
# tensors (the gates themselves are rounded); delta rule 7.4e-6 (float32, operands as two bf16 terms), 3.7e-4, 3.4e-3.
# The float32 decay rule is within 1.2e-7 when every step is summed in order; 1e-5 is what 32-bit sums in another
# order give after a thousand steps.
TOLERANCE = {
    "step": {"float16": 1e-3, "bfloat16": 7e-3},
    "prefill": {"float16": 1.5e-2, "bfloat16": 1.5e-2},
    "train": {"float32": 1e-5, "float16": 1.5e-2, "bfloat16": 1.5e-2},
    "train_heads": {"float16": 1.5e-2, "bfloat16": 3e-2},
    "delta": {"float32": 3e-5, "float16": 1.5e-3, "bfloat16": 1.4e-2},
}


def tolerance(case):
    if case["kind"] == "train" and case["value"] % 64 and case["dtype"] == "float16":
        return {"rel": 1e-3}
    return {"rel": TOLERANCE[case["kind"]][case["dtype"]]}
