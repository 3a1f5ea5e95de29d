"""Workloads of the 2-simplicial attention operator that stand for what its users run.

A case is one problem: element type, batch, sequence length, heads, head_dim, the two windows, the
biases, the window convention and how the five inputs lie in memory.  ``mode`` is "forward" (the
module called on tensors that need no gradients: inference, prefill) or "train" (the module's
forward and the backward to all five inputs).  Both go through ``TwoSimplicialAttention``.

``listed()`` holds fixed cases, ``draw(rng)`` more of the same ranges.
"""
import math

import torch

import simplical_attn_amd as sa

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}

# The largest listed problem: 35.2 TFLOP of matrix products in 16 bits.
_MOST_FLOPS = 3.53e13
_MOST_ELEMENTS = 8 * 32768 * 128        # of one tensor


def _case(mode, dtype, B, N, H, D, w1, w2, k2_bias=0.0, v2_bias=0.0, inclusive=True, packed=False, qk_std=1.0):
    return {"mode": mode, "dtype": dtype, "B": B, "N": N, "H": H, "D": D, "w1": w1, "w2": w2,
            "k2_bias": k2_bias, "v2_bias": v2_bias, "inclusive": inclusive, "packed": packed, "qk_std": qk_std}


def listed():
    rows = (
        # a unit-test sized call: nothing but latency, launches and the host path
        ("tiny_forward", _case("forward", "bf16", 1, 32, 1, 16, 16, 16)),
        # the fp32 plumbing configuration: eight query blocks, latency again, in fp32
        ("small_fp32_forward", _case("forward", "fp32", 1, 128, 2, 64, 32, 16)),
        # the base shape of the scaling sweeps, as one layer of a small training run
        ("sweep_base_train", _case("train", "bf16", 2, 256, 4, 64, 32, 32)),
        # sequence lengths as batches of text have them, inputs that are views of one fused projection
        # [B,N,5,H,D], fp16, biases on K' and V'
        ("ragged_packed_fp16_train", _case("train", "fp16", 3, 777, 6, 64, 100, 20, 0.1, 0.2, packed=True)),
        # both windows wide: the widest point of the window sweep
        ("wide_windows_train", _case("train", "bf16", 2, 512, 4, 64, 256, 256)),
        # head_dim between the powers of two, half-open windows
        ("head_dim_96_train", _case("train", "bf16", 1, 2048, 8, 96, 256, 32, inclusive=False)),
        # the largest head_dim
        ("head_dim_256_train", _case("train", "bf16", 1, 4096, 8, 256, 512, 32)),
        # a middle-sized training layer, head_dim 64
        ("middle_train", _case("train", "bf16", 2, 2048, 8, 64, 512, 32)),
        # the same layer in full precision
        ("middle_fp32_train", _case("train", "fp32", 2, 2048, 8, 64, 512, 32)),
        # prefill at the headline shape
        ("headline_forward", _case("forward", "bf16", 1, 8192, 16, 128, 512, 32)),
        # the headline: a training step of a long-sequence layer
        ("headline_train", _case("train", "bf16", 1, 8192, 16, 128, 512, 32)),
        # the largest: four times the sequence, both windows doubled
        ("long_train", _case("train", "bf16", 1, 32768, 8, 128, 1024, 64, qk_std=0.5)),
    )
    return [dict(case, name=name) for name, case in rows]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    while True:
        mode = "forward" if rng.random() < 0.4 else "train"
        dtype = rng.choice(("bf16", "bf16", "bf16", "fp16", "fp32"))
        D = rng.choice((16, 32, 64, 64, 64, 80, 96, 128, 128, 128, 256)) if dtype != "fp32" else \
            rng.choice((16, 32, 64, 64, 96, 128))
        B, H = _log_int(rng, 1, 8), _log_int(rng, 1, 32)
        N = _log_int(rng, 32, 32768)
        if rng.random() < 0.5 and N >= 64:
            N = N // 64 * 64                          # half of the lengths are padded to blocks, half are as they come
        w1 = _log_int(rng, 16, 1024)
        w2 = _log_int(rng, 8, min(w1, 256))
        if rng.random() < 0.5:                        # half of the windows are the round ones of configurations
            w1, w2 = max(16, w1 // 16 * 16), max(8, w2 // 8 * 8)
        biased = rng.random() < 0.25
        c = _case(mode, dtype, B, N, H, D, w1, w2, round(rng.uniform(-0.5, 0.5), 2) if biased else 0.0,
                  round(rng.uniform(-0.5, 0.5), 2) if biased else 0.0, rng.random() < 0.75, rng.random() < 0.25,
                  0.5 if rng.random() < 0.3 else 1.0)
        # fp32 products run at a sixteenth of the 16-bit rate; the softmax costs the same per triple whatever the
        # head_dim; head_dims off 32, 64 and 128 are used at middle sizes
        most = (_MOST_FLOPS / 16 if dtype == "fp32" else _MOST_FLOPS) * min(D, 128) / 128
        if D == 256:
            most /= 4
        if D in (80, 96):
            most = 2.2e11
        if work(c)["flops"] <= most and B * N * H * D <= _MOST_ELEMENTS:
            return c


def _triples(c):
    """Valid (i, j, k) triples of one case: sum over queries of the two windows' sizes."""
    N = c["N"]
    r1, r2 = (min(w if c["inclusive"] else w - 1, N - 1) for w in (c["w1"], c["w2"]))
    ramp = max(r1, r2)
    head = sum((min(i, r1) + 1) * (min(i, r2) + 1) for i in range(ramp))
    return c["B"] * c["H"] * (head + (N - ramp) * (r1 + 1) * (r2 + 1))


def prepare(case, seed):
    """Inputs as projections leave them: independent normal values, of unit or half unit scale for q, k1, k2."""
    c, dev = case, torch.device("cuda:0")
    B, N, H, D, dtype = c["B"], c["N"], c["H"], c["D"], _DTYPES[c["dtype"]]
    g = torch.Generator(device=dev).manual_seed(seed)

    def normal(*shape):
        return torch.randn(*shape, generator=g, device=dev, dtype=torch.float32)

    std = (c["qk_std"],) * 3 + (1.0, 1.0)
    if c["packed"]:
        inputs = (normal(B, N, 5, H, D) * torch.tensor(std, device=dev).view(5, 1, 1)).to(dtype).unbind(2)
    else:
        inputs = [(normal(B, N, H, D) * s).to(dtype) for s in std]
    state = {"attn": sa.TwoSimplicialAttention(D, c["w1"], c["w2"], None, c["k2_bias"], c["v2_bias"],
                                               window_inclusive=c["inclusive"])}
    if c["mode"] == "train":
        state["inputs"] = [t.detach().requires_grad_(True) for t in inputs]
        state["dout"] = normal(B, N, H, D).to(dtype)
    else:
        state["inputs"] = list(inputs)
    return state


def run(state):
    out = state["attn"](*state["inputs"])
    if "dout" not in state:
        return out
    grads = torch.autograd.grad(out, state["inputs"], state["dout"])
    return (out.detach(), *grads)


def work(case):
    """Matrix products of the valid triples only, 2 per multiply-add: 4 D T forward (logits, values), 12 D T
    backward (both factors again and the four gradient contractions)."""
    c = case
    size = {"bf16": 2, "fp16": 2, "fp32": 4}[c["dtype"]]
    elements = c["B"] * c["N"] * c["H"] * c["D"]
    train = c["mode"] == "train"
    return {"bytes": elements * size * (12 if train else 6), "flops": (16 if train else 4) * c["D"] * _triples(c)}


def tolerance(case):
    """fp32 products and sums to 1e-5; in 16 bits the products q*k2 and dout*v2 and the softmax weights are
    rounded to the element type before they are multiplied on."""
    return {"rel": {"fp32": 1e-5, "fp16": 2e-3, "bf16": 1e-2}[case["dtype"]]}
