"""The work that a user of this package has it do, as measurable cases: single MoE layers (``ScatterMoEBlock``), one
expert-parallel rank's share (``fused_expert_mlp``) and one projection with adapters (``parallel_linear_lora``), from a
single token to a long skewed batch, forward and forward + backward.

``kind``    block: ScatterMoEBlock; share: fused_expert_mlp on pre-dispatched rows; linear: parallel_linear_lora with gates
``mode``    fwd: no gradients; lora: gradients of the input and of the adapters, expert weights frozen; full: gradients of
            the input, the router and the expert weights (no adapters)
``T``       tokens (share: rows that the exchange delivered);  ``d`` hidden size, ``f`` expert ffn size, ``E`` experts,
            ``k`` experts per token, ``r`` adapter rank (0: none), ``dtype`` bf16 / fp16 / fp32, ``skew`` Zipf-like routing
"""
from __future__ import annotations

import math

import torch

import moe_distributed_training_amd as moe
from moe_distributed_training_amd.megablocks_utils.moe_mlp import LoraViews
from moe_distributed_training_amd.megablocks_utils.router import route_and_sort, sort_assignments

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
ALPHA = 32.0
WIDE = dict(d=4096, f=14336, E=8, k=2)     # the layer of the default benchmark workload
LARGEST_FLOPS = None                        # of the listed cases, set below


def _case(name, kind, mode, T, d, f, E, k, r, dtype="bf16", skew=False):
    return dict(name=name, kind=kind, mode=mode, T=T, d=d, f=f, E=E, k=k, r=r, dtype=dtype, skew=skew)


def listed():
    return [
        # the smallest benchmark configuration, in fp32 (no matrix-core path): bringing a model up, checking numerics
        _case("tiny_fp32_forward", "block", "fwd", 256, 128, 256, 4, 2, 0, "fp32"),
        # a small model's adapter training step, where launches and host work are most of the time
        _case("small_train_lora", "block", "lora", 512, 256, 512, 8, 2, 16),
        # token by token generation for one sequence: two experts' weights are streamed for one row each
        _case("decode_one_token", "block", "fwd", 1, r=0, **WIDE),
        # generation for a batch of sequences with the adapters kept apart from the weights: every expert, a few rows each
        _case("decode_batch_lora", "block", "fwd", 24, r=16, **WIDE),
        # prefill / evaluation of a short prompt
        _case("prefill_short", "block", "fwd", 333, r=0, **WIDE),
        # an adapter step on a short, oddly sized micro-batch in fp16
        _case("train_lora_short_fp16", "block", "lora", 777, r=16, dtype="fp16", **WIDE),
        # the default benchmark workload: one sequence of 4096 tokens per micro-batch, rank 16
        _case("train_lora", "block", "lora", 4096, r=16, **WIDE),
        # full fine-tuning of the same layer
        _case("train_full", "block", "full", 4096, r=0, **WIDE),
        # four sequences with skewed routing
        _case("train_lora_long_skewed", "block", "lora", 16384, r=16, skew=True, **WIDE),
        # one expert-parallel rank's share: two resident experts, rows already dispatched
        _case("expert_share_lora", "share", "lora", 8192, 4096, 14336, 2, 1, 16),
        # many narrow experts, wide top-k: most groups are small and ragged
        _case("many_experts_train_lora", "block", "lora", 2048, 2048, 1024, 64, 8, 16),
        # one projection through the per-projection entry point, rank 32, gate-weighted combine
        _case("linear_lora_gates", "linear", "lora", 1500, 4096, 4096, 8, 2, 32),
    ]


def _experts_touched(T, E, k):
    return E * (1.0 - (1.0 - k / E) ** T) if E > 1 else 1.0


def _flops(c):
    R = c["T"] * c["k"]
    d, f, r = c["d"], c["f"], c["r"]
    bwd = c["mode"] != "fwd"
    if c["kind"] == "linear":
        return (4 if bwd else 2) * R * d * f + (8 if bwd else 2) * R * r * (d + f)
    n = 6 * R * d * f * (1 if not bwd else 2 if c["mode"] == "lora" else 3)
    n += 6 * R * r * (d + f) * (4 if bwd else 1)
    if c["kind"] == "block":
        n += 2 * c["T"] * d * c["E"] * (1 if not bwd else 2 if c["mode"] == "lora" else 3)
    return n


LARGEST_FLOPS = max(_flops(c) for c in listed())


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges: the wide layer from 1 to 16384 tokens in each direction, narrow layers, many
    experts, a rank's share and single projections; never more work than the largest listed case."""
    while True:
        what = rng.choice(["tiny", "small", "decode", "wide", "wide", "full", "share", "many", "linear"])
        dt = rng.choice(["bf16", "bf16", "fp16"])
        if what == "tiny":
            c = _case("", "block", rng.choice(["fwd", "full"]), _log_int(rng, 16, 512), rng.randrange(32, 257), rng.randrange(32, 513),
                      rng.randrange(2, 9), 2, 0, "fp32")
        elif what == "small":
            c = _case("", "block", rng.choice(["fwd", "lora", "full"]), _log_int(rng, 16, 4096), 64 * rng.randrange(2, 17),
                      64 * rng.randrange(2, 33), rng.randrange(2, 17), 2, 0, dt)
        elif what == "decode":
            c = _case("", "block", "fwd", _log_int(rng, 1, 128), r=rng.choice([0, 0, 16]), dtype=dt, **WIDE)
        elif what == "wide":
            c = _case("", "block", rng.choice(["fwd", "lora", "lora"]), _log_int(rng, 128, 16384), r=rng.choice([8, 16, 16, 32]), dtype=dt,
                      skew=rng.random() < 0.3, **WIDE)
        elif what == "full":
            c = _case("", "block", "full", _log_int(rng, 256, 8192), r=0, dtype=dt, **WIDE)
        elif what == "share":
            c = _case("", "share", rng.choice(["fwd", "lora"]), _log_int(rng, 64, 16384), 4096, 14336, rng.choice([1, 2, 4]), 1, 16, dt)
        elif what == "many":
            c = _case("", "block", rng.choice(["fwd", "lora", "full"]), _log_int(rng, 64, 8192), 64 * rng.randrange(8, 49),
                      64 * rng.randrange(6, 25), rng.choice([16, 32, 64, 96]), rng.randrange(2, 9), 16, dt)
        else:
            c = _case("", "linear", rng.choice(["fwd", "lora"]), _log_int(rng, 32, 8192), 64 * rng.randrange(8, 81), 64 * rng.randrange(8, 81),
                      rng.randrange(2, 17), rng.randrange(1, 5), rng.choice([8, 16, 32, 64]), dt)
        if c["kind"] == "linear":
            c["k"] = min(c["k"], c["E"])
        if what == "small" and c["mode"] != "full":
            c["r"] = rng.choice([0, 8, 16, 32]) if c["mode"] == "fwd" else rng.choice([8, 16, 32])
        if c["mode"] == "full":
            c["r"] = 0
        if _flops(c) <= LARGEST_FLOPS:
            del c["name"]
            return c


def work(case):
    b = 4 if case["dtype"] == "fp32" else 2
    T, d, f, E, k, r = (case[n] for n in ("T", "d", "f", "E", "k", "r"))
    nproj = 1 if case["kind"] == "linear" else 3
    weights = nproj * d * f * _experts_touched(T, E, k)
    adapters = nproj * r * (d + f) * E
    rows_in, rows_out = T * d, T * (f if case["kind"] == "linear" else d)
    n = weights + adapters + rows_in + rows_out + (E * d if case["kind"] == "block" else 0)
    if case["mode"] != "fwd":
        n += rows_out + rows_in + adapters                 # gradient of the output in; of the input and of the adapters out
        if case["mode"] == "full":
            n += nproj * d * f * E + E * d
    return {"bytes": int(n * b), "flops": int(_flops(case))}


def tolerance(case):
    # About four times what the path shows against the same layer in 32-bit arithmetic (fp32: in 64-bit) on the same inputs:
    # bf16 3.9e-3 / 4.5e-2, fp16 4.9e-4 / 3.8e-3, fp32 4.2e-7 forward.  Skewed routing puts large entries into one column of the
    # router's weight, so that column of the input gradient is a difference of large terms (bf16 0.27 of its scale).
    rel, biggest = {"fp32": (5e-6, 5e-5), "fp16": (2e-3, 2e-2), "bf16": (1.5e-2, 1.8e-1)}[case["dtype"]]
    return {"rel": rel, "max": 5 * biggest if case["skew"] else biggest}


def prepare(case, seed):
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)
    dt = DTYPES[case["dtype"]]
    T, d, f, E, k, r, mode = (case[n] for n in ("T", "d", "f", "E", "k", "r", "mode"))
    train = mode != "fwd"

    def normal(*shape, std=1.0):
        return torch.empty(shape, dtype=dt, device=dev).normal_(0.0, std, generator=g)

    st = dict(case=case, x=normal(T, d), params={})
    x = st["x"]
    if case["kind"] == "block":
        block = moe.ScatterMoEBlock(d, f, E, top_k=k, lora_r=r, lora_alpha=ALPHA, dtype=dt, device=dev)
        with torch.no_grad():
            for p in block.parameters():
                p.normal_(0.0, 0.02, generator=g)
            if case["skew"]:
                # per-expert logit offsets (about the log of a Zipf 1.2 law) along one input direction
                pmf = torch.tensor([1.0 / (i + 1) ** 1.2 for i in range(E)])
                x[:, 0] = 1.0
                block.router[:, 0] = (2.2 * torch.log(pmf / pmf.sum())).to(dev, dt)
        block.requires_grad_(False)
        if mode == "lora":
            st["params"] = {n: p for n, p in block.named_parameters() if n.startswith("lora_")}
        elif mode == "full":
            st["params"] = dict(block.named_parameters())
        st["block"] = block
        out_cols = d
    elif case["kind"] == "share":
        p = torch.tensor([1.0 + 0.2 * (E - 1 - e) for e in range(E)], device=dev)
        experts = torch.multinomial(p / p.sum(), T, replacement=True, generator=g)
        _, st["ssi"], _, st["offsets"], _ = sort_assignments(experts.int(), E)
        st["w1"], st["w2"], st["w3"] = (normal(E, f, d, std=0.02) for _ in range(3))
        st["lora"] = LoraViews(normal(E, d, r, std=0.02), normal(E, r, f, std=0.02), normal(E, d, r, std=0.02),
                               normal(E, r, f, std=0.02), normal(E, f, r, std=0.02), normal(E, r, d, std=0.02))
        if train:
            st["params"] = dict(st["lora"]._asdict())
        out_cols = d
    else:
        # f is the projection's output size; the expert choice comes from a router, as in a layer
        rt = route_and_sort(x, normal(E, d, std=0.02), k)
        st["sei"], st["ssi"] = rt.sorted_expert_idxs, rt.sorted_scattered_idxs
        st["pbi"], st["offsets"] = moe.padded_block_indices(st["sei"], E)
        st["gates"] = rt.weights.to(dt)
        st["w"] = normal(E, f, d, std=0.02).permute(0, 2, 1)
        a, b = normal(E, d, r, std=0.02), normal(E, r, f, std=0.02)
        st["a"], st["b"] = a, b
        if train:
            st["params"] = dict(a=a, b=b, gates=st["gates"])
        out_cols = f
    if train:
        x.requires_grad_(True)
        for p in st["params"].values():
            p.requires_grad_(True)
        st["dout"] = normal(T, out_cols)
    return st


def _forward(st):
    case = st["case"]
    if case["kind"] == "block":
        return st["block"](st["x"])[0]
    if case["kind"] == "share":
        return moe.fused_expert_mlp(st["x"], st["w1"], st["w2"], st["w3"], 1, st["ssi"], st["offsets"], st["lora"], ALPHA)
    return moe.parallel_linear_lora(st["x"], st["w"], st["a"], st["b"], case["r"], ALPHA, case["k"], st["sei"], st["ssi"], st["pbi"],
                                    st["offsets"], gates=st["gates"])


def run(state):
    """One forward pass, or one forward and backward pass with the gradients it leaves."""
    if state["case"]["mode"] == "fwd":
        with torch.no_grad():
            return _forward(state)
    state["x"].grad = None
    for p in state["params"].values():
        p.grad = None
    out = _forward(state)
    out.backward(state["dout"])
    grads = {n: p.grad for n, p in state["params"].items()}
    return dict(out=out.detach(), dx=state["x"].grad, **grads)
