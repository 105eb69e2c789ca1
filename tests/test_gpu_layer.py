"""Whole-path parity: router -> sort -> fused expert MLP (LoRA, SwiGLU) -> combine, forward and backward, against the
fp32 CPU oracle on the same seeded inputs.  Routing indices must be identical; bf16 outputs and gradients within
max rel err 1e-2 (the specification's bar)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


from _metrics import rel, rel_per_expert


# Groups of one to a few rows, measured on their own scale: an adapter gradient is then a product of values that each
# went through bf16 storage (dh, gate / up, dgate / dup, the low-rank interim, the result: five roundings of up to 2^-9
# in a row, as in the reference, whose tensors are bf16 too) with no sum over many rows to average them out, so the
# worst element of the worst slice sits at about 1 %, not well below it as for groups of hundreds of rows.
TINY_GROUP_TOL = 1.5e-2


def check_expert_grads(got, want, what, tol=1e-2):
    """Adapter / weight gradients (first dimension = expert): each expert's slice against its own scale; the RMS
    figure beside the maximum catches an error spread thinly over a slice."""
    mx, rms = rel_per_expert(got, want, with_rms=True)
    assert mx < tol and rms < tol, f"{what}: per-expert max rel err {mx:.4g}, rms rel err {rms:.4g}"


def _make(T, d, f, E, r, dtype, seed=0, lora_std=0.02):
    g = torch.Generator().manual_seed(seed)
    rn = lambda *s, std=1.0: (torch.randn(*s, generator=g) * std).to(dtype)
    x, wg = rn(T, d), rn(E, d, std=0.02)
    w1, w2, w3 = rn(E, f, d, std=0.02), rn(E, f, d, std=0.02), rn(E, f, d, std=0.02)
    lora = None
    if r:
        lora = {"w1": (rn(E, d, r, std=lora_std), rn(E, r, f, std=lora_std)), "w3": (rn(E, d, r, std=lora_std), rn(E, r, f, std=lora_std)),
                "w2": (rn(E, f, r, std=lora_std), rn(E, r, d, std=lora_std))}
    return x, wg, w1, w2, w3, lora, rn(T, d)


def _tiles(R, E, d, f):
    """Tile sizes of the layer's four grouped GEMM launches: gate/up, h W2, dh, dX."""
    from moe_distributed_training_amd._lib import lib
    return tuple(lib.moe_gemm_debug_tile(R, E, K, N, pair, nseg) for K, N, pair, nseg in ((d, f, 1, 1), (f, d, 0, 1), (d, f, 0, 1), (f, d, 0, 2)))


def _views(lora, dev):
    from moe_distributed_training_amd.megablocks_utils.moe_mlp import LoraViews
    t = {n: (a.to(dev).requires_grad_(True), b.to(dev).requires_grad_(True)) for n, (a, b) in lora.items()}
    return t, LoraViews(t["w1"][0], t["w1"][1], t["w3"][0], t["w3"][1], t["w2"][0], t["w2"][1])


def test_config1_tiny_fp32_forward(dev, oracle):
    """T=256, d=128, f=256, E=4, top-2, fp32, seed 0, forward only (the CPU-runnable configuration)."""
    import moe_distributed_training_amd as moe
    x, wg, w1, w2, w3, _, _ = _make(256, 128, 256, 4, 0, torch.float32, seed=0)
    ref, aux = oracle.moe_block(x, wg, w1, w2, w3, 2)
    out, ew, ei = moe.moe_layer_forward(x.to(dev), wg.to(dev), w1.to(dev), w2.to(dev), w3.to(dev), 2)
    assert torch.equal(ei.cpu().long(), aux["indices"])
    assert torch.allclose(ew.cpu(), aux["weights"], atol=1e-6)
    assert rel(out, ref) < 2e-5


@pytest.mark.parametrize("T,d,f,E,r", [(512, 256, 512, 8, 16), (300, 128, 192, 4, 8), (1024, 512, 1024, 8, 0), (64, 64, 64, 2, 16)])
def test_layer_fwd_bwd_bf16(dev, oracle, T, d, f, E, r):
    import moe_distributed_training_amd as moe
    k, alpha = 2, 32.0
    x, wg, w1, w2, w3, lora, dout = _make(T, d, f, E, r, torch.bfloat16, seed=T)
    xo = x.float().requires_grad_(True)
    lo = None if lora is None else {n: (a.float().requires_grad_(True), b.float().requires_grad_(True)) for n, (a, b) in lora.items()}
    ref, aux = oracle.moe_block(xo, wg.float(), w1.float(), w2.float(), w3.float(), k, lo, alpha)
    ref.backward(dout.float())
    xg = x.to(dev).requires_grad_(True)
    lt, views = (None, None) if lora is None else _views(lora, dev)
    full = lora is None    # no adapters: full fine-tuning, the stored expert weights take gradients
    wd = [w.to(dev).requires_grad_(full) for w in (w1, w2, w3)]
    out, ew, ei = moe.moe_layer_forward(xg, wg.to(dev), wd[0], wd[1], wd[2], k, views, alpha)
    out.backward(dout.to(dev))
    assert torch.equal(ei.cpu().long(), aux["indices"])
    assert rel(out, ref) < 1e-2 and rel(xg.grad, xo.grad) < 1e-2
    if full:
        wo = [w.float().requires_grad_(True) for w in (w1, w2, w3)]
        xo2 = x.float().requires_grad_(True)
        ref2, _ = oracle.moe_block(xo2, wg.float(), wo[0], wo[1], wo[2], k, None, alpha)
        ref2.backward(dout.float())
        for n, a, b in zip(("w1", "w2", "w3"), wd, wo):
            assert a.grad is not None and a.grad.shape == b.grad.shape
            check_expert_grads(a.grad, b.grad, f"dW {n}")
    if lora is not None:
        for n in ("w1", "w3", "w2"):
            check_expert_grads(lt[n][0].grad, lo[n][0].grad, f"dA {n}")
            check_expert_grads(lt[n][1].grad, lo[n][1].grad, f"dB {n}")
    # run-to-run determinism (activation checkpointing replays the forward inside backward)
    out2, _, ei2 = moe.moe_layer_forward(xg, wg.to(dev), wd[0], wd[1], wd[2], k, views, alpha)
    assert torch.equal(out2, out) and torch.equal(ei2, ei)


@pytest.mark.parametrize("T,d,f,E,r", [(512, 256, 512, 8, 16), (700, 128, 320, 4, 0), (900, 192, 256, 8, 32), (640, 192, 256, 4, 80)])
def test_layer_fwd_bwd_fp16(dev, oracle, T, d, f, E, r):
    """The reference's fp16 switch (megablocks_utils/shard_moe_utils.py:29-30,43-44): the whole layer in IEEE half runs the
    same matrix-core kernels as bf16 (every grouped GEMM launch is counted; rank 80: five rank chunks, the slabs of the
    gate/up and dh launches found by base and stride); fp16 carries 3 more mantissa bits, so the bound is tighter than
    bf16's."""
    import moe_distributed_training_amd as moe
    from moe_distributed_training_amd._lib import lib
    k, alpha, tol = 2, 32.0, 3e-3
    x, wg, w1, w2, w3, lora, dout = _make(T, d, f, E, r, torch.float16, seed=T)
    xo = x.float().requires_grad_(True)
    lo = None if lora is None else {n: (a.float().requires_grad_(True), b.float().requires_grad_(True)) for n, (a, b) in lora.items()}
    full = lora is None
    wo = [w.float().requires_grad_(full) for w in (w1, w2, w3)]
    ref, aux = oracle.moe_block(xo, wg.float(), wo[0], wo[1], wo[2], k, lo, alpha)
    ref.backward(dout.float())
    xg = x.to(dev).requires_grad_(True)
    lt, views = (None, None) if lora is None else _views(lora, dev)
    wd = [w.to(dev).requires_grad_(full) for w in (w1, w2, w3)]
    n0 = lib.moe_gemm_debug_launch_count()
    out, ew, ei = moe.moe_layer_forward(xg, wg.to(dev), wd[0], wd[1], wd[2], k, views, alpha)
    out.backward(dout.to(dev))
    assert lib.moe_gemm_debug_launch_count() - n0 == 4, "pair, h W2, dh and dX GEMMs on the matrix cores"
    assert out.dtype == torch.float16 and xg.grad.dtype == torch.float16
    assert torch.equal(ei.cpu().long(), aux["indices"])
    assert rel(out, ref) < tol and rel(xg.grad, xo.grad) < tol
    if full:
        for n, a, b in zip(("w1", "w2", "w3"), wd, wo):
            check_expert_grads(a.grad, b.grad, f"dW {n}", tol)
    else:
        for n in ("w1", "w3", "w2"):
            check_expert_grads(lt[n][0].grad, lo[n][0].grad, f"dA {n}", tol)
            check_expert_grads(lt[n][1].grad, lo[n][1].grad, f"dB {n}", tol)


@pytest.mark.parametrize("E,k,r", [(96, 4, 16), (16, 8, 16), (80, 3, 0)])
def test_layer_many_experts_and_wider_top_k(dev, oracle, E, k, r):
    """More than 8 experts (router in groups of 16), more than 64 (group lookup in blocks of 64 in every grouped kernel),
    top-k above 2 (fan-out k in the gathers and the combine); most groups hold a handful of rows, some none."""
    import moe_distributed_training_amd as moe
    T, d, f, alpha = 300, 128, 256, 32.0
    x, wg, w1, w2, w3, lora, dout = _make(T, d, f, E, r, torch.bfloat16, seed=E + k)
    wg = wg * 50      # well separated router scores: the selection does not hinge on the last bits of the logits
    xo = x.float().requires_grad_(True)
    lo = None if lora is None else {n: (a.float().requires_grad_(True), b.float().requires_grad_(True)) for n, (a, b) in lora.items()}
    ref, aux = oracle.moe_block(xo, wg.float(), w1.float(), w2.float(), w3.float(), k, lo, alpha)
    ref.backward(dout.float())
    xg = x.to(dev).requires_grad_(True)
    lt, views = (None, None) if lora is None else _views(lora, dev)
    full = lora is None
    wd = [w.to(dev).requires_grad_(full) for w in (w1, w2, w3)]
    out, ew, ei = moe.moe_layer_forward(xg, wg.to(dev), wd[0], wd[1], wd[2], k, views, alpha)
    out.backward(dout.to(dev))
    assert torch.equal(ei.cpu().long(), aux["indices"])
    assert rel(out, ref) < 1e-2 and rel(xg.grad, xo.grad) < 1e-2
    if full:
        wo = [w.float().requires_grad_(True) for w in (w1, w2, w3)]
        ref2, _ = oracle.moe_block(x.float(), wg.float(), wo[0], wo[1], wo[2], k, None, alpha)
        ref2.backward(dout.float())
        for n, a, b in zip(("w1", "w2", "w3"), wd, wo):
            check_expert_grads(a.grad, b.grad, f"dW {n}", TINY_GROUP_TOL)
    else:
        for n in ("w1", "w3", "w2"):
            check_expert_grads(lt[n][0].grad, lo[n][0].grad, f"dA {n}", TINY_GROUP_TOL)
            check_expert_grads(lt[n][1].grad, lo[n][1].grad, f"dB {n}", TINY_GROUP_TOL)


@pytest.mark.parametrize("E,k", [(16, 8), (24, 2), (64, 4), (80, 3), (104, 2)])
def test_layer_many_experts_router_gradient(dev, oracle, E, k):
    """The router's weight with a gradient, for each width of its kernel, and above the 96 experts that the matrix-core router takes."""
    import moe_distributed_training_amd as moe
    T, d, f = 200, 128, 64
    x, wg, w1, w2, w3, _, dout = _make(T, d, f, E, 0, torch.bfloat16, seed=E)
    wg = wg * 20
    xo, wgo = x.float().requires_grad_(True), wg.float().requires_grad_(True)
    ref, aux = oracle.moe_block(xo, wgo, w1.float(), w2.float(), w3.float(), k, None, 32.0)
    ref.backward(dout.float())
    xg, wgg = x.to(dev).requires_grad_(True), wg.to(dev).requires_grad_(True)
    out, _, ei = moe.moe_layer_forward(xg, wgg, w1.to(dev), w2.to(dev), w3.to(dev), k, None, 32.0)
    out.backward(dout.to(dev))
    assert torch.equal(ei.cpu().long(), aux["indices"])
    assert rel(out, ref) < 1e-2 and rel(xg.grad, xo.grad) < 1e-2
    assert rel(wgg.grad, wgo.grad) < 1e-2


@pytest.mark.parametrize("T,d,f,E,r", [(384, 256, 512, 4, r) for r in (32, 24, 48, 64, 72, 128, 144)] + [(900, 512, 4096, 8, 32), (900, 512, 4096, 8, 24)])
def test_layer_rank_above_16_adapters(dev, oracle, T, d, f, E, r):
    """Adapter rank above 16: up to 128 the fused launches take the adapter as 16-wide rank chunks (24, 72: the last
    chunk partly filled; 48, 72: an odd number of chunks; above 32 the gate/up launch finds its slabs by base and
    stride); above that the layer runs as router + sort + the three grouped calls + combine.  All gradients against
    the oracle.  The small layer's launches of up to four slabs take 128 x 128 tiles, the larger one's 256 x 256."""
    import moe_distributed_training_amd as moe
    k, alpha = 2, 64.0
    assert set(_tiles(T * k, E, d, f)) == {128 if T < 900 else 256}
    x, wg, w1, w2, w3, lora, dout = _make(T, d, f, E, r, torch.bfloat16, seed=5)
    xo = x.float().requires_grad_(True)
    lo = {n: (a.float().requires_grad_(True), b.float().requires_grad_(True)) for n, (a, b) in lora.items()}
    ref, aux = oracle.moe_block(xo, wg.float(), w1.float(), w2.float(), w3.float(), k, lo, alpha)
    ref.backward(dout.float())
    xg = x.to(dev).requires_grad_(True)
    lt, views = _views(lora, dev)
    from moe_distributed_training_amd._lib import lib
    n0 = lib.moe_gemm_debug_launch_count()
    out, ew, ei = moe.moe_layer_forward(xg, wg.to(dev), w1.to(dev), w2.to(dev), w3.to(dev), k, views, alpha)
    out.backward(dout.to(dev))
    # every projection's GEMM runs on the matrix cores at any of these ranks: the fused layer's four launches up to rank 128,
    # three forward and three input-gradient launches of the per-projection route above it
    assert lib.moe_gemm_debug_launch_count() - n0 == (4 if r <= 128 else 6)
    assert torch.equal(ei.cpu().long(), aux["indices"])
    assert rel(out, ref) < 1e-2 and rel(xg.grad, xo.grad) < 1e-2
    for n in ("w1", "w3", "w2"):
        check_expert_grads(lt[n][0].grad, lo[n][0].grad, f"dA {n}")
        check_expert_grads(lt[n][1].grad, lo[n][1].grad, f"dB {n}")


def test_layer_expert_weights_output_carries_grad(dev, oracle):
    """A loss that also uses the returned expert weights (an auxiliary term): their gradient joins the combine's
    d_gates on the way into the router, and a loss on the weights alone works without an output gradient."""
    import moe_distributed_training_amd as moe
    T, d, f, E, r, k = 256, 128, 256, 4, 0, 2
    x, wg, w1, w2, w3, _, dout = _make(T, d, f, E, r, torch.bfloat16, seed=9)
    coef = torch.randn(T, k, generator=torch.Generator().manual_seed(1))
    for use_out in (True, False):
        xo = x.float().requires_grad_(True)
        wgo = wg.float().requires_grad_(True)
        ref, aux = oracle.moe_block(xo, wgo, w1.float(), w2.float(), w3.float(), k, None, 1.0)
        loss = (aux["weights"] * coef).sum() + ((ref * dout.float()).sum() if use_out else 0.0)
        loss.backward()
        xg = x.to(dev).requires_grad_(True)
        wgg = wg.to(dev).requires_grad_(True)
        out, ew, ei = moe.moe_layer_forward(xg, wgg, w1.to(dev), w2.to(dev), w3.to(dev), k, None, 1.0)
        loss = (ew * coef.to(dev)).sum() + ((out.float() * dout.to(dev).float()).sum() if use_out else 0.0)
        loss.backward()
        assert torch.equal(ei.cpu().long(), aux["indices"])
        assert rel(xg.grad, xo.grad) < 1e-2 and rel(wgg.grad, wgo.grad) < 1e-2


def test_block_loaded_from_checkpoint_matches_transformers(dev, tmp_path):
    """A Mixtral-style safetensors checkpoint (per-expert w1 / w3 (f, d), w2 (d, f)) ingested into the fused layout:
    the block's output agrees with transformers' MixtralSparseMoeBlock holding the same tensors."""
    import json, os
    from safetensors.torch import save_file
    from transformers import MixtralConfig
    from transformers.models.mixtral.modeling_mixtral import MixtralSparseMoeBlock
    from moe_distributed_training_amd.megablocks_utils import checkpoint as ck
    from moe_distributed_training_amd.megablocks_utils.moe_mlp import ScatterMoEBlock
    E, d, f, k, T = 4, 128, 256, 2, 96
    g = torch.Generator().manual_seed(21)
    p = "model.layers.3.block_sparse_moe"
    t = {f"{p}.gate.weight": (torch.randn(E, d, generator=g) * 0.3).bfloat16()}
    for e in range(E):
        t[f"{p}.experts.{e}.w1.weight"] = (torch.randn(f, d, generator=g) * 0.1).bfloat16()
        t[f"{p}.experts.{e}.w2.weight"] = (torch.randn(d, f, generator=g) * 0.1).bfloat16()
        t[f"{p}.experts.{e}.w3.weight"] = (torch.randn(f, d, generator=g) * 0.1).bfloat16()
    save_file(t, os.path.join(tmp_path, "model-00001-of-00001.safetensors"))
    with open(os.path.join(tmp_path, ck.FILE_SAFETENSOR_INDEX), "w") as fh:
        json.dump({"weight_map": {key: "model-00001-of-00001.safetensors" for key in t}}, fh)
    block = ScatterMoEBlock(d, f, E, top_k=k, dtype=torch.bfloat16, device=dev)
    ck.load_moe_block(block, str(tmp_path), "model.layers.3")
    cfg = MixtralConfig(hidden_size=d, intermediate_size=f, num_local_experts=E, num_experts_per_tok=k,
                        num_hidden_layers=1, num_attention_heads=4, num_key_value_heads=4, vocab_size=32)
    hf = MixtralSparseMoeBlock(cfg).eval()
    with torch.no_grad():
        hf.gate.weight.copy_(t[f"{p}.gate.weight"].float())
        for e in range(E):
            hf.experts.gate_up_proj[e].copy_(torch.cat([t[f"{p}.experts.{e}.w1.weight"], t[f"{p}.experts.{e}.w3.weight"]]).float())
            hf.experts.down_proj[e].copy_(t[f"{p}.experts.{e}.w2.weight"].float())
    x = torch.randn(2, T // 2, d, generator=g).bfloat16()
    with torch.no_grad():
        ref = hf(x.float())
        ref = ref[0] if isinstance(ref, tuple) else ref
        out, none = block(x.to(dev))
    assert none is None and out.shape == x.shape
    assert rel(out.view(-1, d), ref.view(-1, d)) < 1e-2


def test_reference_caller_both_modes(dev, oracle):
    """scattermoe_permute_and_compute with the reference's storage layout and _lora_pointers tuples, in the
    expert-parallel mode (fan-out 1, scattered output) and the tensor-parallel mode (fan-out k, grouped output),
    bf16 (fused kernels) and fp32 (the three generic calls)."""
    import moe_distributed_training_amd as moe
    from moe_distributed_training_amd.megablocks_utils.moe_mlp import get_mlp_weights_lora
    torch.manual_seed(7)
    T, d, f, E, k, r, alpha = 200, 128, 192, 4, 2, 16, 16.0
    for dtype, tol in ((torch.bfloat16, 1e-2), (torch.float32, 3e-5)):
        w = {n: (torch.randn(E * f, d) * 0.05).to(dtype) for n in ("w1", "w2", "w3")}
        lA = {n: (torch.randn(E * d, r) * 0.05).to(dtype) for n in w}      # lora_A.weight, stored transposed
        lB = {n: (torch.randn(E * f, r) * 0.05).to(dtype) for n in w}      # lora_B.weight
        views = {n: get_mlp_weights_lora(w[n].float(), lA[n].float(), lB[n].float(), r, f, d, n) for n in w}
        lo = {n: (views[n][1], views[n][2]) for n in w}
        W3 = {n: w[n].float().view(E, f, d) for n in w}
        idx = torch.stack([torch.randperm(E)[:k] for _ in range(T)])
        # tensor-parallel style: x (T,d), fan-out k, grouped output, combine done by the caller
        x = torch.randn(T, d).to(dtype)
        sei, ssi = oracle.flatten_and_sort(idx)
        gw = torch.rand(T, k)
        ref, _ = oracle.moe_block(x.float(), None, W3["w1"], W3["w2"], W3["w3"], k, lo, alpha, routing=(gw, idx))
        ptrs = {n: (lA[n].to(dev), lB[n].to(dev), r, alpha, d, f) for n in w}
        yg = moe.scattermoe_permute_and_compute(x.to(dev), w["w1"].to(dev), w["w2"].to(dev), w["w3"].to(dev), f, d, k,
                                                sei.to(dev), ssi.to(dev), E, ptrs, moe_expert_model_parallelism=False)
        out = oracle.combine(yg.float().cpu(), ssi, gw, T, k)
        assert rel(out, ref) < tol
        # expert-parallel style: rows already one per assignment, output scattered back to `indices`
        xr = torch.randn(T * k, d).to(dtype)
        e_of_row = torch.randint(0, E, (T * k,))
        sei2, ssi2 = oracle.flatten_and_sort(e_of_row)
        y = moe.scattermoe_permute_and_compute(xr.to(dev), w["w1"].to(dev), w["w2"].to(dev), w["w3"].to(dev), f, d, k,
                                               sei2.to(dev), ssi2.to(dev), E, ptrs, moe_expert_model_parallelism=True)
        ref2, _ = oracle.moe_block(xr.float(), None, W3["w1"], W3["w2"], W3["w3"], 1, lo, alpha,
                                   routing=(torch.ones(T * k, 1), e_of_row[:, None]))
        assert rel(y, ref2) < tol


@pytest.mark.parametrize("use_gates", [False, True])
def test_fused_mlp_full_finetune_weight_grads(dev, oracle, use_gates):
    """No adapters, trainable expert weights (the reference's full fine-tuning mode): the fused backward returns
    dW1 / dW3 / dW2 in the stored (E, f, d) orientation; pre-dispatched rows (fan-out 1) and the gate-combined form."""
    from moe_distributed_training_amd.megablocks_utils.moe_mlp import fused_expert_mlp
    torch.manual_seed(12)
    T, d, f, E, k = 160, 128, 192, 4, 2
    w = [(torch.randn(E, f, d) * 0.05).bfloat16() for _ in range(3)]      # w1, w2, w3
    if use_gates:
        x = torch.randn(T, d).bfloat16()
        idx = torch.stack([torch.randperm(E)[:k] for _ in range(T)])
        gw = torch.rand(T, k)
        fan = k
    else:
        x = torch.randn(T * k, d).bfloat16()
        idx = torch.randint(0, E, (T * k, 1))
        gw = torch.ones(T * k, 1)
        fan = 1
    sei, ssi = oracle.flatten_and_sort(idx)
    eo = torch.bincount(sei, minlength=E).cumsum(0)
    dout = torch.randn(x.shape[0], d).bfloat16()
    wo = [t.float().requires_grad_(True) for t in w]
    xo = x.float().requires_grad_(True)
    ref, _ = oracle.moe_block(xo, None, wo[0], wo[1], wo[2], fan, None, 1.0, routing=(gw, idx))
    ref.backward(dout.float())
    wd = [t.to(dev).requires_grad_(True) for t in w]
    xg = x.to(dev).requires_grad_(True)
    out = fused_expert_mlp(xg, wd[0], wd[1], wd[2], fan, ssi.to(dev), eo.to(dev), None, 1.0,
                           gates=gw.to(dev) if use_gates else None)
    out.backward(dout.to(dev))
    assert rel(out, ref) < 1e-2 and rel(xg.grad, xo.grad) < 1e-2
    for n, a, b in zip(("w1", "w2", "w3"), wd, wo):
        check_expert_grads(a.grad, b.grad, f"dW {n}")


def test_block_module_returns_hidden_and_none(dev):
    import moe_distributed_training_amd as moe
    torch.manual_seed(8)
    blk = moe.ScatterMoEBlock(128, 256, 4, top_k=2, lora_r=16, lora_alpha=32.0, device=dev)
    with torch.no_grad():
        blk.lora_B_w1.normal_(0, 0.02)
    x = torch.randn(2, 64, 128, device=dev, dtype=torch.bfloat16, requires_grad=True)
    out, aux = blk(x)
    assert aux is None and out.shape == x.shape
    out.float().pow(2).sum().backward()
    assert x.grad is not None and blk.lora_A_w1.grad is not None and blk.lora_B_w2.grad is not None
    assert blk.w1.grad is None


def test_block_bias_branch_follows_the_reference(dev):
    """ParallelMLP.forward's bias branch (config_utils.py:80-84): (hidden, bias) with return_bias, else hidden + bias as a
    single tensor; without a bias the (hidden, None) pair."""
    import moe_distributed_training_amd as moe
    torch.manual_seed(4)
    kw = dict(top_k=2, device=dev)
    plain = moe.ScatterMoEBlock(128, 256, 4, **kw)
    summed = moe.ScatterMoEBlock(128, 256, 4, bias=True, **kw)
    paired = moe.ScatterMoEBlock(128, 256, 4, bias=True, return_bias=True, **kw)
    for blk in (summed, paired):
        blk.load_state_dict(plain.state_dict(), strict=False)
        with torch.no_grad():
            blk.bias.normal_()
    x = torch.randn(3, 40, 128, device=dev, dtype=torch.bfloat16)
    with torch.no_grad():
        base, none = plain(x)
        assert none is None
        y = summed(x)
        assert torch.is_tensor(y) and torch.equal(y, base + summed.bias)
        h, b = paired(x)
        assert torch.equal(h, base) and b is paired.bias


@pytest.mark.slow
@pytest.mark.parametrize("dtype,tol", [(torch.bfloat16, 1e-2), (torch.float16, 3e-3)])
def test_mixtral_shape_full_size(dev, oracle, dtype, tol):
    """BASELINE configs[1]/[2]: T=4096, d=4096, f=14336, E=8, top-2, LoRA r=16 alpha=32, fwd+bwd at full size against
    the fp32 oracle on the host (a few seconds of CPU GEMMs); in bf16 and, for the reference's fp16 switch, in fp16."""
    import moe_distributed_training_amd as moe
    T, d, f, E, k, r, alpha = 4096, 4096, 14336, 8, 2, 16, 32.0
    g = torch.Generator(device=dev).manual_seed(0)
    rn = lambda *s, std=1.0: (torch.randn(*s, generator=g, device=dev) * std).to(dtype)
    x, wg = rn(T, d), rn(E, d, std=0.02)
    w1, w2, w3 = rn(E, f, d, std=0.02), rn(E, f, d, std=0.02), rn(E, f, d, std=0.02)
    lora = {"w1": (rn(E, d, r, std=0.02), rn(E, r, f, std=0.02)), "w3": (rn(E, d, r, std=0.02), rn(E, r, f, std=0.02)),
            "w2": (rn(E, f, r, std=0.02), rn(E, r, d, std=0.02))}
    dout = rn(T, d)
    lt, views = _views({n: (a.cpu(), b.cpu()) for n, (a, b) in lora.items()}, dev)
    xg = x.clone().requires_grad_(True)
    out, ew, ei = moe.moe_layer_forward(xg, wg, w1, w2, w3, k, views, alpha)
    out.backward(dout)
    torch.cuda.synchronize()
    torch.set_num_threads(16)
    xo = x.float().cpu().requires_grad_(True)
    lo = {n: (a.float().cpu().requires_grad_(True), b.float().cpu().requires_grad_(True)) for n, (a, b) in lora.items()}
    ref, aux = oracle.moe_block(xo, wg.float().cpu(), w1.float().cpu(), w2.float().cpu(), w3.float().cpu(), k, lo, alpha)
    ref.backward(dout.float().cpu())
    flips = int((ei.cpu().long() != aux["indices"]).any(-1).sum())
    assert flips == 0, f"{flips} tokens routed differently from the fp32 oracle"
    assert out.dtype == dtype and rel(out, ref) < tol and rel(xg.grad, xo.grad) < tol
    for n in ("w1", "w3", "w2"):
        check_expert_grads(lt[n][0].grad, lo[n][0].grad, f"dA {n}", tol)
        check_expert_grads(lt[n][1].grad, lo[n][1].grad, f"dB {n}", tol)


@pytest.mark.slow
def test_mixtral_shape_forward_without_adapters_full_size(dev, oracle):
    """BASELINE configs[1] exactly: T=4096, d=4096, f=14336, E=8, top-2, near-uniform routing, no adapters, forward
    only -- the adapter-free gate/up kernel variant and its tile plan at the full size, against the fp32 oracle."""
    import moe_distributed_training_amd as moe
    T, d, f, E, k = 4096, 4096, 14336, 8, 2
    g = torch.Generator(device=dev).manual_seed(1)
    rn = lambda *s, std=1.0: (torch.randn(*s, generator=g, device=dev) * std).bfloat16()
    x, wg = rn(T, d), rn(E, d, std=0.02)
    w1, w2, w3 = rn(E, f, d, std=0.02), rn(E, f, d, std=0.02), rn(E, f, d, std=0.02)
    with torch.no_grad():
        out, ew, ei = moe.moe_layer_forward(x, wg, w1, w2, w3, k, None, 1.0)
        torch.cuda.synchronize()
        torch.set_num_threads(16)
        ref, aux = oracle.moe_block(x.float().cpu(), wg.float().cpu(), w1.float().cpu(), w2.float().cpu(), w3.float().cpu(), k)
    counts = torch.bincount(aux["indices"].flatten(), minlength=E)
    assert counts.min() > 0.8 * T * k / E and counts.max() < 1.2 * T * k / E   # near-uniform, as the configuration says
    flips = int((ei.cpu().long() != aux["indices"]).any(-1).sum())
    assert flips == 0, f"{flips} tokens routed differently from the fp32 oracle"
    assert torch.allclose(ew.float().cpu(), aux["weights"], atol=2e-3)
    assert rel(out, ref) < 1e-2


@pytest.mark.slow
def test_mixtral_shape_full_finetune_full_size(dev, oracle):
    """Full fine-tuning (no adapters, the stored expert weights take gradients) at the Mixtral shape, T=4096, fwd+bwd:
    out, dX and dW1 / dW3 / dW2 of every expert (max and RMS on the expert's own scale) against the fp32 oracle."""
    import moe_distributed_training_amd as moe
    T, d, f, E, k = 4096, 4096, 14336, 8, 2
    g = torch.Generator(device=dev).manual_seed(2)
    rn = lambda *s, std=1.0: (torch.randn(*s, generator=g, device=dev) * std).bfloat16()
    x, wg = rn(T, d), rn(E, d, std=0.02)
    wd = [rn(E, f, d, std=0.02).requires_grad_(True) for _ in range(3)]      # w1, w2, w3
    dout = rn(T, d)
    xg = x.clone().requires_grad_(True)
    out, ew, ei = moe.moe_layer_forward(xg, wg, wd[0], wd[1], wd[2], k, None, 1.0)
    out.backward(dout)
    torch.cuda.synchronize()
    torch.set_num_threads(16)
    xo = x.float().cpu().requires_grad_(True)
    wo = [w.detach().float().cpu().requires_grad_(True) for w in wd]
    ref, aux = oracle.moe_block(xo, wg.float().cpu(), wo[0], wo[1], wo[2], k)
    ref.backward(dout.float().cpu())
    assert torch.equal(ei.cpu().long(), aux["indices"])
    assert rel(out, ref) < 1e-2 and rel(xg.grad, xo.grad) < 1e-2
    for n, a, b in zip(("w1", "w2", "w3"), wd, wo):
        assert a.grad is not None and a.grad.shape == b.grad.shape
        check_expert_grads(a.grad, b.grad, f"dW {n}")
        a.grad = None
        b.grad = None


@pytest.mark.slow
def test_mixtral_shape_skewed_routing_full_gradients(dev, oracle):
    """BASELINE configs[3]'s routing (Zipf s=1.2 logit offsets: the top expert takes ~40 % of the assignments, the
    last ones are near-empty) at the real d, f with LoRA, T=4096, fwd+bwd: out, dX and all six adapter gradients
    against the fp32 oracle, every expert's slice on its own scale -- a ragged tail whose rows were dropped, or a
    near-empty group that was mishandled, cannot hide behind the large groups."""
    import moe_distributed_training_amd as moe
    T, d, f, E, k, r, alpha = 4096, 4096, 14336, 8, 2, 16, 32.0
    g = torch.Generator(device=dev).manual_seed(4)
    rn = lambda *s, std=1.0: (torch.randn(*s, generator=g, device=dev) * std).bfloat16()
    x, wg = rn(T, d), rn(E, d, std=0.02)
    pmf = torch.tensor([1.0 / (i + 1) ** 1.2 for i in range(E)]); pmf /= pmf.sum()
    x[:, 0] = 1.0
    wg[:, 0] = (2.2 * torch.log(pmf)).bfloat16().to(dev)
    w1, w2, w3 = rn(E, f, d, std=0.02), rn(E, f, d, std=0.02), rn(E, f, d, std=0.02)
    lora = {"w1": (rn(E, d, r, std=0.02), rn(E, r, f, std=0.02)), "w3": (rn(E, d, r, std=0.02), rn(E, r, f, std=0.02)),
            "w2": (rn(E, f, r, std=0.02), rn(E, r, d, std=0.02))}
    dout = rn(T, d)
    lt, views = _views({n: (a.cpu(), b.cpu()) for n, (a, b) in lora.items()}, dev)
    xg = x.clone().requires_grad_(True)
    out, ew, ei = moe.moe_layer_forward(xg, wg, w1, w2, w3, k, views, alpha)
    out.backward(dout)
    torch.cuda.synchronize()
    torch.set_num_threads(16)
    xo = x.float().cpu().requires_grad_(True)
    lo = {n: (a.float().cpu().requires_grad_(True), b.float().cpu().requires_grad_(True)) for n, (a, b) in lora.items()}
    ref, aux = oracle.moe_block(xo, wg.float().cpu(), w1.float().cpu(), w2.float().cpu(), w3.float().cpu(), k, lo, alpha)
    ref.backward(dout.float().cpu())
    assert torch.equal(ei.cpu().long(), aux["indices"])
    counts = torch.bincount(aux["indices"].flatten(), minlength=E)
    assert counts.max() > 0.3 * T * k and counts.min() < 0.05 * T * k, counts.tolist()
    assert rel(out, ref) < 1e-2 and rel(xg.grad, xo.grad) < 1e-2
    for n in ("w1", "w3", "w2"):
        check_expert_grads(lt[n][0].grad, lo[n][0].grad, f"dA {n} counts={counts.tolist()}")
        check_expert_grads(lt[n][1].grad, lo[n][1].grad, f"dB {n} counts={counts.tolist()}")


@pytest.mark.slow
def test_ep_share_full_size(dev, oracle):
    """BASELINE configs[4] at its real size: one expert-parallel rank's share, 2 resident experts, 8192 pre-dispatched
    rows (group sizes from a 0.55 / 0.45 draw, arrival order a permutation), fan-out 1, LoRA r=16, fwd+bwd, against the
    fp32 oracle (two experts over 8 XCDs, ~18 row tiles each: the tile plan of few, large groups)."""
    import moe_distributed_training_amd as moe
    d, f, r, alpha, E, R = 4096, 14336, 16, 32.0, 2, 8192
    g = torch.Generator(device=dev).manual_seed(6)
    rn = lambda *s, std=1.0: (torch.randn(*s, generator=g, device=dev) * std).bfloat16()
    w1, w2, w3 = rn(E, f, d, std=0.02), rn(E, f, d, std=0.02), rn(E, f, d, std=0.02)
    lora = {"w1": (rn(E, d, r, std=0.02), rn(E, r, f, std=0.02)), "w3": (rn(E, d, r, std=0.02), rn(E, r, f, std=0.02)),
            "w2": (rn(E, f, r, std=0.02), rn(E, r, d, std=0.02))}
    xr, dy = rn(R, d), rn(R, d)
    e_of_row = (torch.rand(R, generator=torch.Generator().manual_seed(7)) > 0.55).long()
    sei, ssi = oracle.flatten_and_sort(e_of_row)
    eo = torch.bincount(sei, minlength=E).cumsum(0)
    lt, views = _views({n: (a.cpu(), b.cpu()) for n, (a, b) in lora.items()}, dev)
    xg = xr.clone().requires_grad_(True)
    y = moe.fused_expert_mlp(xg, w1, w2, w3, 1, ssi.int().to(dev), eo.int().to(dev), views, alpha)
    y.backward(dy)
    torch.cuda.synchronize()
    torch.set_num_threads(16)
    xo = xr.float().cpu().requires_grad_(True)
    lo = {n: (a.float().cpu().requires_grad_(True), b.float().cpu().requires_grad_(True)) for n, (a, b) in lora.items()}
    ref, _ = oracle.moe_block(xo, None, w1.float().cpu(), w2.float().cpu(), w3.float().cpu(), 1, lo, alpha,
                              routing=(torch.ones(R, 1), e_of_row[:, None]))
    ref.backward(dy.float().cpu())
    assert rel(y, ref) < 1e-2 and rel(xg.grad, xo.grad) < 1e-2
    for n in ("w1", "w3", "w2"):
        check_expert_grads(lt[n][0].grad, lo[n][0].grad, f"dA {n}")
        check_expert_grads(lt[n][1].grad, lo[n][1].grad, f"dB {n}")


@pytest.mark.slow
def test_skewed_routing_and_ep_share(dev, oracle):
    """BASELINE configs[3] (Zipf-skewed routing, ragged groups, one near-empty expert) at reduced T and configs[4]
    (one expert-parallel rank's share: 2 resident experts, pre-dispatched rows, fan-out 1) at reduced rows, both at
    the real d=4096, f=14336; plus size-independent properties of the full path."""
    import moe_distributed_training_amd as moe
    from moe_distributed_training_amd.megablocks_utils import router
    d, f, r, alpha = 4096, 14336, 16, 32.0
    g = torch.Generator(device=dev).manual_seed(1)
    rn = lambda *s, std=1.0: (torch.randn(*s, generator=g, device=dev) * std).bfloat16()
    # --- EP share: E=2, rows pre-dispatched, sizes from a 0.55/0.45 split, indices a permutation
    E, R = 2, 2048
    w1, w2, w3 = rn(E, f, d, std=0.02), rn(E, f, d, std=0.02), rn(E, f, d, std=0.02)
    lora = {"w1": (rn(E, d, r, std=0.02), rn(E, r, f, std=0.02)), "w3": (rn(E, d, r, std=0.02), rn(E, r, f, std=0.02)),
            "w2": (rn(E, f, r, std=0.02), rn(E, r, d, std=0.02))}
    xr, dy = rn(R, d), rn(R, d)
    e_of_row = (torch.rand(R, generator=torch.Generator().manual_seed(2)) > 0.55).long()
    sei, ssi = oracle.flatten_and_sort(e_of_row)
    eo = torch.bincount(sei, minlength=E).cumsum(0)
    lt, views = _views({n: (a.cpu(), b.cpu()) for n, (a, b) in lora.items()}, dev)
    xg = xr.clone().requires_grad_(True)
    y = moe.fused_expert_mlp(xg, w1, w2, w3, 1, ssi.int().to(dev), eo.int().to(dev), views, alpha)
    y.backward(dy)
    xo = xr.float().cpu().requires_grad_(True)
    lo = {n: (a.float().cpu().requires_grad_(True), b.float().cpu().requires_grad_(True)) for n, (a, b) in lora.items()}
    ref, _ = oracle.moe_block(xo, None, w1.float().cpu(), w2.float().cpu(), w3.float().cpu(), 1, lo, alpha,
                              routing=(torch.ones(R, 1), e_of_row[:, None]))
    ref.backward(dy.float().cpu())
    assert rel(y, ref) < 1e-2 and rel(xg.grad, xo.grad) < 1e-2
    for n in ("w1", "w3", "w2"):
        check_expert_grads(lt[n][0].grad, lo[n][0].grad, f"dA {n}"); check_expert_grads(lt[n][1].grad, lo[n][1].grad, f"dB {n}")
    # --- skewed routing through the whole layer with the same two experts' weights replicated to E=8 views
    E8 = 8
    w1e, w2e, w3e = (t.repeat(4, 1, 1) for t in (w1, w2, w3))
    T = 2048
    x = rn(T, d)
    wg = rn(E8, d, std=0.02)
    pmf = torch.tensor([1.0 / (i + 1) ** 1.2 for i in range(E8)]); pmf /= pmf.sum()
    x[:, 0] = 1.0
    wg[:, 0] = (2.2 * torch.log(pmf)).bfloat16().to(dev)
    out, ew, ei = moe.moe_layer_forward(x, wg, w1e, w2e, w3e, 2)
    ref, aux = oracle.moe_block(x.float().cpu(), wg.float().cpu(), w1e.float().cpu(), w2e.float().cpu(), w3e.float().cpu(), 2)
    assert torch.equal(ei.cpu().long(), aux["indices"])
    counts = torch.bincount(ei.flatten().cpu().long(), minlength=E8)
    assert counts.max() > 0.3 * 2 * T and counts.min() < 0.05 * 2 * T       # really skewed
    assert rel(out, ref) < 1e-2
    # size-independent properties: rows are independent (any subset of tokens gives the same rows), and the
    # output is linear in the combine weights
    sub = torch.arange(0, T, 7, device=dev)
    out_sub, _, ei_sub = moe.moe_layer_forward(x[sub].contiguous(), wg, w1e, w2e, w3e, 2)
    assert torch.equal(ei_sub, ei[sub]) and rel(out_sub, out[sub].float().cpu()) < 1e-2


@pytest.mark.parametrize("counts", [
    [1, 16, 17, 32, 33, 48, 64, 65],              # wave row 0 with 1, 1, 2, 2, 3, 3, 4 and 5 live blocks; wave row 1 without rows
    [100, 128, 129, 144, 160, 161, 193, 224],     # wave row 0 full; wave row 1 with 0, 0, 1, 1, 2, 3, 5 and 6 live blocks
    [225, 255, 256, 257, 300, 511, 513, 0],       # tiles that run the unchecked loop, tails behind full tiles, an empty group
])
def test_ragged_row_tiles_of_every_block_count(dev, oracle, counts):
    """Groups whose last row tile has every number of live 16-row blocks a wave can meet: each count runs its own copy
    of the grouped GEMMs' K loop, blocks inside a count but past the group compute on rows that were never loaded, and
    the fused epilogues (SwiGLU with the h A2 product; SwiGLU backward with the adapter gradients' row and column sums)
    must keep those rows out of every sum.  (The counts are those of tiles of 256 rows, which the next test's larger launches take; here the tiles have 128, and a
    wave at most four blocks.)  Pre-dispatched rows, LoRA r=16, forward and backward against the fp32 oracle."""
    import moe_distributed_training_amd as moe
    d, f, r, alpha = 256, 512, 16, 32.0
    E, R = len(counts), sum(counts)
    g = torch.Generator(device=dev).manual_seed(11)
    rn = lambda *s, std=1.0: (torch.randn(*s, generator=g, device=dev) * std).bfloat16()
    w1, w2, w3 = rn(E, f, d, std=0.05), rn(E, f, d, std=0.05), rn(E, f, d, std=0.05)
    lora = {"w1": (rn(E, d, r, std=0.05), rn(E, r, f, std=0.05)), "w3": (rn(E, d, r, std=0.05), rn(E, r, f, std=0.05)),
            "w2": (rn(E, f, r, std=0.05), rn(E, r, d, std=0.05))}
    xr, dy = rn(R, d), rn(R, d)
    e_of_row = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(R, generator=torch.Generator().manual_seed(5))]
    sei, ssi = oracle.flatten_and_sort(e_of_row)
    eo = torch.bincount(sei, minlength=E).cumsum(0)
    lt, views = _views({n: (a.cpu(), b.cpu()) for n, (a, b) in lora.items()}, dev)
    xg = xr.clone().requires_grad_(True)
    y = moe.fused_expert_mlp(xg, w1, w2, w3, 1, ssi.int().to(dev), eo.int().to(dev), views, alpha)
    y.backward(dy)
    xo = xr.float().cpu().requires_grad_(True)
    lo = {n: (a.float().cpu().requires_grad_(True), b.float().cpu().requires_grad_(True)) for n, (a, b) in lora.items()}
    ref, _ = oracle.moe_block(xo, None, w1.float().cpu(), w2.float().cpu(), w3.float().cpu(), 1, lo, alpha,
                              routing=(torch.ones(R, 1), e_of_row[:, None]))
    ref.backward(dy.float().cpu())
    assert torch.isfinite(y.float()).all() and torch.isfinite(xg.grad.float()).all()
    assert rel(y, ref) < 1e-2 and rel(xg.grad, xo.grad) < 1e-2
    for n in ("w1", "w3", "w2"):
        assert torch.isfinite(lt[n][0].grad.float()).all() and torch.isfinite(lt[n][1].grad.float()).all()
        check_expert_grads(lt[n][0].grad, lo[n][0].grad, f"dA {n}", tol=TINY_GROUP_TOL)
        check_expert_grads(lt[n][1].grad, lo[n][1].grad, f"dB {n}", tol=TINY_GROUP_TOL)


@pytest.mark.parametrize("counts", [[1, 16, 17, 32, 33, 48, 64, 65], [100, 128, 129, 144, 160, 161, 193, 224], [225, 255, 256, 257, 300, 511, 513, 0]])
@pytest.mark.parametrize("d,f,tiles", [(1088, 2112, (256, 256, 256, 256)), (192, 320, (128, 128, 128, 128)), (1024, 512, (128, 128, 128, None))])
def test_ragged_row_tiles_in_large_and_small_tiles(dev, oracle, counts, d, f, tiles):
    """The row counts above where the launches take 256 x 256 tiles (1088 x 2112: the chip is more than half full) and where they take 128 x 128
    ones with a last column tile that is not full (192 x 320); the row tiles' partials of the adapter gradients differ in number.  1024 x 512: the dh and dX launches cut every
    tile along K (that of dX in tiles of either size), and the dh launch's row-tile partials lie behind what they exchange, in the same area, until the sums at the end read them."""
    import moe_distributed_training_amd as moe
    r, alpha, E, R = 16, 32.0, len(counts), sum(counts)
    assert all(want in (None, got) for got, want in zip(_tiles(R, E, d, f), tiles))
    if d == 1024:
        from moe_distributed_training_amd._lib import lib
        from test_gpu_ops import _plan
        for K, N, nseg in ((d, f, 1), (f, d, 2)):
            plan, _ = _plan(dev, counts, K, N, False, nseg)
            assert (plan[plan[:, 0] == 1][:, 6] == 2).all()
        # adapters add to the workspace their packed factors, the interims and the column-tile partials, and nothing for row tiles: those lie in the exchange area
        up = lambda n: (n + 255) // 256 * 256
        factors = 3 * up(E * 32 * d) + 3 * up(E * 32 * f)
        interims, columns = 7 * up(((R + 31) // 32 * 32 + 32) * 32), up(max(f // 64, 2 * (f // 128)) * R * 64)
        assert lib.moe_mlp_workspace_bytes(R, E, d, f, r) == lib.moe_mlp_workspace_bytes(R, E, d, f, 0) + factors + interims + columns
    g = torch.Generator().manual_seed(12)
    rn = lambda *s, std=1.0: (torch.randn(*s, generator=g) * std).bfloat16()
    w1, w2, w3 = rn(E, f, d, std=0.03), rn(E, f, d, std=0.03), rn(E, f, d, std=0.03)
    lora = {"w1": (rn(E, d, r, std=0.03), rn(E, r, f, std=0.03)), "w3": (rn(E, d, r, std=0.03), rn(E, r, f, std=0.03)),
            "w2": (rn(E, f, r, std=0.03), rn(E, r, d, std=0.03))}
    xr, dy = rn(R, d), rn(R, d)
    e_of_row = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(R, generator=g)]
    sei, ssi = oracle.flatten_and_sort(e_of_row)
    eo = torch.bincount(sei, minlength=E).cumsum(0)
    lt, views = _views(lora, dev)
    xg = xr.to(dev).requires_grad_(True)
    y = moe.fused_expert_mlp(xg, w1.to(dev), w2.to(dev), w3.to(dev), 1, ssi.int().to(dev), eo.int().to(dev), views, alpha)
    y.backward(dy.to(dev))
    xo = xr.float().requires_grad_(True)
    lo = {n: (a.float().requires_grad_(True), b.float().requires_grad_(True)) for n, (a, b) in lora.items()}
    ref, _ = oracle.moe_block(xo, None, w1.float(), w2.float(), w3.float(), 1, lo, alpha, routing=(torch.ones(R, 1), e_of_row[:, None]))
    ref.backward(dy.float())
    assert rel(y, ref) < 1e-2 and rel(xg.grad, xo.grad) < 1e-2
    for n in ("w1", "w3", "w2"):
        check_expert_grads(lt[n][0].grad, lo[n][0].grad, f"dA {n}", tol=TINY_GROUP_TOL)
        check_expert_grads(lt[n][1].grad, lo[n][1].grad, f"dB {n}", tol=TINY_GROUP_TOL)


@pytest.mark.slow
def test_skewed_full_size_properties(dev, oracle):
    """BASELINE configs[3] at its full size (T=16384, E=8, top-2, Zipf-skewed routing, LoRA r=16, fwd+bwd) through
    properties that do not need a full-size oracle run: (1) tokens are independent, so the output and dX rows of a
    slice of the batch equal the fp32 oracle run on that slice alone (same router, same weights); (2) the backward
    pass is linear in the upstream gradient, which ties the adapter gradients -- sums over ALL rows of the ragged
    groups -- of two runs to a third; (3) the sorted order is a permutation with the histogram the indices imply."""
    import moe_distributed_training_amd as moe
    from moe_distributed_training_amd.megablocks_utils import router
    T, d, f, E, k, r, alpha = 16384, 4096, 14336, 8, 2, 16, 32.0
    g = torch.Generator(device=dev).manual_seed(3)
    rn = lambda *s, std=1.0: (torch.randn(*s, generator=g, device=dev) * std).bfloat16()
    x, wg = rn(T, d), rn(E, d, std=0.02)
    pmf = torch.tensor([1.0 / (i + 1) ** 1.2 for i in range(E)]); pmf /= pmf.sum()
    x[:, 0] = 1.0
    wg[:, 0] = (2.2 * torch.log(pmf)).bfloat16().to(dev)
    w1, w2, w3 = rn(E, f, d, std=0.02), rn(E, f, d, std=0.02), rn(E, f, d, std=0.02)
    lora = {"w1": (rn(E, d, r, std=0.02), rn(E, r, f, std=0.02)), "w3": (rn(E, d, r, std=0.02), rn(E, r, f, std=0.02)),
            "w2": (rn(E, f, r, std=0.02), rn(E, r, d, std=0.02))}
    d1, d2 = rn(T, d), rn(T, d)

    def run(dout):
        lt, views = _views({n: (a.cpu(), b.cpu()) for n, (a, b) in lora.items()}, dev)
        xg = x.clone().requires_grad_(True)
        out, ew, ei = moe.moe_layer_forward(xg, wg, w1, w2, w3, k, views, alpha)
        out.backward(dout)
        return out.detach(), ei, xg.grad, {n: (lt[n][0].grad, lt[n][1].grad) for n in lt}, ew.detach()

    out, ei, dx1, g1, ew = run(d1)
    _, _, dx2, g2, _ = run(d2)
    _, _, dx3, g3, _ = run((d1.float() + d2.float()).bfloat16())
    counts = torch.bincount(ei.flatten().cpu().long(), minlength=E)
    assert int(counts.sum()) == T * k and counts.max() > 0.3 * T * k and counts.min() < 0.05 * T * k   # really skewed
    rt = router.route_and_sort(x, wg, k)
    assert torch.equal(torch.sort(rt.sorted_scattered_idxs.long()).values, torch.arange(T * k, device=dev))
    assert torch.equal(rt.tokens_per_expert.cpu().long(), counts)
    # (2) linearity of the backward pass (the sum of two bf16 gradients is itself rounded to bf16: 2^-8 relative)
    assert rel(dx3, (dx1.float() + dx2.float()).cpu()) < 1.5e-2
    for n in ("w1", "w3", "w2"):
        for j in (0, 1):
            assert rel(g3[n][j], (g1[n][j].float() + g2[n][j].float()).cpu()) < 1.5e-2, (n, j)
    # (1) a slice of the batch against the oracle on that slice alone
    sl = slice(5000, 5768)
    xo = x[sl].float().cpu().requires_grad_(True)
    lo = {n: (a.float().cpu(), b.float().cpu()) for n, (a, b) in lora.items()}
    torch.set_num_threads(16)
    ref, aux = oracle.moe_block(xo, wg.float().cpu(), w1.float().cpu(), w2.float().cpu(), w3.float().cpu(), k, lo, alpha)
    ref.backward(d1[sl].float().cpu())
    assert torch.equal(ei[sl].cpu().long(), aux["indices"])
    assert rel(out[sl], ref) < 1e-2 and rel(dx1[sl], xo.grad) < 1e-2
    # (4) adapter gradients of single experts against the oracle: an expert's dA / dB depend only on the rows routed to
    # it, so the oracle run on those tokens alone (one assignment each, the layer's own routing weight) gives them.  The
    # smallest group (near-empty), a mid-sized one and the largest (the only group with more than 50 row tiles).
    ewc, eic = ew.float().cpu(), ei.cpu().long()
    order = torch.argsort(counts)
    for e in (int(order[0]), int(order[E // 2]), int(order[-1])):
        tok, slot = torch.where(eic == e)
        loe = {n: (a.float().cpu().requires_grad_(True), b.float().cpu().requires_grad_(True)) for n, (a, b) in lora.items()}
        refe, _ = oracle.moe_block(x[tok.to(dev)].float().cpu(), None, w1.float().cpu(), w2.float().cpu(), w3.float().cpu(), 1, loe, alpha,
                                   routing=(ewc[tok, slot][:, None], torch.full((tok.numel(), 1), e)))
        refe.backward(d1[tok.to(dev)].float().cpu())
        for n in ("w1", "w3", "w2"):
            for j, nm in ((0, "dA"), (1, "dB")):
                check_expert_grads(g1[n][j][e:e + 1], loe[n][j].grad[e:e + 1], f"{nm} {n} expert {e} ({tok.numel()} rows)")


@pytest.mark.slow
def test_layer_with_intermediates_above_2GiB(dev, oracle):
    """T=40960 tokens (R=81920 rows) at the Mixtral shape: gate, up, h, dgate and dup are 2.35 GB each, beyond what a
    32-bit byte offset from the tensor's start reaches in the SwiGLU epilogues.  Tokens are independent, so out and dX of
    slices of the batch (the first rows, the last rows, the rows around the 2 GiB mark of the grouped order is not
    addressable by token -- slices spread over the batch) equal the fp32 oracle run on those slices alone."""
    import moe_distributed_training_amd as moe
    T, d, f, E, k, r, alpha = 40960, 4096, 14336, 8, 2, 16, 32.0
    g = torch.Generator(device=dev).manual_seed(8)
    rn = lambda *s, std=1.0: (torch.randn(*s, generator=g, device=dev) * std).bfloat16()
    x, wg = rn(T, d), rn(E, d, std=0.02)
    w1, w2, w3 = rn(E, f, d, std=0.02), rn(E, f, d, std=0.02), rn(E, f, d, std=0.02)
    lora = {"w1": (rn(E, d, r, std=0.02), rn(E, r, f, std=0.02)), "w3": (rn(E, d, r, std=0.02), rn(E, r, f, std=0.02)),
            "w2": (rn(E, f, r, std=0.02), rn(E, r, d, std=0.02))}
    dout = rn(T, d)
    lt, views = _views({n: (a.cpu(), b.cpu()) for n, (a, b) in lora.items()}, dev)
    xg = x.clone().requires_grad_(True)
    out, ew, ei = moe.moe_layer_forward(xg, wg, w1, w2, w3, k, views, alpha)
    out.backward(dout)
    torch.cuda.synchronize()
    assert T * k * f * 2 > (1 << 31)
    torch.set_num_threads(16)
    W = [t.float().cpu() for t in (wg, w1, w2, w3)]
    lo = {n: (a.float().cpu(), b.float().cpu()) for n, (a, b) in lora.items()}
    for sl in (slice(0, 192), slice(T // 2 - 96, T // 2 + 96), slice(T - 192, T)):
        xo = x[sl].float().cpu().requires_grad_(True)
        ref, aux = oracle.moe_block(xo, W[0], W[1], W[2], W[3], k, lo, alpha)
        ref.backward(dout[sl].float().cpu())
        assert torch.equal(ei[sl].cpu().long(), aux["indices"])
        assert rel(out[sl], ref) < 1e-2 and rel(xg.grad[sl], xo.grad) < 1e-2, sl
    # adapter gradients of the last expert -- its rows sit at the end of the grouped order, past the 2 GiB mark of every
    # (R, f) tensor -- against the oracle run on the tokens routed to it (one assignment each, the layer's own weight)
    e = E - 1
    ewc, eic = ew.detach().float().cpu(), ei.cpu().long()
    tok, slot = torch.where(eic == e)
    loe = {n: (a.float().cpu().requires_grad_(True), b.float().cpu().requires_grad_(True)) for n, (a, b) in lora.items()}
    refe, _ = oracle.moe_block(x[tok.to(dev)].float().cpu(), None, W[1], W[2], W[3], 1, loe, alpha,
                               routing=(ewc[tok, slot][:, None], torch.full((tok.numel(), 1), e)))
    refe.backward(dout[tok.to(dev)].float().cpu())
    for n in ("w1", "w3", "w2"):
        for j, nm in ((0, "dA"), (1, "dB")):
            check_expert_grads(lt[n][j].grad[e:e + 1], loe[n][j].grad[e:e + 1], f"{nm} {n} expert {e} ({tok.numel()} rows)")


def test_step_captures_into_a_graph_and_replays_bit_identically(dev):
    """The library enqueues kernels only (no host synchronisation, no memset nodes, no allocation of its own), so a
    whole forward+backward step can be captured into a HIP graph.  Every replay -- with eager work and synchronisations
    in between -- must reproduce the eager result bit for bit, also after the inputs change in place."""
    import moe_distributed_training_amd as moe
    T, d, f, E, r, k, alpha = 512, 256, 512, 8, 16, 2, 32.0
    x, wg, w1, w2, w3, lora, dout = _make(T, d, f, E, r, torch.bfloat16, seed=31)
    lt, views = _views(lora, dev)
    xg = x.to(dev).requires_grad_(True)
    wgd, w1d, w2d, w3d, doutd = wg.to(dev), w1.to(dev), w2.to(dev), w3.to(dev), dout.to(dev)
    params = [xg] + [t for n in ("w1", "w3", "w2") for t in lt[n]]

    def step():
        for p in params:
            p.grad = None
        out, _, _ = moe.moe_layer_forward(xg, wgd, w1d, w2d, w3d, k, views, alpha)
        out.backward(doutd)
        return out

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out_g = step()
    grads_g = [p.grad for p in params]          # the tensors the captured step writes
    for trial in range(3):
        if trial:                                # new inputs, written in place into the captured buffers
            with torch.no_grad():
                xg.copy_(torch.randn(T, d, generator=torch.Generator().manual_seed(100 + trial)).bfloat16())
                doutd.copy_(torch.randn(T, d, generator=torch.Generator().manual_seed(200 + trial)).bfloat16())
        graph.replay()
        torch.cuda.synchronize()
        got = [out_g.clone()] + [g.clone() for g in grads_g]
        ref_out = step()                         # eager work between the replays
        torch.cuda.synchronize()
        ref = [ref_out] + [p.grad for p in params]
        for a, b in zip(got, ref):
            assert torch.equal(a, b), f"replay {trial} differs from the eager step"


@pytest.mark.parametrize("T", [0, 1, 3])
@pytest.mark.parametrize("r", [16, 0])
def test_tiny_and_empty_batches(dev, oracle, T, r):
    """Fewer assignments than experts (most groups empty) and the empty batch: the latter returns empty outputs and an
    empty input gradient without launching anything."""
    import moe_distributed_training_amd as moe
    d, f, E, k, alpha = 64, 128, 8, 2, 32.0
    x, wg, w1, w2, w3, lora, dout = _make(max(T, 1), d, f, E, r, torch.bfloat16, seed=5)
    x, dout = x[:T], dout[:T]
    xg = x.to(dev).requires_grad_(True)
    lt, views = (None, None) if lora is None else _views(lora, dev)
    out, ew, ei = moe.moe_layer_forward(xg, wg.to(dev), w1.to(dev), w2.to(dev), w3.to(dev), k, views, alpha)
    out.backward(dout.to(dev))
    assert out.shape == (T, d) and ew.shape == (T, k) and ei.shape == (T, k) and xg.grad.shape == (T, d)
    if T == 0:
        return
    xo = x.float().requires_grad_(True)
    lo = None if lora is None else {n: (a.float().requires_grad_(True), b.float().requires_grad_(True)) for n, (a, b) in lora.items()}
    ref, aux = oracle.moe_block(xo, wg.float(), w1.float(), w2.float(), w3.float(), k, lo, alpha)
    ref.backward(dout.float())
    assert torch.equal(ei.cpu().long(), aux["indices"])
    assert rel(out, ref) < 1e-2 and rel(xg.grad, xo.grad) < 1e-2
    if lora is not None:
        for n in ("w1", "w3", "w2"):   # experts that received no row get exact zeros
            check_expert_grads(lt[n][0].grad, lo[n][0].grad, f"dA {n}", TINY_GROUP_TOL); check_expert_grads(lt[n][1].grad, lo[n][1].grad, f"dB {n}", TINY_GROUP_TOL)
            unused = [e for e in range(E) if e not in aux["indices"].flatten().tolist()]
            assert float(lt[n][0].grad[unused].abs().max()) == 0.0 and float(lt[n][1].grad[unused].abs().max()) == 0.0


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_empty_batch_without_gradients(dev, dtype):
    import moe_distributed_training_amd as moe
    x, wg, w1, w2, w3, _, _ = (t.to(dev) if torch.is_tensor(t) else t for t in _make(1, 64, 128, 8, 0, dtype, seed=5))
    with torch.no_grad():
        out, ew, ei = moe.moe_layer_forward(x[:0], wg, w1, w2, w3, 2, None, 32.0)
    assert out.shape == (0, 64) and ew.shape == (0, 2) and ei.shape == (0, 2)


@pytest.mark.parametrize("seed", range(16))
def test_layer_seeded_shape_sweep(dev, oracle, seed):
    """Seeded draws over the supported shape space of the fused layer (hidden and ffn sizes that are multiples of 64 but
    not of the 256-wide tiles, one to many experts, top-k from 1 to E, adapter ranks off the 16-wide chunks, token counts
    that leave ragged and empty groups), each against the fp32 oracle."""
    import random
    import moe_distributed_training_amd as moe
    rng = random.Random(1000 + seed)
    d = rng.choice([64, 128, 192, 320, 512])
    f = rng.choice([64, 128, 448, 576, 832])
    E = rng.choice([1, 2, 3, 5, 8, 17, 70])
    k = rng.choice(sorted({1, min(2, E), min(3, E), min(E, 6)}))
    T = rng.choice([1, 2, 17, 130, 257, 600, 1100])
    r = rng.choice([0, 4, 8, 16, 20, 32])
    alpha = 32.0
    x, wg, w1, w2, w3, lora, dout = _make(T, d, f, E, r, torch.bfloat16, seed=seed)
    wg = wg * 30      # well separated router scores
    xo = x.float().requires_grad_(True)
    lo = None if lora is None else {n: (a.float().requires_grad_(True), b.float().requires_grad_(True)) for n, (a, b) in lora.items()}
    ref, aux = oracle.moe_block(xo, wg.float(), w1.float(), w2.float(), w3.float(), k, lo, alpha)
    ref.backward(dout.float())
    xg = x.to(dev).requires_grad_(True)
    lt, views = (None, None) if lora is None else _views(lora, dev)
    out, ew, ei = moe.moe_layer_forward(xg, wg.to(dev), w1.to(dev), w2.to(dev), w3.to(dev), k, views, alpha)
    out.backward(dout.to(dev))
    case = f"T={T} d={d} f={f} E={E} k={k} r={r}"
    assert torch.equal(ei.cpu().long(), aux["indices"]), case
    assert rel(out, ref) < 1e-2 and rel(xg.grad, xo.grad) < 1e-2, case
    if lora is not None:
        for n in ("w1", "w3", "w2"):
            check_expert_grads(lt[n][0].grad, lo[n][0].grad, f"dA {n} {case}", TINY_GROUP_TOL)
            check_expert_grads(lt[n][1].grad, lo[n][1].grad, f"dB {n} {case}", TINY_GROUP_TOL)
