"""The layer's autograd node among the tools that work on autograd graphs: activation checkpointing, saved-tensor hooks, tracing and
forward mode; and the shapes and layouts that the node takes as they are."""
import pytest
import torch

pytestmark = pytest.mark.gpu

T, D, F, E, K, R = 48, 128, 192, 4, 2, 16


def _block(dev, dtype=torch.bfloat16, r=R, seed=0):
    import moe_distributed_training_amd as moe
    torch.manual_seed(seed)
    b = moe.ScatterMoEBlock(D, F, E, top_k=K, lora_r=r, lora_alpha=32.0, dtype=dtype, device=dev)
    with torch.no_grad():
        for p in b.parameters():
            p.normal_(0.0, 0.05)
    return b


def _step(fn, block, x, dout):
    """Output and gradients of one forward and backward pass of fn(x)."""
    for p in block.parameters():
        p.grad = None
    x = x.detach().requires_grad_(True)
    out = fn(x)
    out.backward(dout)
    return [out.detach(), x.grad] + [p.grad for p in block.parameters() if p.requires_grad]


def _same(a, b):
    return len(a) == len(b) and all(torch.equal(p, q) for p, q in zip(a, b))


@pytest.mark.parametrize("dtype,r", [(torch.bfloat16, R), (torch.bfloat16, 0), (torch.float32, R)])   # fp32: the unfused route
def test_checkpointing_and_saved_tensor_hooks_change_no_bit(dev, dtype, r):
    from torch.utils.checkpoint import checkpoint
    block = _block(dev, dtype, r)
    x, dout = torch.randn(T, D, device=dev, dtype=dtype), torch.randn(T, D, device=dev, dtype=dtype)
    want = _step(lambda v: block(v)[0], block, x, dout)
    # without reentry, the recomputation ends with an exception out of the pack hook of the last tensor it needs
    assert _same(_step(lambda v: checkpoint(lambda u: block(u)[0], v, use_reentrant=False), block, x, dout), want)
    assert _same(_step(lambda v: checkpoint(lambda u: block(u)[0], v, use_reentrant=True), block, x, dout), want)
    with torch.autograd.graph.save_on_cpu():
        assert _same(_step(lambda v: block(v)[0], block, x, dout), want)


def test_an_exception_of_a_pack_hook_arrives_as_itself(dev):
    class Stop(Exception):
        pass

    def pack(t):
        raise Stop()

    block = _block(dev)
    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t), pytest.raises(Stop):
        block(torch.randn(T, D, device=dev, dtype=torch.bfloat16, requires_grad=True))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_a_traced_block_computes_on_its_inputs(dev, dtype):
    block = _block(dev, dtype)
    x, x2, dout = (torch.randn(T, D, device=dev, dtype=dtype) for _ in range(3))

    class Hidden(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.block = block

        def forward(self, v):
            return self.block(v)[0]

    traced = torch.jit.trace(Hidden(), (x,), check_trace=False)
    with torch.no_grad():
        assert torch.equal(traced(x2), block(x2)[0])
    assert _same(_step(traced, block, x2, dout), _step(lambda v: block(v)[0], block, x2, dout))


@pytest.mark.parametrize("grad", [True, False])
def test_forward_mode_is_refused(dev, grad):
    import torch.autograd.forward_ad as fwad
    block = _block(dev).requires_grad_(False)
    x = torch.randn(T, D, device=dev, dtype=torch.bfloat16)
    with torch.set_grad_enabled(grad), fwad.dual_level(), pytest.raises(RuntimeError, match="(?i)jvp|forward"):
        block(fwad.make_dual(x, torch.randn_like(x)))


def test_weights_that_do_not_fit_the_layer_are_refused(dev):
    x = torch.randn(T, D, device=dev, dtype=torch.bfloat16)
    for name, shape in (("w1", ((E - 1) * F, D)), ("w2", (E * F // 2, D)), ("w3", (E * F, D // 2)), ("router", (E - 1, D)),
                        ("lora_A_w1", (E * D // 2, R)), ("lora_B_w2", (E * F // 2, R)), ("lora_A_w3", (E * D, R // 2))):
        block = _block(dev)
        setattr(block, name, torch.nn.Parameter(torch.zeros(shape, device=dev, dtype=torch.bfloat16)))
        with pytest.raises(RuntimeError):
            block(x)


def test_weights_and_factors_in_other_layouts_take_the_same_route(dev):
    """Non-contiguous weights are laid out on the way in, non-contiguous adapter storage is read through views: the same bits."""
    block = _block(dev)
    x, dout = (torch.randn(T, D, device=dev, dtype=torch.bfloat16) for _ in range(2))
    want = _step(lambda v: block(v)[0], block, x, dout)
    for name, _ in list(block.named_parameters()):
        p = getattr(block, name)
        wide = torch.zeros(p.size(0), 2 * p.size(1), device=dev, dtype=p.dtype)
        wide[:, ::2] = p.detach()
        if name != "router":
            setattr(block, name, torch.nn.Parameter(wide[:, ::2], requires_grad=p.requires_grad))
    assert _same(_step(lambda v: block(v)[0], block, x, dout), want)


def _routing(dev, t=T, k=K):
    import moe_distributed_training_amd as moe
    idx = torch.randint(0, E, (t, k), generator=torch.Generator().manual_seed(3)).to(dev)
    sei, ssi = moe.flatten_and_sort(idx, E)
    return (sei, ssi) + moe.padded_block_indices(sei, E)


def _factor(dev, *shape):
    return (torch.randn(shape, device=dev) * 0.05).bfloat16().requires_grad_(True)


@pytest.mark.parametrize("lora", [True, False])
def test_gradients_of_gates_over_a_grouped_output_are_refused(dev, lora):
    """The gradient of the combined output has one row per token; a grouped output has one per assignment."""
    import moe_distributed_training_amd as moe
    sei, ssi, pbi, eo = _routing(dev)
    x, w, gates = _factor(dev, T, D), (torch.randn(E, D, F, device=dev) * 0.05).bfloat16(), torch.rand(T, K, device=dev)
    if lora:
        y = moe.parallel_linear_lora(x, w, _factor(dev, E, D, R), _factor(dev, E, R, F), R, 32.0, K, sei, ssi, pbi, eo, gates, False, True)
    else:
        y = moe.parallel_linear(x, w, K, sei, ssi, pbi, eo, gates, False, True)
    with pytest.raises(AssertionError, match="token order"):
        y.sum().backward()


def test_gradients_without_assignments_are_refused(dev):
    import moe_distributed_training_amd as moe
    x, w, none = _factor(dev, T, D), (torch.randn(E, D, F, device=dev) * 0.05).bfloat16(), torch.zeros(0, dtype=torch.int64, device=dev)
    y = moe.parallel_linear(x, w, 0, none, none, None, torch.zeros(E, dtype=torch.int64, device=dev))
    assert y.shape == (0, F)
    with pytest.raises(AssertionError, match="assignments"):
        y.sum().backward()


@pytest.mark.parametrize("lora,weight_grad", [(True, False), (False, True), (False, False)])
def test_backward_of_a_projection_holds_one_copy_of_its_rows(dev, lora, weight_grad):
    """Peak memory: gathered X and the rows of dX share a buffer, and without adapters and weight gradients X is not gathered at all."""
    import moe_distributed_training_amd as moe
    from moe_distributed_training_amd._lib import MOE_BF16, lib
    t, d, n = 4096, 4096, 256
    L = t * K
    sei, ssi, pbi, eo = _routing(dev, t)
    x, w = _factor(dev, t, d), (torch.randn(E, d, n, device=dev) * 0.02).bfloat16().requires_grad_(weight_grad)
    if lora:
        y = moe.parallel_linear_lora(x, w, _factor(dev, E, d, R), _factor(dev, E, R, n), R, 32.0, K, sei, ssi, pbi, eo)
    else:
        y = moe.parallel_linear(x, w, K, sei, ssi, pbi, eo)
    dout = torch.ones_like(y)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated(dev)
    torch.cuda.reset_peak_memory_stats(dev)
    y.backward(dout)
    grown = torch.cuda.max_memory_allocated(dev) - before
    workspaces = [lib.moe_scatter2scatter_workspace_bytes(L, E, n, d, R if lora else 0), t * d * 2]   # of the dX product, or its fan-out sum
    if lora:
        workspaces.append(lib.moe_group_bwd_ab_workspace_bytes(L, E, d, n, R, MOE_BF16))
    grads = (E * R * (d + n) * 2 if lora else 0) + (E * d * n * 2 if weight_grad else 0)
    rows = L * n * 2 + L * d * 2          # grouped dY; gathered X, then the rows of dX
    assert grown <= rows + max(workspaces) + grads + (4 << 20), (grown, rows, workspaces, grads)
