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


@pytest.mark.parametrize("r", [R, 0])   # r = 0: all weights' gradients, whose rows take the gate weights again
@pytest.mark.parametrize("turn", [lambda t: t.t().contiguous().t(), lambda t: torch.stack([t, t], -1)[..., 0]], ids=["columns", "every_other"])
def test_saved_gates_of_other_strides_change_no_bit(dev, r, turn):
    """A hook that hands the layer's scores, weights and choices back with other strides (same values)."""
    block = _block(dev, torch.bfloat16, r)
    x, dout = torch.randn(T, D, device=dev).bfloat16(), torch.randn(T, D, device=dev).bfloat16()
    want = _step(lambda v: block(v)[0], block, x, dout)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: turn(t) if t.dim() == 2 and t.shape[0] == T and t.shape[1] <= 8 else t):
        assert _same(_step(lambda v: block(v)[0], block, x, dout), want)


@pytest.mark.parametrize("dtype,what", [(torch.bfloat16, "linear"), (torch.float16, "linear"), (torch.bfloat16, "mlp"), (torch.float32, "block")])
@pytest.mark.parametrize("turn", [lambda t: t.t().contiguous().t(), lambda t: torch.stack([t, t], -1)[..., 0]], ids=["columns", "every_other"])
def test_saved_gates_of_single_calls_may_have_other_strides(dev, dtype, what, turn):
    """The same for the gates of a projection (both of its backward routes), of the expert MLP (with its weights' gradients) and of the unfused layer."""
    import moe_distributed_training_amd as moe
    from moe_distributed_training_amd.megablocks_utils.router import sort_assignments
    torch.manual_seed(1)
    g = lambda *s: (torch.randn(*s, device=dev) * 0.1).to(dtype).requires_grad_(True)
    idx = torch.stack([torch.randperm(E, device=dev)[:K] for _ in range(T)]).int()
    sei, ssi, _, offs, _ = sort_assignments(idx, E)
    x, gates, dout = g(T, D), torch.rand(T, K, device=dev).requires_grad_(True), torch.randn(T, F if what == "linear" else D, device=dev).to(dtype)
    if what == "linear":
        w, leaves = g(E, D, F).detach(), [x, gates, g(E, D, R), g(E, R, F)]
        call = lambda: moe.parallel_linear_lora(x, w, leaves[2], leaves[3], R, 32.0, K, sei, ssi, None, offs, gates=gates)
    elif what == "mlp":
        leaves = [x, gates, g(E, F, D), g(E, F, D), g(E, F, D)]
        call = lambda: moe.fused_expert_mlp(x, leaves[2], leaves[3], leaves[4], K, ssi, offs, gates=gates)
    else:
        block = _block(dev, dtype, 0)
        leaves = [x] + list(block.parameters())
        call = lambda: block(x)[0]

    def step(hook):
        for t in leaves:
            t.grad = None
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, hook):
            call().backward(dout)
        return [t.grad for t in leaves]
    want = step(lambda t: t)
    assert _same(step(lambda t: turn(t) if t.shape == (T, K) and t.is_floating_point() else t), want)


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


class _Call(torch.nn.Module):
    """One call of an entry point below the block, its factors, gates and router weight as parameters."""

    def __init__(self, dev, which):
        import moe_distributed_training_amd as moe
        super().__init__()
        torch.manual_seed(5)
        self.which, self.moe = which, moe
        self.sei, self.ssi, self.pbi, self.eo = _routing(dev)
        shapes = {"linear": [(E, D, R), (E, R, F), (T, K)], "router": [(E, D)],
                  "mlp": [(E, D, R), (E, R, F), (E, D, R), (E, R, F), (E, F, R), (E, R, D), (T, K)]}[which]
        self.p = torch.nn.ParameterList([torch.nn.Parameter((torch.randn(s, device=dev) * 0.05).bfloat16()) for s in shapes])
        self.w = [(torch.randn(E, F, D, device=dev) * 0.05).bfloat16() for _ in range(3)]

    def forward(self, x):
        p = list(self.p)
        if self.which == "linear":
            return self.moe.parallel_linear_lora(x, self.w[0].permute(0, 2, 1), p[0], p[1], R, 32.0, K, self.sei, self.ssi, self.pbi, self.eo, p[2])
        if self.which == "router":
            return self.moe.forward_router(x, p[0], K)[1]
        from moe_distributed_training_amd.megablocks_utils.moe_mlp import LoraViews
        return self.moe.fused_expert_mlp(x, *self.w, K, self.ssi, self.eo, LoraViews(*p[:6]), 32.0, p[6])


CALLS = ["linear", "mlp", "router"]


def _call_case(dev, which):
    call = _Call(dev, which)
    x, x2 = (torch.randn(T, D, device=dev, dtype=torch.bfloat16) for _ in range(2))
    with torch.no_grad():
        dout = torch.randn_like(call(x))
    return call, x, x2, dout


@pytest.mark.parametrize("which", CALLS)
def test_checkpointing_and_hooks_of_single_calls_change_no_bit(dev, which):
    from torch.utils.checkpoint import checkpoint
    call, x, _, dout = _call_case(dev, which)
    want = _step(call, call, x, dout)
    for reentrant in (False, True):
        assert _same(_step(lambda v: checkpoint(call, v, use_reentrant=reentrant), call, x, dout), want)
    with torch.autograd.graph.save_on_cpu():
        assert _same(_step(call, call, x, dout), want)
    again = x.detach().requires_grad_(True)
    out = call(again)
    first = torch.autograd.grad(out, [again, *call.parameters()], dout, retain_graph=True)
    assert _same(torch.autograd.grad(out, [again, *call.parameters()], dout), first) and _same(first, want[1:])   # a second pass over one graph


@pytest.mark.parametrize("which", CALLS)
def test_traced_single_calls_compute_on_their_inputs(dev, which):
    call, x, x2, dout = _call_case(dev, which)
    traced = torch.jit.trace(call, (x,), check_trace=False)
    with torch.no_grad():
        assert torch.equal(traced(x2), call(x2))
    assert _same(_step(traced, call, x2, dout), _step(call, call, x2, dout))


@pytest.mark.parametrize("which", CALLS)
@pytest.mark.parametrize("grad", [True, False])
def test_forward_mode_of_single_calls_is_refused(dev, which, grad):
    import torch.autograd.forward_ad as fwad
    call, x, _, _ = _call_case(dev, which)
    call.requires_grad_(False)
    with torch.set_grad_enabled(grad), fwad.dual_level(), pytest.raises(RuntimeError, match="(?i)jvp|forward"):
        call(fwad.make_dual(x, torch.randn_like(x)))


@pytest.mark.parametrize("gates_dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gates_of_any_type(dev, oracle, dtype, gates_dtype):
    """Gates keep a type of their own, whatever that of the rows, and so does their gradient."""
    import moe_distributed_training_amd as moe
    from moe_distributed_training_amd.megablocks_utils.moe_mlp import LoraViews
    from _metrics import rel
    torch.manual_seed(8)
    rn = lambda *s, std=0.05: (torch.randn(*s) * std).to(dtype)
    f32 = lambda t: t.detach().float().clone().requires_grad_(True)
    on = lambda t: t.detach().to(dev).requires_grad_(True)
    x, w, gates = rn(T, D, std=1.0), [rn(E, F, D) for _ in range(3)], torch.rand(T, K).to(gates_dtype)
    idx = torch.stack([torch.randperm(E)[:K] for _ in range(T)])
    sei, ssi = oracle.flatten_and_sort(idx)
    eo = torch.bincount(sei, minlength=E).cumsum(0)
    fac = [rn(E, D, R), rn(E, R, F), rn(E, D, R), rn(E, R, F), rn(E, F, R), rn(E, R, D)]

    def compare(out, xg, gg, ref, xo, go):
        dout = torch.randn_like(ref).to(dtype)
        ref.backward(dout.float())
        out.backward(dout.to(dev))
        assert gg.grad.dtype == gates_dtype
        for got, want in ((out, ref), (xg.grad, xo.grad), (gg.grad, go.grad)):
            assert rel(got, want) < 1e-2

    xo, go, xg, gg = f32(x), f32(gates), on(x), on(gates)
    ref = oracle.parallel_linear_lora(xo, w[0].float().permute(0, 2, 1), fac[0].float(), fac[1].float(), R, 32.0, K, sei, ssi, None, eo, go, False, False)
    compare(moe.parallel_linear_lora(xg, w[0].to(dev).permute(0, 2, 1), fac[0].to(dev), fac[1].to(dev), R, 32.0, K, sei.to(dev), ssi.to(dev), None,
                                     eo.to(dev), gg), xg, gg, ref, xo, go)
    xo, go, xg, gg = f32(x), f32(gates), on(x), on(gates)
    lo = {"w1": (fac[0].float(), fac[1].float()), "w3": (fac[2].float(), fac[3].float()), "w2": (fac[4].float(), fac[5].float())}
    ref, _ = oracle.moe_block(xo, None, w[0].float(), w[1].float(), w[2].float(), K, lo, 32.0, routing=(go, idx))
    compare(moe.fused_expert_mlp(xg, w[0].to(dev), w[1].to(dev), w[2].to(dev), K, ssi.to(dev), eo.to(dev), LoraViews(*(t.to(dev) for t in fac)), 32.0,
                                 gg), xg, gg, ref, xo, go)
