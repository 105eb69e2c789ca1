"""Calls that the entry points refuse on the host, before anything is enqueued.  The tensors are fakes that only claim to lie on a GPU, so
every check runs without one; a call that got past its checks would fail differently where there is none, and not run where there is one."""
import warnings

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

pytestmark = pytest.mark.skipif(torch.cuda.is_available(), reason="a fake's pointer must not reach a kernel")

T, D, F, E, K, R = 24, 64, 128, 4, 2, 16
BF16, F32, I32 = torch.bfloat16, torch.float32, torch.int32
_MODE = FakeTensorMode(allow_non_fake_inputs=True)


def _fake(*shape, dtype=BF16, device="cuda:0"):
    with _MODE:
        return torch.empty(shape, dtype=dtype, device=device)


def _mlp_args(**changed):
    args = dict(x=_fake(T, D), w1=_fake(E, F, D), w2=_fake(E, F, D), w3=_fake(E, F, D), k=K, sorted_scattered_idxs=_fake(T * K, dtype=I32),
                expert_offsets=_fake(E, dtype=I32))
    return {**args, **changed}


def _linear_args(**changed):
    args = dict(inputs=_fake(T, D), expert_weights=_fake(E, D, F), k=K, sorted_expert_idxs=_fake(T * K, dtype=I32),
                sorted_scattered_idxs=_fake(T * K, dtype=I32), padded_block_idxs=None, expert_offsets=_fake(E, dtype=I32))
    return {**args, **changed}


def _refused(match, fn, *args, **kw):
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")   # (a fake's data pointer)
        with pytest.raises((RuntimeError, AssertionError), match=match):
            fn(*args, **kw)


def _factors(**changed):
    """a1, b1, a3, b3, a2, b2 as views (E, K, r) / (E, r, N)"""
    from moe_distributed_training_amd.megablocks_utils.moe_mlp import LoraViews
    v = dict(a1=_fake(E, D, R), b1=_fake(E, R, F), a3=_fake(E, D, R), b3=_fake(E, R, F), a2=_fake(E, F, R), b2=_fake(E, R, D))
    return LoraViews(**{**v, **changed})


def _layer_args(**changed):
    args = dict(x=_fake(T, D), wg=_fake(E, D), w1=_fake(E, F, D), w2=_fake(E, F, D), w3=_fake(E, F, D), top_k=K)
    return {**args, **changed}


ELSEWHERE = [("GPU only", "cpu"), ("same device", "cuda:1")]


@pytest.mark.parametrize("match,device", ELSEWHERE)
def test_gates_elsewhere_are_refused(match, device):
    import moe_distributed_training_amd as moe
    gates = _fake(T, K, dtype=F32, device=device)
    _refused(match, moe.fused_expert_mlp, **_mlp_args(gates=gates))
    _refused(match, moe.parallel_linear, **_linear_args(gates=gates))


@pytest.mark.parametrize("match,device", ELSEWHERE)
@pytest.mark.parametrize("name", ["a1", "b1", "a3", "b3", "a2", "b2"])
def test_adapter_factors_elsewhere_are_refused(match, device, name):
    import moe_distributed_training_amd as moe
    shape = getattr(_factors(), name).shape
    lora = _factors(**{name: _fake(*shape, device=device)})
    _refused(match, moe.fused_expert_mlp, **_mlp_args(lora=lora))
    _refused(match, moe.moe_layer_forward, **_layer_args(lora=lora))
    block = moe.ScatterMoEBlock(D, F, E, top_k=K, lora_r=R, dtype=BF16, device="meta")
    for n, p in list(block.named_parameters()):
        where = device if n == "lora_" + {"a2": "B_w2", "b2": "A_w2"}.get(name, name[0].upper() + "_w" + name[1]) else "cuda:0"
        setattr(block, n, torch.nn.Parameter(_fake(*p.shape, device=where), requires_grad=False))
    _refused(match, block, _fake(T, D))


@pytest.mark.parametrize("shape", [(T, K, 2), (T * K,), (T + 1, K), (T // 2, K), (K, T, 1)])
def test_gates_of_another_shape_are_refused(shape):
    import moe_distributed_training_amd as moe
    gates = _fake(*shape, dtype=F32)
    _refused("gates of", moe.fused_expert_mlp, **_mlp_args(gates=gates))
    _refused("gates of", moe.parallel_linear, **_linear_args(gates=gates))
    _refused("gates of", moe.parallel_linear_lora, **_linear_args(gates=gates), expert_lora_A=_fake(E, D, R), expert_lora_B=_fake(E, R, F), lora_r=R,
             lora_alp=32.0)


@pytest.mark.parametrize("shape", [(T, D, 2), (2, T, D), (D,)])
def test_inputs_that_are_no_matrix_are_refused(shape):
    import moe_distributed_training_amd as moe
    from moe_distributed_training_amd._lib import native
    _refused("takes", moe.moe_layer_forward, **_layer_args(x=_fake(*shape)))
    _refused("takes", native.router, _fake(*shape), _fake(E, D), K, True)


@pytest.mark.parametrize("name", ["w1", "w2", "w3"])
@pytest.mark.parametrize("shape", [(E, 2 * F, D), (E, F // 2, D), (E + 1, F, D), (E - 1, F, D), (E * F // 2, D), (E, F, D // 2), (E, F * D)])
def test_expert_weights_that_do_not_fit_are_refused(name, shape):
    import moe_distributed_training_amd as moe
    if name != "w1":   # (sizes are those of w1; its own misfits show in the others, or in the input's columns)
        _refused("do not fit", moe.fused_expert_mlp, **_mlp_args(**{name: _fake(*shape)}))
    _refused("fit", moe.moe_layer_forward, **_layer_args(**{name: _fake(*shape)}))


@pytest.mark.parametrize("name", ["w1", "w2", "w3"])
def test_expert_weights_of_another_type_are_refused(name):
    """Two 2-byte types in one call would be read bit for bit as one of them."""
    import moe_distributed_training_amd as moe
    _refused("throughout", moe.fused_expert_mlp, **_mlp_args(**{name: _fake(E, F, D, dtype=torch.float16)}))
    _refused("dtype", moe.moe_layer_forward, **_layer_args(**{name: _fake(E, F, D, dtype=torch.float16)}))


def test_rows_of_another_width_are_refused():
    import moe_distributed_training_amd as moe
    _refused("rows of", moe.fused_expert_mlp, **_mlp_args(x=_fake(T, 2 * D)))
    _refused("rows of", moe.fused_expert_mlp, **_mlp_args(x=_fake(T, D, 1)))


@pytest.mark.parametrize("name", ["a1", "b1", "a3", "b3", "a2", "b2"])
@pytest.mark.parametrize("change", ["experts", "fewer_experts", "rows", "rank", "dims"])
def test_adapter_factors_that_do_not_fit_are_refused(name, change):
    import moe_distributed_training_amd as moe
    shape = list(getattr(_factors(), name).shape)
    a_like = name[0] == "a"
    if change == "experts":
        shape[0] += 1
    elif change == "fewer_experts":
        shape[0] -= 1
    elif change == "rows":
        shape[1 if a_like else 2] //= 2
    elif change == "rank":
        shape[2 if a_like else 1] //= 2
    else:
        shape = [shape[0] * shape[1], shape[2]]
    lora = _factors(**{name: _fake(*shape)})
    _refused("adapter factor", moe.fused_expert_mlp, **_mlp_args(lora=lora))
    _refused("adapter factor", moe.moe_layer_forward, **_layer_args(lora=lora))
    _refused("six adapter", moe.fused_expert_mlp, **_mlp_args(lora=list(_factors())[:5]))


@pytest.mark.parametrize("a,b", [((E - 1, D, R), (E, R, F)), ((E, D, R), (E - 1, R, F)), ((E, D, R), (E, R, F, 1))])
def test_factors_of_a_projection_cover_every_expert(a, b):
    import moe_distributed_training_amd as moe
    _refused("every expert", moe.parallel_linear_lora, **_linear_args(), expert_lora_A=_fake(*a), expert_lora_B=_fake(*b), lora_r=R, lora_alp=32.0)


@pytest.mark.parametrize("shape", [(E - 1,), (0,), ()])
def test_offsets_that_do_not_cover_the_experts_are_refused(shape):
    import moe_distributed_training_amd as moe
    eo = _fake(*shape, dtype=I32)
    _refused("expert offsets", moe.fused_expert_mlp, **_mlp_args(expert_offsets=eo))
    _refused("expert offsets", moe.parallel_linear, **_linear_args(expert_offsets=eo))


@pytest.mark.parametrize("changed", [dict(sorted_scattered_idxs=(T * K + 1,)), dict(k=1), dict(k=0)])
def test_positions_beyond_the_rows_are_refused(changed):
    import moe_distributed_training_amd as moe
    args = {n: _fake(*v, dtype=I32) if isinstance(v, tuple) else v for n, v in changed.items()}
    _refused("positions of", moe.fused_expert_mlp, **_mlp_args(**args))


def test_grouped_rows_take_no_fan_out():
    """One row per assignment: with k of them for each row of X, most would be read past its end."""
    import moe_distributed_training_amd as moe
    _refused("grouped rows", moe.parallel_linear, **_linear_args(grouped_in=True))
    _refused("grouped rows", moe.scatter2scatter, _fake(T, D), _fake(E, D, F), _fake(T * K, dtype=I32), _fake(T * K, dtype=I32), K, x_grouped=True)


@pytest.mark.parametrize("transform", ["vmap", "grad", "jvp"])
def test_function_transforms_are_refused(transform):
    """Their tensors are wrappers without memory (plain CPU tensors inside here: the refusal comes before that matters)."""
    import moe_distributed_training_amd as moe
    x, wg, w, wt = torch.randn(3, T, D), torch.randn(E, D), torch.randn(E, F, D), torch.randn(E, D, F)
    i, o = torch.zeros(T * K, dtype=I32), torch.zeros(E, dtype=I32)
    calls = [lambda v: moe.moe_layer_forward(v, wg, w, w, w, K)[0], lambda v: moe.forward_router(v, wg, K)[0],
             lambda v: moe.fused_expert_mlp(v, w, w, w, K, i, o), lambda v: moe.parallel_linear(v, wt, K, i, i, None, o)]
    for f in calls:
        run = {"vmap": lambda: torch.vmap(f)(x), "grad": lambda: torch.func.grad(lambda v: f(v).sum())(x[0]),
               "jvp": lambda: torch.func.jvp(f, (x[0],), (x[0],))}[transform]
        _refused("function transforms", run)
