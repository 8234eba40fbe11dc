"""Calls of the ops go straight to their implementation only where nothing but the kernel has a
part in them (ops._Op): every torch mechanism that must see a dispatched op still does, recorded
calls have the gradients of the dispatched op, and mutated operands' versions count up."""
from __future__ import annotations  # as in ops.py, whose op entry reads the parameters' declared types

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.utils._python_dispatch import TorchDispatchMode

from weightshared_torchtitan_amd import ops


class Seen(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.append(str(func))
        return func(*args, **(kwargs or {}))


def test_mechanisms_that_need_the_dispatcher_are_seen():
    assert not ops._dispatcher_only()
    with Seen():
        assert ops._dispatcher_only()
    with FakeTensorMode():
        assert ops._dispatcher_only()
    with torch.device("meta"):
        assert ops._dispatcher_only()
    with torch.autocast("cpu", dtype=torch.bfloat16):
        assert ops._dispatcher_only()
    with torch.autograd.forward_ad.dual_level():
        assert ops._dispatcher_only()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]):
        assert ops._dispatcher_only()
    seen = []
    torch.func.vmap(lambda t: (seen.append(ops._dispatcher_only()), t)[1])(torch.zeros(2))
    torch.func.grad(lambda t: (seen.append(ops._dispatcher_only()), t.sum())[1])(torch.zeros(2))
    torch.jit.trace(lambda t: (seen.append(ops._dispatcher_only()), t + 1)[1], torch.zeros(2), check_trace=False)
    assert seen == [True] * 3

    class Seer(torch.autograd.Function):
        @staticmethod
        def forward(ctx, t):
            return t * 2

        @staticmethod
        def backward(ctx, g):
            seen.append(ops._dispatcher_only())
            return g * 2

    x = torch.zeros(2, requires_grad=True)
    torch.autograd.grad(Seer.apply(x), x, torch.eye(2), is_grads_batched=True)
    assert seen == [True] * 4
    assert not ops._dispatcher_only()


def test_tensors_off_the_gpu_and_subclasses_go_to_the_dispatcher(monkeypatch):
    monkeypatch.setattr(ops.swiglu_op, "_fn", lambda *a: pytest.fail("called directly"))
    with pytest.raises((RuntimeError, NotImplementedError)):
        ops.swiglu_op(torch.zeros(2, 16, dtype=torch.bfloat16))
    assert ops.swiglu_op(torch.zeros(2, 16, dtype=torch.bfloat16, device="meta")).shape == (2, 8)
    assert ops.swiglu_op(gate_up=torch.zeros(2, 16, dtype=torch.bfloat16, device="meta")).shape == (2, 8)


ALL_OPS = sorted(n for n in vars(ops) if n.endswith("_op") and not n.startswith("_"))


@pytest.fixture(scope="module")
def probe():
    """An op made as the module's own are: a scaled copy, with a CUDA implementation and a gradient."""
    def entry_probe(x: torch.Tensor, s: float, n: int, flag: bool, sizes: list[int]) -> torch.Tensor:
        return x * s + n

    op = ops._custom_op("entry_probe")(entry_probe)
    op.register_fake(lambda x, s, n, flag, sizes: torch.empty_like(x))
    op.register_autograd(lambda ctx, g: (g * ctx.s, None, None, None, None),
                         setup_context=lambda ctx, inputs, output: setattr(ctx, "s", inputs[1]))
    return op


@pytest.mark.parametrize("name", ALL_OPS)
def test_ops_are_custom_op_definitions(name):
    """What torch.library takes and offers for a custom op it takes and offers for these."""
    op = getattr(ops, name)
    assert isinstance(op, torch.library.CustomOpDef)
    for method in ("register_kernel", "register_fake", "register_vmap", "register_autograd", "register_autocast",
                   "register_torch_dispatch", "set_kernel_enabled"):
        assert callable(getattr(op, method))


def test_torch_library_functions_take_the_ops(probe):
    x = torch.arange(6.0)
    torch.library.register_kernel(probe, "cpu", lambda x, s, n, flag, sizes: x * s + n)
    assert probe._direct  # a CPU kernel leaves the CUDA one in its place
    assert torch.equal(probe(x, 2.0, 1, False, [1]), 2 * x + 1)
    torch.library.register_vmap(probe, lambda info, dims, x, *a: (probe(x, *a), dims[0]))
    assert torch.equal(torch.func.vmap(lambda t: probe(t, 3.0, 0, True, [1, 2]))(x.view(2, 3)), 3 * x.view(2, 3))
    y = x.clone().requires_grad_()
    probe(y, 2.0, 1, False, []).sum().backward()
    assert torch.equal(y.grad, torch.full_like(x, 2.0))
    torch.library.opcheck(probe, (y, 2.0, 1, False, [1]))


@pytest.mark.gpu
def test_registered_kernels_and_formulas_have_the_last_word(gpu):
    def entry_late(x: torch.Tensor, s: float) -> torch.Tensor:
        return x * s

    op = ops._custom_op("entry_late")(entry_late)
    x = torch.ones(4, device=gpu, requires_grad=True)
    assert torch.equal(op(x.detach(), 2.0), 2 * x)
    op.register_autograd(lambda ctx, g: (ctx.saved_tensors[0] * g, None),  # a formula that keeps the output
                         setup_context=lambda ctx, inputs, output: ctx.save_for_backward(output))
    assert torch.equal(torch.autograd.grad(op(x, 3.0).sum(), x)[0], torch.full_like(x, 3.0))
    torch.library.register_kernel(op, "cuda", lambda x, s: x * 0 - s)
    assert torch.equal(op(x.detach(), 2.0), torch.full_like(x, -2.0))
    assert torch.equal(torch.autograd.grad(op(x, 2.0).sum(), x)[0], torch.full_like(x, -2.0))
    torch.library.opcheck(ops.swiglu_op, (torch.randn(3, 16, device=gpu).bfloat16(),))


@pytest.mark.parametrize("change", [{1: "2.0"}, {2: 1.5}, {2: None}, {4: [1.5]}, {4: 3}, {4: "1"}, {0: None}, {3: "yes"},
                                    {1: torch.tensor(2.0)}, {2: True}, {3: 1}, {4: (1, 2)}, {4: [True]}, {1: True}])
def test_arguments_off_the_schema_are_the_dispatchers(probe, monkeypatch, change):
    """Only arguments of the declared types go straight to the implementation: the others are converted
    or refused as in any call of a custom op."""
    args = [torch.zeros(2), 2.0, 1, False, [1]]
    for i, v in change.items():
        args[i] = v
    monkeypatch.setattr(probe, "_fn", lambda *a: pytest.fail("called directly"))
    seen = []
    monkeypatch.setattr(probe, "_op", lambda *a, **k: seen.append(a))
    monkeypatch.setattr(ops, "_PLAIN_TYPES", (OnGpu, *ops._PLAIN_TYPES))
    if args[0] is not None:
        args[0] = OnGpu()
    probe(*args)
    assert len(seen) == 1
    args = [OnGpu(), 2, 1, False, []]
    monkeypatch.setattr(probe, "_fn", lambda *a: seen.append("direct"))
    probe(*args)
    assert seen[1:] == ["direct"]


class OnGpu:
    """Stands for a tensor on the GPU in the route's checks."""
    is_cuda, requires_grad = True, False


@pytest.mark.gpu
def test_arguments_of_other_types_are_refused(gpu):
    x, w, _, a, b = _args(gpu, False)
    for op in (ops.lora_linear_op, torch.ops.wsl.lora_linear):
        for args in ((x, w, None, a[:8], b, "2.0"), (None, w, None, a[:8], b, 2.0), (x, w, None, a[:8], 3.0, 2.0)):
            with pytest.raises((RuntimeError, TypeError, AttributeError)):
                op(*args)
    for op in (ops.lora_linear_bcast_op, torch.ops.wsl.lora_linear_bcast):
        with pytest.raises((RuntimeError, TypeError)):
            op(x, w, None, a[:8], b, 2.0, 1.0, 1)
    for op in (ops.lora_linear_grouped_op, torch.ops.wsl.lora_linear_grouped):
        with pytest.raises((RuntimeError, TypeError)):
            op(x, w, None, a, b, 2.0, [128.0, 128.0, 128.0])


def _args(gpu, grad):
    g = torch.Generator(device="cuda").manual_seed(0)
    mk = lambda *s: torch.randn(*s, device=gpu, generator=g).bfloat16().requires_grad_(grad)  # noqa: E731
    return mk(2, 50, 256), mk(384, 256), None, mk(24, 256), mk(384, 8)


@pytest.mark.gpu
@pytest.mark.parametrize("name,tail", [("lora_linear", (2.0,)), ("lora_linear_grouped", (2.0, [128, 128, 128])),
                                       ("lora_linear_bcast", (2.0, 1, 1))])
def test_direct_calls_equal_dispatched_ones(gpu, name, tail):
    x, w, ws, a, b = _args(gpu, True)
    if name != "lora_linear_grouped":
        a = a[:8].detach().requires_grad_()
    direct, op = getattr(ops, name + "_op"), getattr(torch.ops.wsl, name)
    gy = torch.randn(2, 50, 384, device=gpu).bfloat16()
    got = []
    for f in (direct, op):
        packed = []
        with torch.autograd.graph.saved_tensors_hooks(lambda t: (packed.append(t.shape), t)[1], lambda t: t):
            y = f(x, w, ws, a, b, *tail)
        assert len(packed) == 4
        got.append([y, *torch.autograd.grad(y, [x, w, a, b], gy)])
        with torch.no_grad():
            got[-1].append(f(x, w, ws, a, b, *tail))
        assert not got[-1][-1].requires_grad and y.requires_grad
        for needs in ([x], [b], [a, w]):  # any subset of the inputs
            ins = [t if any(t is n for n in needs) else t.detach() for t in (x, w, a, b)]
            y = f(ins[0], ins[1], ws, ins[2], ins[3], *tail)
            got[-1] += torch.autograd.grad(y, needs, gy)
    for p, q in zip(*got):
        assert torch.equal(p, q)


@pytest.mark.gpu
def test_transforms_see_the_op(gpu):
    x, w, _, a, b = _args(gpu, False)
    a = a[:8]
    want = ops.lora_linear_op(x, w, None, a, b, 2.0)
    with Seen() as s:
        assert torch.equal(ops.lora_linear_op(x, w, None, a, b, 2.0), want)
    assert any("wsl.lora_linear" in n for n in s.names)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert torch.equal(ops.lora_linear_op(x.float(), w.float(), None, a, b, 2.0), want)
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(x, torch.ones_like(x))
        out = []
        for f in (ops.lora_linear_op, torch.ops.wsl.lora_linear):  # neither drops the tangent in silence
            try:
                out.append(torch.autograd.forward_ad.unpack_dual(f(dual, w, None, a, b, 2.0)).tangent is None)
            except (RuntimeError, NotImplementedError):
                out.append("raised")
        assert out[0] == out[1]


@pytest.mark.gpu
@pytest.mark.parametrize("name,tail", [("lora_linear", (2.0,)), ("lora_linear_bcast", (2.0, 1, 1))])
def test_batches_of_gradients(gpu, name, tail):
    """torch.autograd.grad over a batch of output gradients, one backward each (the grouped op's backward
    writes slices in place, which the batching does not take)."""
    x, w, _, a, b = _args(gpu, True)
    a = a[:8].detach().requires_grad_()
    y = getattr(ops, name + "_op")(x, w, None, a, b, *tail)
    gy = torch.randn(3, 2, 50, 384, device=gpu).bfloat16()
    got = torch.autograd.grad(y, [x, w, a, b], gy, is_grads_batched=True, retain_graph=True)
    for i in range(3):
        for g, want in zip(got, torch.autograd.grad(y, [x, w, a, b], gy[i], retain_graph=True)):
            assert torch.equal(g[i], want)


@pytest.mark.gpu
def test_mutated_operands_count_up(gpu):
    k = torch.randn(8, 128, device=gpu).bfloat16()
    kc = torch.zeros(2, 2, 4, 64, device=gpu, dtype=torch.bfloat16)
    vc = kc.clone()
    rope = torch.zeros(4, 128, device=gpu)
    kw = torch.ones(64, device=gpu, dtype=torch.bfloat16)
    for f in (ops.kv_norm_rope_op, torch.ops.wsl.kv_norm_rope):
        before = kc._version, vc._version, k._version
        f(k, k, kw, 1e-6, rope, kc, vc)
        assert kc._version > before[0] and vc._version > before[1] and k._version == before[2]
    with torch.inference_mode():
        ops.kv_norm_rope_op(k, k, kw, 1e-6, rope, torch.zeros_like(kc), torch.zeros_like(vc))


@pytest.mark.gpu
def test_calls_follow_the_current_stream(gpu):
    x, w, _, a, b = _args(gpu, False)
    a = a[:8]
    want = ops.lora_linear_op(x, w, None, a, b, 2.0)
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        assert ops._stream(x.device) == s.cuda_stream
        y = ops.lora_linear_op(x, w, None, a, b, 2.0)
    s.synchronize()
    assert ops._stream(x.device) == torch.cuda.current_stream().cuda_stream and torch.equal(y, want)


def test_fused_prompt_needs_plain_norms():
    """The prompt kernels stand for RMSNorm.forward: a norm that does anything else keeps the model
    on its modules."""
    from weightshared_torchtitan_amd.qwen3_shared import RMSNorm, SharedQwen3, SharedQwen3Args

    class Other(RMSNorm):
        pass

    m = SharedQwen3(SharedQwen3Args(dim=64, n_layers=2, n_unique_blocks=1, n_heads=1, n_kv_heads=1, head_dim=64,
                                    hidden_dim=64, vocab_size=64, embed_rank=64, lora_rank=8, max_seq_len=16))
    assert m._norms_plain()
    at = m.base_blocks[0].attention
    for other in (Other(64, 1e-6), torch.nn.Identity()):
        kept, at.q_norm = at.q_norm, other
        assert not m._norms_plain()
        at.q_norm = kept
    m.norm.forward = lambda x: x
    assert not m._norms_plain()
    del m.norm.forward
    for register in (at.k_norm.register_forward_hook, torch.nn.modules.module.register_module_forward_hook):
        h = register(lambda *_: None)
        assert not m._norms_plain()
        h.remove()
    h = torch.nn.modules.module.register_module_forward_pre_hook(lambda *_: None)
    assert not m._norms_plain()
    h.remove()
    assert m._norms_plain()
