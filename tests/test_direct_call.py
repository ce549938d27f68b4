"""When an eager linear call may skip the dispatcher: only plain tensors with nothing tracing,
transforming or intercepting; everything else keeps the custom op.  No kernel runs here."""
import pytest
import torch
import torch.autograd.forward_ad as fwad
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode


class _Sub(torch.Tensor):
    pass


def test_direct_only_for_plain_eager_tensors():
    from gguf_hip.ops import _direct

    x = torch.randn(4, 8)
    assert _direct(x, None, torch.nn.Parameter(x, requires_grad=False))
    g = torch.randn(4, 8, requires_grad=True)
    assert not _direct(x, g)
    with torch.no_grad():
        assert _direct(g)
    with torch.inference_mode():
        assert _direct(torch.randn(2))
    assert not _direct(x.as_subclass(_Sub))
    assert not _direct(torch._neg_view(x))
    assert not _direct(torch._efficientzerotensor((3,)))
    assert not _direct(torch._to_functional_tensor(x))
    mode = FakeTensorMode()
    with mode:
        assert not _direct(x)
        fake = torch.empty(3)
    assert not _direct(fake)
    with TorchDispatchMode():
        assert not _direct(x)
    with TorchFunctionMode():
        assert not _direct(x)
    with fwad.dual_level():
        assert not _direct(x)
    seen = []
    torch.func.vmap(lambda t: (seen.append(_direct(x)), t)[1])(x)
    torch.func.jvp(lambda t: (seen.append(_direct(x)), t)[1], (x,), (x,))
    torch.func.functionalize(lambda t: (seen.append(_direct(x)), t)[1])(x)
    torch.jit.trace(lambda t: (seen.append(_direct(t)), t + 1)[1], (x,), check_trace=False)
    assert seen and not any(seen), seen


def test_direct_write_bumps_the_output_version(monkeypatch):
    import types

    from gguf_hip import ops

    monkeypatch.setattr(ops, "_require_gpu", lambda t, what: None)
    monkeypatch.setattr(ops, "_grouped_into", lambda *a: None)   # the library writes past torch
    gl = types.SimpleNamespace(K=256, n_total=64, packed=torch.zeros(8, dtype=torch.uint8), descs=[], plans=[],
                               workspace=torch.zeros(8, dtype=torch.int32))
    x, out = (torch.ones(4, k, dtype=torch.bfloat16) for k in (256, 64))
    w = torch.ones(4, 64, dtype=torch.bfloat16, requires_grad=True)
    loss = (w * out).sum()   # saves out
    ops.mul_mat_grouped(x, gl, out=out)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        loss.backward()


def test_a_profiler_sees_the_op():
    import threading

    from gguf_hip.ops import _direct

    x, seen = torch.randn(4, 8), []
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]):
        seen.append(_direct(x))
        t = threading.Thread(target=lambda: seen.append(_direct(x)))
        t.start()
        t.join()
    with torch.autograd.profiler.profile():
        seen.append(_direct(x))
    assert seen == [False] * 3 and _direct(x)


@pytest.mark.parametrize("where,name", [
    (torch._C, "_len_torch_dispatch_stack"), (torch._C, "_len_torch_function_stack"), (torch._C, "_get_tracing_state"),
    (torch._C._functorch, "peek_interpreter_stack"), (torch.autograd, "_profiler_enabled"),
    (torch, "_is_functional_tensor"), (fwad, "_current_level"), (torch.autograd.profiler, "_is_profiler_enabled"),
], ids=lambda v: v if isinstance(v, str) else "")
def test_a_torch_without_one_of_the_names_takes_the_op(monkeypatch, where, name):
    import importlib.util

    from gguf_hip import eager

    monkeypatch.delattr(where, name)
    spec = importlib.util.spec_from_file_location("eager_without", eager.__file__)
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    no = mod.direct(torch.zeros(1))
    monkeypatch.undo()
    assert no is False and eager.direct(torch.zeros(1))


def test_the_stream_without_the_raw_handle(monkeypatch):
    import types

    from gguf_hip import eager

    monkeypatch.setattr(eager, "_raw_stream", None)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device: types.SimpleNamespace(cuda_stream=77))
    assert eager.stream(torch.device("cuda", 0)) == 77


@pytest.mark.gpu
def test_direct_and_dispatched_calls_agree(dev):
    import gguf_hip
    from gguf_hip import ops
    from gguf_hip.synth import random_shard

    gl = gguf_hip.pack_layer([random_shard(200, 512, 12, dev)], [200], [12])
    for M in (1, 20, 70):
        x = torch.randn(M, 512, device=dev).to(torch.bfloat16)
        b = torch.randn(200, device=dev).to(torch.bfloat16)
        y = ops.fused_mul_mat_gguf_grouped(x, gl.packed, gl.descs, gl.plans, gl.n_total, gl.workspace, b)
        assert torch.equal(gguf_hip.mul_mat_grouped(x, gl, b), y)
        wide = torch.zeros(M, 300, device=dev, dtype=torch.bfloat16)
        gguf_hip.mul_mat_grouped(x, gl, b, out=wide[:, 50:250])
        assert torch.equal(wide[:, 50:250], y) and not wide[:, :50].any() and not wide[:, 250:].any()
        with torch.enable_grad():   # an input that records a graph goes through the op
            z = gguf_hip.mul_mat_grouped(x.clone().requires_grad_(), gl, b)
        assert z.requires_grad and torch.equal(z.detach(), y)
        st = torch.cuda.Stream()
        st.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(st):
            w = gguf_hip.mul_mat_grouped(x, gl, b)
        torch.cuda.current_stream().wait_stream(st)
        assert torch.equal(w, y)
