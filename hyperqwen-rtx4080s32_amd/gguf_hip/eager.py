"""When an eager call may go to the library without torch's dispatcher, and the stream it goes to.

Both need torch names that are not public.  They are looked up once, here: where a torch release lacks
one, every call takes the op (and the stream comes from the public call), which is only slower."""
from __future__ import annotations

import torch
from torch.autograd import forward_ad, profiler

try:
    _dispatch_modes, _function_modes = torch._C._len_torch_dispatch_stack, torch._C._len_torch_function_stack
    _transforms, _jit_trace = torch._C._functorch.peek_interpreter_stack, torch._C._get_tracing_state
    _profiled, _functional = torch.autograd._profiler_enabled, torch._is_functional_tensor
    forward_ad._current_level, profiler._is_profiler_enabled, torch.Tensor._is_zerotensor
    _KNOWN = True
except AttributeError:
    _KNOWN = False
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def stream(device: torch.device) -> int:
    """The device's current stream as a raw handle (no Stream object is made)."""
    return torch.cuda.current_stream(device).cuda_stream if _raw_stream is None else _raw_stream(device.index)


def direct(*tensors: torch.Tensor | None) -> bool:
    """Whether an eager call may go to the library without the dispatcher: nothing traces, transforms
    or intercepts it (compile, fx and jit tracing, dispatch and function modes, functorch, forward-mode
    AD), no profiler records the ops, and no tensor needs more than its data pointer (subclasses, lazy
    negation, functional and zero tensors, autograd).  The dispatcher's share of a custom op call with
    its two list arguments is about 30 us, several times the launch of a small layer (8 us of GPU time
    for a 4096 x 4096 Q8_0 layer at one row, whose eager call took 46 us).  An ExecutionTraceObserver
    that runs without a profiler cannot be seen from here: it misses the op."""
    if (torch.compiler.is_compiling() or not _KNOWN or profiler._is_profiler_enabled or _profiled()
            or _dispatch_modes() or _function_modes() or _transforms() is not None or _jit_trace() is not None
            or forward_ad._current_level >= 0):
        return False
    grad = torch.is_grad_enabled()
    for t in tensors:
        if t is not None and ((type(t) is not torch.Tensor and type(t) is not torch.nn.Parameter) or t.is_neg()
                              or t._is_zerotensor() or _functional(t) or (grad and t.requires_grad)):
            return False
    return True
