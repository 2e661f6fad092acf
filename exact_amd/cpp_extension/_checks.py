"""Argument checks with the reference's error convention
(exact/exact/cpp_extension/ext_common.h:2-27): RuntimeError with the same
message for non-device, non-contiguous, wrong-rank or wrong-dtype tensors.
fp32 everywhere; fp16 where the library has fp16 kernels (pack / unpack and the
mask activations), as the reference's AT_DISPATCH_FLOATING_TYPES_AND_HALF admits."""
import torch


def _fail(msg):
    raise RuntimeError(msg)


def on_device(t):
    """True for tensors the kernels may touch (device memory)."""
    return t.is_cuda


def plain_values(*tensors):
    """True where a kernel may stand in for differentiable operations on these
    tensors (None is skipped) without anyone missing them: no tensor subclass, no
    forward-mode tangent, no trace or compilation in progress, no dispatch mode
    listening; and where memory holds their values as they are: no wrapper of a
    function transform (vmap, a batched backward, functionalisation), no sparse
    layout, no negation still to be made."""
    if torch.compiler.is_compiling() or torch.jit.is_tracing() or torch._C._len_torch_dispatch_stack() > 0:
        return False
    unpack = torch.autograd.forward_ad.unpack_dual
    wrapped, batched = torch._C._functorch.is_functorch_wrapped_tensor, torch._C._functorch.is_legacy_batchedtensor
    return all(type(t) in (torch.Tensor, torch.nn.Parameter) and not wrapped(t) and not batched(t) and t.layout is torch.strided
               and not t.is_neg() and unpack(t).tangent is None for t in tensors if t is not None)


def recorded(*tensors):
    """True where operations on these tensors are being recorded for a derivative (a
    backward under create_graph): kernels that autograd knows nothing of would end
    the record without a word."""
    return torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in tensors)


def check_device_tensor(t, name, dim=None, dtypes=(torch.float32,)):
    if not isinstance(t, torch.Tensor):
        _fail(f"{name} must be a tensor!")
    if not on_device(t):
        _fail(f"{name} must be a CUDA tensor!")
    if not t.is_contiguous():
        _fail(f"{name} must be contiguous!")
    if dim is not None and t.dim() != dim:
        _fail(f"The dimension of {name} is not correct!")
    if t.dtype not in dtypes:
        _fail(f"The type of {name} is not correct!")


FLOAT_OR_HALF = (torch.float32, torch.float16)


def suffix(t):
    """Entry-point suffix for the element type of t."""
    return "f16" if t.dtype == torch.float16 else "f32"


def stream_ptr(t):
    """The handle of the current stream of t's device, as torch.cuda.current_stream(t.device).cuda_stream
    gives it; without the Stream object in between, 0.2 instead of 4 us."""
    return torch._C._cuda_getCurrentRawStream(t.get_device())


def ptr(t):
    return 0 if t is None else t.data_ptr()
