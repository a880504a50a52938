"""megablocks/layers/common.py:9-26."""
import torch

from megablocks_amd import _lib
from megablocks_amd.layers.arguments import Arguments


def dtype(args: Arguments):
    if args.fp16:
        return torch.float16
    elif args.bf16:
        return torch.bfloat16
    return None


def cast_if_autocast_enabled(tensor):
    if torch.is_autocast_enabled():
        if tensor.device.type == 'cuda':
            target = _lib.autocast_gpu_dtype()
        elif tensor.device.type == 'cpu':
            target = torch.get_autocast_cpu_dtype()
        else:
            raise NotImplementedError()
        return tensor.to(dtype=target)
    return tensor


def only_computed(autocast: bool = False) -> bool:
    """Whether operations are carried out as they are called and nothing else: not traced, compiled, transformed (torch.func),
    differentiated forward or, unless `autocast` says that the caller sees to that, cast, all of which act on torch's operators and see
    nothing of a raw launch.  A torch that does not say counts as one that is doing it."""
    return not ((not autocast and torch.is_autocast_enabled()) or torch.compiler.is_compiling() or torch.jit.is_tracing() or
                getattr(torch._C, '_are_functorch_transforms_active', lambda: True)() or
                getattr(torch.autograd.forward_ad, '_current_level', 0) >= 0)   # -1: outside of any dual level
