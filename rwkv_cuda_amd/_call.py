"""The two ways from Python into the library: the operators as C++ autograd functions, and single C-ABI entry points."""

import torch

from . import _lib

_ops = None


def ops():
    """The C++ autograd functions (csrc/autograd.cpp); loads the extension once."""
    global _ops
    if _ops is None:
        from . import binding
        _ops = binding.load().ops
    return _ops


def call(name, dev, *args):
    """Call one C-ABI entry point on torch's current stream of `dev`.  Tensors become raw pointers."""
    lib = _lib.load()
    with torch.cuda.device(dev):
        stream = torch.cuda.current_stream(dev).cuda_stream
        conv = [a.data_ptr() if isinstance(a, torch.Tensor) else a for a in args]
        _lib.check(getattr(lib, name)(stream, *conv))
