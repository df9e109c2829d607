"""Helpers shared by the SO3part / SO3vec classes (python/src/gelib/gelib_common.py:15-20 in the reference)."""
import functools

import torch


def without_torch_function(f):
    """f with the __torch_function__ hooks of the tensor subclasses off while it runs: the parts are torch.Tensor
    subclasses whose every size, shape or dtype would otherwise take a detour through Python (3 us each; a gather of three
    parts and its gradient spent more time there than on the GPU)."""
    @functools.wraps(f)
    def g(*args):
        with torch._C.DisableTorchFunctionSubclass():
            return f(*args)
    return g


def output(shape, x, y):
    """The complex64 tensor that receives a product of parts x and y, on the device of x.  Every element is written by one launch, so
    it starts uninitialised: at 65536 cells of (2, 32 channels) x (3, 32 channels) -> 4 the zero-fill and the reading of
    what it wrote made the forward pass 3.0 ms instead of 0.9.  A product with an empty operand launches nothing."""
    make = torch.empty if x.numel() and y.numel() else torch.zeros
    return make(shape, dtype=torch.complex64, device=x.device)


def resolved(*ts):
    """ts with copies in place of views that torch conjugates (or negates) on reading only: kernels read memory.  (Asked in one call of
    the extension: two methods of each of ten tensors are 4 us.)"""
    if backend().in_memory(*ts):
        return ts
    return tuple(t.resolve_conj().resolve_neg() for t in ts)


def packed(t):
    """t with its elements in memory as they read: contiguous, and no view that torch conjugates (or negates) on reading only, which
    contiguous() leaves as it is (the gradient of out.conj().sum() is one)."""
    return resolved(t)[0].contiguous()


def common_batch(x, y):
    assert x.dim() >= 1
    assert y.dim() >= 1
    if x.size(0) > 1 and y.size(0) > 1:
        assert x.size(0) == y.size(0)
    return max(x.size(0), y.size(0))


@functools.lru_cache(maxsize=None)
def backend():
    """The compiled extension; importing it fails loudly if it has not been built."""
    from gelib_amd import gelib_base
    return gelib_base
