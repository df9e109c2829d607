"""SO3weights / SO3linear: the channel-mixing linear layer that consumes a product
(python/src/gelib/SO3weights.py:22-85; SO3vec.__mul__, python/src/gelib/SO3vec.py:174-177).  One complex
(n_in, n_out) matrix per l, applied to the channel index of every part.  The reference does this with torch.matmul; on
the GPU the product of a part with its matrix and the gradient with respect to the part run on the library's
matrix-core kernels for tall, skinny complex matrices (mix_channels below), as does the gradient with respect to the
matrix; tensors on the host stay with torch."""
import functools

import torch

from gelib_amd.SO3type import SO3type
from gelib_amd.gelib_common import packed, resolved


class MixChannelsFn(torch.autograd.Function):
    """r = x w over the last index of a contiguous complex64 GPU tensor x, w of shape (n_in, n_out)."""

    @staticmethod
    def forward(ctx, x, w):
        from gelib_amd import cabi
        ctx.save_for_backward(x, w)
        r = torch.empty(x.shape[:-1] + (w.shape[1],), dtype=x.dtype, device=x.device)
        cabi.part_mix_channels(r, x, w)
        return r

    @staticmethod
    def backward(ctx, g):
        from gelib_amd import cabi
        x, w = ctx.saved_tensors
        gx = gw = None
        g = packed(g)
        if ctx.needs_input_grad[0]:
            if cabi.mix_channels_ok(g):
                gx = torch.empty_like(x)
                cabi.part_mix_channels(gx, g, w, adjoint=True)
            else:
                gx = torch.matmul(g, w.conj().transpose(0, 1))
        if ctx.needs_input_grad[1]:
            gw = torch.empty_like(w)
            cabi.part_mix_channels_wgrad(gw, x, g)
        return gx, gw


def mix_channels(x, w):
    """torch.matmul(x, w) for a part x (..., n_in) and a matrix w (n_in, n_out): on the GPU through the library's kernel
    when the part is complex64 with an even number of channels, else torch's own matmul."""
    if x.is_cuda and x.dtype == torch.complex64 and w.dtype == torch.complex64 and w.dim() == 2 and x.numel() > 0:
        from gelib_amd import cabi
        xp = packed(x.as_subclass(torch.Tensor))
        wp = packed(w.as_subclass(torch.Tensor))
        if cabi.mix_channels_ok(xp):
            return MixChannelsFn.apply(xp, wp)
    return torch.matmul(x, w)


class MixPartsFn(torch.autograd.Function):
    """x_k w_k for all parts of a vector in one call, any channel counts; contiguous complex64 GPU tensors.  classes: what the
    results are (mix_channels gives tensors, torch.matmul of a part with an odd number of channels its class)."""

    @staticmethod
    def forward(ctx, k, classes, *args):
        from gelib_amd import cabi
        xs, ws = list(args[:k]), list(args[k:])
        ctx.k = k
        ctx.set_materialize_grads(False)   # parts that a loss does not use get no gradients
        need = ctx.needs_input_grad[2:]    # a part is kept for the gradient of its matrix, a matrix for that of its part
        ctx.save_for_backward(*[t if n else None for t, n in zip(args, need[k:] + need[:k])])
        rs = [torch.empty(x.shape[:-1] + w.shape[1:], dtype=x.dtype, device=x.device) for x, w in zip(xs, ws)]
        cabi.vec_mix_channels(rs, xs, ws, 0)
        return tuple(r if c is torch.Tensor else r.as_subclass(c) for r, c in zip(rs, classes))

    @staticmethod
    def backward(ctx, *gs):
        from gelib_amd import cabi
        k = ctx.k
        xs, ws = ctx.saved_tensors[:k], ctx.saved_tensors[k:]
        need = ctx.needs_input_grad[2:]
        gs = [None if g is None else packed(g.as_subclass(torch.Tensor)) for g in gs]
        gx, gw = [None] * k, [None] * k
        if torch.is_grad_enabled():   # a graph of the gradients is wanted: torch's own operations
            for i, (x, w, g) in enumerate(zip(xs, ws, gs)):
                if g is None:
                    continue
                if need[i]:
                    gx[i] = torch.matmul(g, w.conj().transpose(0, 1))
                if need[k + i]:
                    gw[i] = torch.matmul(x.reshape(-1, x.shape[-1]).conj().transpose(0, 1), g.reshape(-1, g.shape[-1]))
            return tuple([None, None] + gx + gw)
        todo = [i for i in range(k) if need[i] and gs[i] is not None]
        if todo:
            for i in todo:
                gx[i] = torch.empty(gs[i].shape[:-1] + ws[i].shape[:1], dtype=gs[i].dtype, device=gs[i].device)
            cabi.vec_mix_channels([gx[i] for i in todo], [gs[i] for i in todo], [ws[i] for i in todo], 1)
        todo = [i for i in range(k) if need[k + i] and gs[i] is not None]
        if todo:
            for i in todo:
                gw[i] = torch.empty(xs[i].shape[-1:] + gs[i].shape[-1:], dtype=gs[i].dtype, device=gs[i].device)
            cabi.vec_mix_channels([gw[i] for i in todo], [xs[i] for i in todo], [gs[i] for i in todo], 2)
        return tuple([None, None] + gx + gw)


def plain_autograd():
    """False inside forward-mode derivatives, function transforms, tracing and dispatch modes (shapes without data, counters of
    operations), which only torch's own operations support."""
    return (torch.autograd.forward_ad._current_level < 0 and torch._C._functorch.peek_interpreter_stack() is None and
            torch._C._len_torch_dispatch_stack() == 0 and torch._C._get_tracing_state() is None and
            not torch.compiler.is_compiling())


def one_launch_holds(xs, ws):
    """Do the tiles of all parts fit a launch of vec_mix_channels, in either direction (2^24 blocks of at least 64 rows and 32
    columns)?  Rows beyond that stay with torch's product."""
    return sum((x.numel() // w.shape[0] + 64) * (max(w.shape) // 32 + 1) for x, w in zip(xs, ws)) <= 1 << 30


def matmul_class(x, w):
    """The class of torch.matmul(x, w); None where only torch can tell (classes with hooks of their own, or two that know nothing of
    each other).  A parameter is as a tensor there."""
    kinds = {type(t) for t in (x, w)} - {torch.Tensor, torch.nn.Parameter}
    if not kinds:
        return torch.Tensor
    c = kinds.pop()
    hook = getattr(c.__torch_function__, "__func__", None)
    return c if not kinds and hook is torch.Tensor.__torch_function__.__func__ else None


def torch_is_faster(x, w):
    """Is torch's product of a part with an odd number of channels over before the call of the library is made?  All parts of a vector in
    one call / part by part, forward and backward, 1 to 101 channels, 5 and 24 outputs: one part, 4 to 512 rows 1.7 to 1.9, 1024 1.11, 2048
    .58; up to l = 1, 384 rows 1.45, 1536 .72; l = 2, 640 1.28, 2560 .41; l = 4, 288 1.17, 1152 .73; l = 6, 416 1.08, 1664 .5 (torch's
    gradient of a matrix takes .3 ms from about a thousand rows on, and a millisecond every eight thousand).  Without that gradient: 1.7
    for one part, 1.4, 1.25, 1.07, .98 for two to seven, below about 20 MB of parts (l = 2, 18 MB 1.0, 37 MB .65; l = 4, 13 MB 1.07, 25 MB .8)."""
    if w.numel() >= LARGE_MATRIX:
        return False
    if torch.is_grad_enabled() and w.requires_grad:
        return x.numel() <= 1024 * x.shape[-1]
    return x.numel() < 2500000


# Elements of a matrix from which on mix.hip's kernels for long rows lose to the one call, also with one part of an even number of
# channels (one call / part by part, 4 to 8192 rows: 64 x 64 1.0, 512 x 6 1.07 to 1.17, 512 x 24 .73 to .95, 2048 x 6 .75 to .92, 2048 x 24 .3 to .6).
LARGE_MATRIX = 8192


def parts_of_one_call(pairs):
    """The parts that are mixed in one call of the library: even numbers of channels from two parts on (one part 1.03 to 1.13, two .96,
    three .9, five .84, seven .8 of the time part by part), odd ones where torch's product takes its time, and then all."""
    even, large = [], False
    for k, (x, w) in enumerate(pairs):
        if x.shape[-1] % 2 == 0:
            even.append(k)
            large = large or w.numel() >= LARGE_MATRIX
        elif not torch_is_faster(x, w):
            return list(range(len(pairs)))
    return even if large or len(even) > 1 else []


def mix_parts(xs, ws):
    """[torch.matmul(x, w) for x, w in zip(xs, ws)], on the GPU in one call of the library where that pays."""
    pairs = list(zip(xs, ws))
    with torch._C.DisableTorchFunctionSubclass():
        together = parts_of_one_call(pairs) if pairs and xs[0].is_cuda else []
        # (the library's launches go to the current device)
        if together and plain_autograd() and xs[0].get_device() == torch.cuda.current_device() and all(
                x.is_cuda and w.is_cuda and x.device == w.device == xs[0].device and x.dtype == w.dtype == torch.complex64 and w.dim() == 2 and
                x.numel() > 0 and w.numel() > 0 and x.shape[-1] == w.shape[0] for x, w in pairs) and one_launch_holds(xs, ws):
            from gelib_amd import cabi
            xp = [packed(pairs[k][0].as_subclass(torch.Tensor)) for k in together]
            classes = [torch.Tensor if cabi.mix_channels_ok(p) else matmul_class(*pairs[k]) for p, k in zip(xp, together)]
            if None in classes:
                together = []
        else:
            together = []
        if together:
            wp = [packed(pairs[k][1].as_subclass(torch.Tensor)) for k in together]
            mixed = dict(zip(together, MixPartsFn.apply(len(together), classes, *(xp + wp))))
    return [mixed[k] if k in together else mix_channels(*pairs[k]) for k in range(len(pairs))]


class SO3weights:

    def __init__(self, *args):
        self.parts = list(args)

    @classmethod
    def zeros(cls, tau_in, tau_out, device='cpu'):
        assert isinstance(tau_in, SO3type) and isinstance(tau_out, SO3type)
        R = SO3weights()
        for l in tau_in:
            R.parts.append(torch.zeros([tau_in[l], tau_out[l]], dtype=torch.complex64, device=device))
        return R

    @classmethod
    def randn(cls, tau_in, tau_out, device='cpu'):
        assert isinstance(tau_in, SO3type) and isinstance(tau_out, SO3type)
        R = SO3weights()
        for l in tau_in:
            R.parts.append(torch.randn([tau_in[l], tau_out[l]], dtype=torch.complex64, device=device))
        return R

    def requires_grad_(self):
        for w in self.parts:
            w.requires_grad_()
        return self

    def __repr__(self):
        return "<SO3weights " + ",".join("(%d,%d)" % (w.size(0), w.size(1)) for w in self.parts) + ">"


class SO3linear(torch.nn.Module):

    def __init__(self, tau_in, tau_out, device='cpu'):
        super().__init__()
        assert isinstance(tau_in, SO3type) and isinstance(tau_out, SO3type)
        self.W = SO3weights.randn(tau_in, tau_out, device)
        self.weights = torch.nn.ParameterList([torch.nn.Parameter(w) for w in self.W.parts])
        self.W.parts = list(self.weights)

    def forward(self, x):
        return x * self.W


class CGproductLinearFn(torch.autograd.Function):
    """CGproduct(x, y, maxl) * W with the product formed and consumed inside one kernel (forward).  The backward pass works
    through the batch a chunk at a time (gelib_hip_so3vec_cg_linear_bwd): the product's gradient, and the product where
    the matrices' gradients are not formed straight from the operands, exist only for the chunk at hand, in a workspace of
    at most BWD_WORKSPACE_BYTES, and nothing of the product's size is kept between the two passes.  The waves of a launch
    share the channel sums of a group of cells as the launch's size allows, so the last bits of a cell's result depend on
    the size of the batch it is in; from run to run they do not change."""

    BWD_WORKSPACE_BYTES = 8 << 30   # headline type, 32768 cells: 24.1 ms with 1 GiB, 19.1 with 4, 19.1 with 8, 18.5 with 28 (one chunk)

    @staticmethod
    def forward(ctx, k1, k2, maxl, *args):
        from gelib_amd import cabi
        xs, ys, ws = list(args[0:k1]), list(args[k1:k1 + k2]), list(args[k1 + k2:])
        ctx.k1, ctx.k2, ctx.maxl = k1, k2, maxl
        ctx.save_for_backward(*args)
        lead = list(xs[0].shape[:-2])
        out = [torch.empty(lead + [2 * l + 1, w.shape[1]], dtype=torch.complex64, device=xs[0].device)
               for l, w in enumerate(ws)]
        if not cabi.so3vec_cg_linear_fwd(out, xs, ys, ws, accumulate=False):
            raise RuntimeError("CGproduct_linear: shapes outside what the fused kernel takes")
        return tuple(out)

    @staticmethod
    def backward(ctx, *gargs):
        from gelib_amd import cabi
        from gelib_amd.SO3vec import SO3vec
        k1, k2 = ctx.k1, ctx.k2
        saved = ctx.saved_tensors
        xs, ys, ws = list(saved[0:k1]), list(saved[k1:k1 + k2]), list(saved[k1 + k2:])
        need = ctx.needs_input_grad[3:]
        gs = [packed(g) for g in gargs]
        xg = [torch.empty_like(t, memory_format=torch.contiguous_format) for t in xs] if any(need[0:k1]) else None
        yg = [torch.empty_like(t, memory_format=torch.contiguous_format) for t in ys] if any(need[k1:k1 + k2]) else None
        wg = [torch.empty_like(t, memory_format=torch.contiguous_format) for t in ws] if any(need[k1 + k2:]) else None
        if cabi.so3vec_cg_linear_bwd(xg, yg, wg, gs, xs, ys, ws, accumulate=False,
                                     workspace_bytes=CGproductLinearFn.BWD_WORKSPACE_BYTES):
            grads = (xg or [None] * k1) + (yg or [None] * k2) + (wg or [None] * len(ws))
            return tuple([None, None, None] + [g if n else None for g, n in zip(grads, need)])
        if not torch.is_grad_enabled():
            # shapes that call does not take (odd channel counts): the product again, and the kernels for any counts
            from gelib_amd.SO3vec import SO3vec
            with torch._C.DisableTorchFunctionSubclass():
                P = list(SO3vec(*xs).CGproduct(SO3vec(*ys), ctx.maxl).parts.values())
                return tuple([None, None, None] + _mixed_product_grads(k1, k2, xs, ys, ws, [p.as_subclass(torch.Tensor) for p in P], gs, need,
                                                                               [p.shape for p in P]))
        return tuple([None, None, None] + _two_step_grads(k1, k2, ctx.maxl, saved, gs, need))


def _two_step_grads(k1, k2, maxl, saved, gs, need, graph=False):
    """Gradients of the product followed by its matrices through the two separate autograd functions; gs: None for a result that is
    not used; graph: a graph of the gradients themselves is wanted, back to the saved tensors and gs."""
    from gelib_amd.SO3vec import SO3vec
    with torch.enable_grad():
        # (views, so that a tensor which is both operands has a gradient for each)
        leaves = [t.view_as(t) if graph else t.detach().requires_grad_() for t in saved]
        x, y = SO3vec(*leaves[0:k1]), SO3vec(*leaves[k1:k1 + k2])
        out = x.CGproduct(y, maxl) * SO3weights(*leaves[k1 + k2:])
        outs = [(o, g) for o, g in zip(out.parts.values(), gs) if g is not None]
    wanted = [t for t, n in zip(leaves, need) if n]
    got = iter(torch.autograd.grad([o for o, _ in outs], wanted, [g for _, g in outs], create_graph=graph, allow_unused=True))
    return [next(got) if n else None for n in need]


def _mixed_product_grads(k1, k2, xs, ys, ws, P, gs, need, shapes):
    """Gradients of P_l W_l with P = CGproduct(x, y), of these shapes, at hand where a matrix needs a gradient: the
    matrices' in one call, the product's in one, and the product's backward pass.  gs: None for a result that is not used, whose
    matrix gets no gradient and whose part of the product a zero one."""
    from gelib_amd import cabi
    from gelib_amd.SO3vec import SO3vec_CGproductFn
    used = [i for i, g in enumerate(gs) if g is not None]
    wg = [None] * len(ws)
    todo = [i for i in used if need[k1 + k2 + i]]
    if todo:
        for i in todo:
            wg[i] = torch.empty_like(ws[i])
        cabi.vec_mix_channels([wg[i] for i in todo], [P[i] for i in todo], [gs[i] for i in todo], 2)
    xyg = [None] * (k1 + k2)
    if any(need[0:k1 + k2]):
        gP = [(torch.zeros if g is None else torch.empty)(s, dtype=xs[0].dtype, device=xs[0].device) for s, g in zip(shapes, gs)]
        cabi.vec_mix_channels([gP[i] for i in used], [gs[i] for i in used], [ws[i] for i in used], 1)
        xyg = SO3vec_CGproductFn.grads(k1, k2, xs + ys, gP, need)
    return [g if n else None for g, n in zip(list(xyg) + wg, need)]


class CGproductMixFn(torch.autograd.Function):
    """CGproduct(x, y, maxl) * W for the shapes the fused kernel does not take: the product is formed and kept, as the two
    separate functions keep it, but all its parts are mixed in one call, forward and backward.  part_cls: the class of the
    product's parts, which mixed parts of an odd number of channels have as well (torch.matmul's rule)."""

    @staticmethod
    def forward(ctx, part_cls, k1, k2, maxl, *args):
        from gelib_amd import cabi
        from gelib_amd.SO3vec import SO3vec
        xs, ys, ws = list(args[0:k1]), list(args[k1:k1 + k2]), list(args[k1 + k2:])
        ctx.k1, ctx.k2, ctx.maxl = k1, k2, maxl
        ctx.set_materialize_grads(False)   # a matrix whose result a loss does not use gets no gradient
        P = [p.as_subclass(torch.Tensor) for p in SO3vec(*xs).CGproduct(SO3vec(*ys), maxl).parts.values()]
        out = [torch.empty(p.shape[:-1] + w.shape[1:], dtype=p.dtype, device=p.device) for p, w in zip(P, ws)]
        cabi.vec_mix_channels(out, P, ws, 0)
        ctx.shapes = [p.shape for p in P]
        # the product is kept for the gradients of the matrices
        ctx.save_for_backward(*args, *[p if n else None for p, n in zip(P, ctx.needs_input_grad[4 + k1 + k2:])])
        return tuple(r.as_subclass(part_cls) if p.shape[-1] % 2 else r for r, p in zip(out, P))

    @staticmethod
    def backward(ctx, *gargs):
        k1, k2 = ctx.k1, ctx.k2
        saved = ctx.saved_tensors
        need = ctx.needs_input_grad[4:]
        args, P = list(saved[:len(need)]), list(saved[len(need):])
        gs = [None if g is None else packed(g.as_subclass(torch.Tensor)) for g in gargs]
        if all(g is None for g in gs):
            grads = [None] * len(need)
        elif torch.is_grad_enabled():   # a graph of the gradients is wanted
            grads = _two_step_grads(k1, k2, ctx.maxl, args, gs, need, graph=True)
        else:
            grads = _mixed_product_grads(k1, k2, args[0:k1], args[k1:k1 + k2], args[k1 + k2:], P, gs, need, ctx.shapes)
        return tuple([None, None, None, None] + grads)


def fused_linear_ok(x, y, W, maxl):
    """True when CGproduct(x, y, maxl) * W is a case of the fused kernel: complex64 parts on one GPU, contiguous, the same
    leading dimensions, l <= 4 and at most 16 channels everywhere, a product with exactly the parts l = 0..4."""
    xs, ys, ws = list(x.parts.values()), list(y.parts.values()), list(W.parts)
    ts = xs + ys + ws
    if not ts or not all(t.is_cuda and t.dtype == torch.complex64 and t.is_contiguous() and t.device == ts[0].device
                         for t in ts):
        return False
    if any(t.shape[:-2] != xs[0].shape[:-2] for t in xs + ys) or xs[0].numel() == 0:
        return False
    if max(x.parts) > 4 or max(y.parts) > 4 or any(t.shape[-1] > 16 for t in xs + ys):
        return False
    from gelib_amd import cabi
    taus = cabi.so3type_product(x.tau(), y.tau(), maxl)
    if sorted(taus) != [0, 1, 2, 3, 4] or len(ws) != 5:
        return False
    return all(w.dim() == 2 and w.shape[0] == taus[l] and 1 <= w.shape[1] <= 16 for l, w in enumerate(ws))


def mixed_product_ok(x, y, W, maxl):
    """True when CGproductMixFn takes CGproduct(x, y, maxl) * W: two vectors or two arrays of vectors of complex64 parts on one GPU,
    contiguous, the same leading dimensions, one matrix (a tensor or parameter) for every part of the product, and nothing that
    only torch's own operations support (forward-mode derivatives, function transforms)."""
    if len(W.parts) == 1:
        return False   # (the two steps: even counts 1.06, odd ones up to 512 rows 1.17 to 1.25 of their time here; two parts .91 to .99)
    from gelib_amd.SO3vec import SO3vec
    from gelib_amd.SO3vecArr import SO3vecArr
    if type(x) is not type(y) or type(x) not in (SO3vec, SO3vecArr) or any(type(w) not in (torch.Tensor, torch.nn.Parameter) for w in W.parts):
        return False
    xs, ys, ws = list(x.parts.values()), list(y.parts.values()), list(W.parts)
    ts = xs + ys + ws
    if not xs or not ys or not ws or not all(t.is_cuda and t.dtype == torch.complex64 and t.is_contiguous() and
                                             t.device == ts[0].device and t.numel() > 0 for t in ts):
        return False
    if any(t.shape[:-2] != xs[0].shape[:-2] for t in xs + ys) or any(w.dim() != 2 for w in ws):
        return False
    if not plain_autograd():
        return False
    from gelib_amd import cabi
    from gelib_amd.SO3vec import _one_channel_side
    if _one_channel_side(xs, ys) is not None and max(t.shape[-1] for t in xs + ys) > 64:
        return False   # (SO3vec.CGproduct repeats the channel there, and its backward pass is that of the Diag product)
    taus = cabi.so3type_product(x.tau(), y.tau(), maxl)
    if [w.shape[0] for w in ws] != list(taus.values()):
        return False
    cells = xs[0].numel() // (xs[0].shape[-1] * xs[0].shape[-2])
    return sum((cells * (2 * l + 1) + 64) * (max(w.shape) // 32 + 1) for l, w in zip(taus, ws)) <= 1 << 30   # one_launch_holds


def CGproduct_linear(x, y, W, maxl=-1):
    """x.CGproduct(y, maxl) * W (python/src/gelib/SO3vec.py:174-177 applied to the result of SO3vec.CGproduct).  On the GPU,
    for the shapes fused_linear_ok accepts, one kernel forms the product and multiplies it by the matrices without
    storing it; other shapes keep the product, and mix all its parts in one call.  What neither takes runs the two steps one after
    the other.  A vector of the class that the two steps give."""
    from gelib_amd.SO3vecArr import SO3partArr, SO3vecArr
    arrays = isinstance(x, SO3vecArr) and isinstance(y, SO3vecArr)
    if arrays and maxl is None:
        maxl = -1
    if fused_linear_ok(x, y, W, maxl):
        fn = CGproductLinearFn.apply
    elif mixed_product_ok(x, y, W, maxl):
        from gelib_amd.SO3part import SO3part
        fn = functools.partial(CGproductMixFn.apply, SO3partArr if arrays else SO3part)
    else:
        return x.CGproduct(y, maxl) * W
    from gelib_amd.SO3vec import SO3vec
    ts = resolved(*[t.as_subclass(torch.Tensor) for t in (*x.parts.values(), *y.parts.values(), *W.parts)])
    return (SO3vecArr if arrays else SO3vec)(*fn(len(x.parts), len(y.parts), maxl, *ts))
