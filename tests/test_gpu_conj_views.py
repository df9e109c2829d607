"""Operands that torch conjugates or negates on reading only (x.conj(), a negated view): the kernels read memory, so the products,
layers, gathers and harmonics have to work on what the tensor reads as.  Results and gradients are the bits that copies give."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

VIEWS = {"conj": lambda t: t.conj(), "neg": torch._neg_view, "both": lambda t: torch._neg_view(t.conj())}


def rand(shape, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.view_as_complex(torch.randn(*shape, 2, device="cuda", generator=g))


def parts(lead, tau, seed):
    return [rand((*lead, 2 * l + 1, n), seed + l).requires_grad_() for l, n in tau.items()]


def part_pair(cls, lead, l1, l2, n1, n2, diag, l):
    x, y = rand((*lead, 2 * l1 + 1, n1), 1).requires_grad_(), rand((*lead, 2 * l2 + 1, n2), 2).requires_grad_()

    def op(view):
        a, b = view(x).as_subclass(cls), view(y).as_subclass(cls)
        return [a.DiagCGproduct(b, l) if diag else a.CGproduct(b, l)]
    return [x, y], op


def vec_pair(cls, lead, tx, ty, maxl, diag):
    xs, ys = parts(lead, tx, 10), parts(lead, ty, 20)

    def op(view):
        x, y = cls(*[view(t) for t in xs]), cls(*[view(t) for t in ys])
        return list((x.DiagCGproduct(y, maxl) if diag else x.CGproduct(y, maxl)).parts.values())
    return xs + ys, op


def o3_pair(diag):
    import gelib_amd as gelib
    mus = [(0, 1), (1, -1), (2, 1)]
    xs, ys = [rand((5, 2 * l + 1, 3), 30 + l).requires_grad_() for l, _ in mus], [rand((5, 2 * l + 1, 3), 40 + l).requires_grad_() for l, _ in mus]

    def op(view):
        x, y = gelib.O3vec({mu: view(t) for mu, t in zip(mus, xs)}), gelib.O3vec({mu: view(t) for mu, t in zip(mus, ys)})
        out = list((x.DiagCGproduct(y, 2) if diag else x.CGproduct(y, 2)).parts.values())
        p, q = gelib.O3part(view(xs[1]), mus[1]), gelib.O3part(view(ys[2]), mus[2])
        return out + [(p.DiagCGproduct(q, (1, -1)) if diag else p.CGproduct(q, (1, -1))).as_subclass(torch.Tensor)]
    return xs + ys, op


def layer(L, n, out, lead=(9,), cls=None):
    import gelib_amd as gelib
    from gelib_amd import cabi
    cls = cls or gelib.SO3vec
    tau = {l: n for l in range(L + 1)}
    xs, ys = parts(lead, tau, 50), parts(lead, tau, 60)
    ws = [rand((c, out), 70 + l).requires_grad_() for l, c in cabi.so3type_product(tau, tau, L).items()]

    def op(view):
        return list(gelib.CGproduct_linear(cls(*[view(t) for t in xs]), cls(*[view(t) for t in ys]),
                                           gelib.SO3weights(*[view(w) for w in ws]), L).parts.values())
    return xs + ys + ws, op


def gathers():
    import gelib_amd as gelib
    xs = parts((1, 6), {0: 3, 2: 2}, 80)
    m = gelib.gather_map.sources_targets([0, 5, 2, 2], [1, 1, 0, 3], 6, 4)

    def op(view):
        return list(gelib.SO3vecArr(*[view(t) for t in xs]).gather(m).parts.values()) + [view(xs[1]).as_subclass(gelib.SO3partArr).gather(m)]
    return xs, op


def cases():
    import gelib_amd as gelib
    return {
        "part": part_pair(gelib.SO3part, (7,), 2, 1, 3, 4, False, 2), "part diag": part_pair(gelib.SO3part, (7,), 2, 1, 4, 4, True, 2),
        "part array": part_pair(gelib.SO3partArr, (2, 3), 1, 1, 3, 2, False, 1), "part array diag": part_pair(gelib.SO3partArr, (2, 3), 1, 1, 3, 3, True, 1),
        "vec": vec_pair(gelib.SO3vec, (6,), {0: 3, 1: 4, 2: 2}, {0: 2, 1: 5}, -1, False), "vec diag": vec_pair(gelib.SO3vec, (6,), {0: 3, 1: 3}, {0: 3, 1: 3}, 1, True),
        "one wide side": vec_pair(gelib.SO3vec, (6,), {0: 70, 1: 70}, {0: 1, 1: 1}, 1, False),
        "vec array": vec_pair(gelib.SO3vecArr, (2, 3), {0: 3, 1: 4}, {0: 2, 1: 5}, -1, False),
        "vec array diag": vec_pair(gelib.SO3vecArr, (2, 3), {0: 3, 1: 3}, {0: 3, 1: 3}, -1, True),
        "O(3)": o3_pair(False), "O(3) diag": o3_pair(True),
        "layer in one kernel": layer(4, 4, 8), "layer of arrays in one kernel": layer(4, 2, 4, (2, 5), gelib.SO3vecArr),
        "layer, odd": layer(2, 3, 5), "layer, even": layer(2, 4, 6), "gather": gathers(),
    }


NAMES = ["part", "part diag", "part array", "part array diag", "vec", "vec diag", "one wide side", "vec array", "vec array diag", "O(3)",
         "O(3) diag", "layer in one kernel", "layer of arrays in one kernel", "layer, odd", "layer, even", "gather"]


@pytest.mark.parametrize("view", list(VIEWS))
@pytest.mark.parametrize("name", NAMES)
def test_operands(name, view):
    leaves, op = cases()[name]

    def run(v):
        rs = [r.as_subclass(torch.Tensor) for r in op(v)]
        gs = [rand(tuple(r.shape), 100 + k) for k, r in enumerate(rs)]
        return [t.resolve_conj().resolve_neg() for t in rs + list(torch.autograd.grad(rs, leaves, gs))]
    got, want = run(VIEWS[view]), run(lambda t: VIEWS[view](t).resolve_conj().resolve_neg())
    assert all(torch.equal(a.as_subclass(torch.Tensor), b.as_subclass(torch.Tensor)) for a, b in zip(got, want))


def test_directions():
    import gelib_amd as gelib
    X = torch.randn(9, 3, 2, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    for l in (0, 1, 3):
        assert torch.equal(gelib.SO3part.spharm(l, torch._neg_view(X)), gelib.SO3part.spharm(l, -X))
        A, B = torch._neg_view(X).unsqueeze(1), (-X).unsqueeze(1)
        assert torch.equal(gelib.SO3partArr.spharm(l, A), gelib.SO3partArr.spharm(l, B))


def test_memory_is_not_read_in_their_place():
    """Entry points that take an address refuse such a view; the one that makes the result itself reads it."""
    from gelib_amd import cabi, gelib_base
    x, y, w = rand((4, 3, 2), 1), rand((4, 3, 2), 2), rand((2, 2), 3)
    r = torch.zeros(4, 3, 4, dtype=torch.complex64, device="cuda")
    for view in VIEWS.values():
        want = gelib_base.CGproduct(view(x).resolve_conj().resolve_neg(), y, 1)
        assert torch.equal(gelib_base.CGproduct(view(x), y, 1), want)
        with pytest.raises(RuntimeError, match="conjugat"):
            gelib_base.SO3part.view(view(x))
        with pytest.raises(RuntimeError, match="conjugat"):
            gelib_base.SO3vec.view([view(x)])
        with pytest.raises(ValueError, match="conjugat"):
            cabi.so3part_cg_fwd(r, view(x), y)
        with pytest.raises(ValueError, match="conjugat"):
            cabi.vec_mix_channels([torch.empty_like(x)], [view(x)], [w], 0)
        with pytest.raises(ValueError, match="conjugat"):
            cabi.vec_mix_channels([torch.empty_like(x)], [x], [view(w)], 0)
