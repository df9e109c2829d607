"""Channel mixing of all parts of a vector in one call (any channel counts) against numpy's complex128 matmul, and the layer
built on it against the two separate steps.  Tolerance: that of test_gpu_mix.py, 1e-6 + 4 eps32 times the sum of the moduli
of an element's terms (16 terms are added at a time here, so the chains are shorter than there)."""
import numpy as np
import pytest

from tests import gpu_util as U

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def cabi():
    assert torch.cuda.is_available()
    from gelib_amd import cabi as c
    c.lib()
    return c


def rand(shape, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.view_as_complex(torch.randn(*shape, 2, device="cuda", generator=g))


# (rows, n_in, n_out) per part: edges of the tiles (4, 8, 16, 32 columns; 64 and 128 rows; 16 terms a step), one of everything,
# sums long enough to be cut into pieces, parts of different sizes in one call, and more parts than a launch takes
CASES = [
    [(1, 1, 1)],
    [(129, 15, 4), (7, 17, 3)],
    [(128, 16, 8), (64, 33, 5), (3, 1, 7)],
    [(65, 31, 16), (63, 300, 9)],
    [(64, 2001, 32), (5, 7, 33), (1, 5, 70)],
    [(40000, 3, 3), (13, 4097, 2)],
    [(k + 1, 2 * k + 1, 3) for k in range(19)],
]


@pytest.mark.parametrize("mode", [-1, 0, 1])
@pytest.mark.parametrize("kind", [0, 1, 2])
@pytest.mark.parametrize("case", CASES, ids=[str(i) for i in range(len(CASES))])
def test_vec_mix(cabi, case, kind, mode):
    xs = [rand((rows, n_in), 1 + k) for k, (rows, n_in, _) in enumerate(case)]
    ws = [rand({0: (i, o), 1: (o, i), 2: (rows, o)}[kind], 50 + k) for k, (rows, i, o) in enumerate(case)]
    rs = [torch.full((i, o) if kind == 2 else (rows, o), float("nan"), dtype=torch.complex64, device="cuda") for rows, i, o in case]
    cabi.set_option("vec_mix", mode)   # -1 by the shape, 0 the matrix-core kernels wherever they can, 1 never
    try:
        cabi.vec_mix_channels(rs, xs, ws, kind)
    finally:
        cabi.set_option("vec_mix", -1)
    for r, x, w in zip(rs, xs, ws):
        hx, hw = U.host(x).astype(np.complex128), U.host(w).astype(np.complex128)
        a = hx.conj().T if kind == 2 else hx
        b = hw.conj().T if kind == 1 else hw
        tol = 1e-6 + 4 * np.finfo(np.float32).eps * (np.abs(a) @ np.abs(b))
        err = np.abs(U.host(r) - a @ b)
        assert (err <= tol).all(), "kind %d %s x %s: worst error / tolerance %.2f" % (kind, x.shape, w.shape, (err / tol).max())


def test_vec_mix_refuses(cabi):
    x, w, r = rand((5, 3), 1), rand((3, 2), 2), rand((5, 2), 3)
    with pytest.raises(ValueError):
        cabi.vec_mix_channels([r], [x], [rand((4, 2), 2)], 0)
    with pytest.raises(cabi.GelibHipError):   # a sum long enough to be cut, and no workspace
        import ctypes
        a, b, c = rand((4, 4096), 1), rand((4096, 2), 2), rand((4, 2), 3)
        P = ctypes.c_void_p * 1
        cabi.check(cabi.lib().gelib_hip_vec_mix_channels(1, P(c.data_ptr()), P(a.data_ptr()), P(b.data_ptr()),
                                                         (ctypes.c_int64 * 1)(4), (ctypes.c_int * 1)(4096), (ctypes.c_int * 1)(2),
                                                         0, None, 0, None))


@pytest.mark.parametrize("lx,ly,maxl,n1,n2,out,b", [(2, 2, 2, 4, 2, 5, 33), (3, 3, 3, 3, 3, 3, 130), (4, 4, 4, 3, 1, 3, 70),
                                                   (2, 1, -1, 2, 3, 8, 5), (4, 4, 4, 13, 6, 13, 22), (3, 3, 3, 16, 8, 20, 300)])
def test_layer_matches_the_two_steps(cabi, lx, ly, maxl, n1, n2, out, b):
    """Values and all gradients of CGproduct_linear where the fused kernels do not take it (l other than 0..4, odd counts),
    against the product and torch's matmul in complex128; a second pass gives the same bits."""
    import gelib_amd as gelib
    xs = [rand((b, 2 * l + 1, n1), l).requires_grad_() for l in range(lx + 1)]
    ys = [rand((b, 2 * l + 1, n2), 10 + l).requires_grad_() for l in range(ly + 1)]
    tau = cabi.so3type_product({l: n1 for l in range(lx + 1)}, {l: n2 for l in range(ly + 1)}, maxl)
    ws = [(rand((n, out), 20 + l) / np.sqrt(n)).requires_grad_() for l, n in tau.items()]
    gs = [rand((b, 2 * l + 1, out), 40 + l) for l in tau]

    def run():
        r = gelib.CGproduct_linear(gelib.SO3vec(*xs), gelib.SO3vec(*ys), gelib.SO3weights(*ws), maxl)
        rs = list(r.parts.values())
        return rs + list(torch.autograd.grad(rs, xs + ys + ws, gs))

    got, again = run(), run()
    assert all(torch.equal(a, c) for a, c in zip(got, again))
    P = [p.detach() for p in gelib.SO3vec(*xs).CGproduct(gelib.SO3vec(*ys), maxl).parts.values()]
    P64 = [p.as_subclass(torch.Tensor).cpu().to(torch.complex128) for p in P]
    w64, g64 = [w.detach().cpu().to(torch.complex128) for w in ws], [g.cpu().to(torch.complex128) for g in gs]
    want = [torch.matmul(p, w) for p, w in zip(P64, w64)]
    gP = [torch.matmul(g, w.conj().T).to(torch.complex64).cuda() for g, w in zip(g64, w64)]
    xg, yg = [torch.empty_like(x) for x in xs], [torch.empty_like(y) for y in ys]
    cabi.so3vec_bwd(xg, yg, gP, [x.detach() for x in xs], [y.detach() for y in ys], accumulate=False)
    want += [t.cpu() for t in xg + yg]
    want += [torch.matmul(p.reshape(-1, p.shape[-1]).conj().T, g.reshape(-1, out)) for p, g in zip(P64, g64)]
    for k, (a, c) in enumerate(zip(got, want)):
        c = c.to(torch.complex128)
        d = (a.detach().cpu().to(torch.complex128) - c).norm() / c.norm()
        assert d < 2e-6, "output %d: relative error %.2g" % (k, d)   # sums of up to 3000 float32 terms, rounded randomly


@pytest.mark.parametrize("nout", [16, 5])
def test_matrix_gradient_from_strided_parts(cabi, nout):
    """Matrix gradients straight from operands whose cells and rows do not follow each other in memory: the bits of packed ones."""
    B, n1, n2 = 43, 8, 16
    xs, ys = [rand((B, 2 * l + 1, n1), l) for l in range(5)], [rand((B, 2 * l + 1, n2), 10 + l) for l in range(5)]
    tau = cabi.so3type_product({l: n1 for l in range(5)}, {l: n2 for l in range(5)}, 4)
    ws, gs = [rand((n, 16), 20 + l) for l, n in tau.items()], [rand((B, 2 * l + 1, 16), 40 + l) for l in tau]
    if nout != 16:   # even, as the call wants it, and less than the columns of a tile
        nout += 1
        ws, gs = [w[:, :nout].contiguous() for w in ws], [g[..., :nout].contiguous() for g in gs]
    def strided(t):
        w = torch.zeros(t.shape[0], t.shape[1], t.shape[2] + 3, dtype=t.dtype, device=t.device)
        w[..., :t.shape[2]] = t
        return w[..., :t.shape[2]]
    out = []
    for px in (xs, [strided(t) for t in xs]):
        wg = [torch.full_like(w, float("nan")) for w in ws]
        assert cabi.so3vec_cg_linear_bwd(None, None, wg, gs, px, ys, ws, accumulate=False)
        assert cabi.last_path() == 6
        out.append(wg)
    assert all(torch.equal(a, b) for a, b in zip(*out))


def layer(cabi, n1, n2, out, b, L=2):
    xs = [rand((b, 2 * l + 1, n1), l).requires_grad_() for l in range(L + 1)]
    ys = [rand((b, 2 * l + 1, n2), 10 + l).requires_grad_() for l in range(L + 1)]
    tau = cabi.so3type_product({l: n1 for l in range(L + 1)}, {l: n2 for l in range(L + 1)}, L)
    return xs, ys, [(rand((n, out), 20 + l) / np.sqrt(n)).requires_grad_() for l, n in tau.items()]


def near(got, want):
    for a, c in zip(got, want):
        a, c = a.detach().cpu().to(torch.complex128), c.detach().cpu().to(torch.complex128)
        assert (a - c).norm() <= 2e-6 * c.norm()   # sums of up to a few hundred float32 terms, as above


@pytest.mark.parametrize("n1,n2", [(3, 3), (4, 2)])
def test_conjugate_views(cabi, n1, n2):
    """Parts, matrices and gradients that torch conjugates on reading only: as their copies."""
    import gelib_amd as gelib
    xs, ys, ws = layer(cabi, n1, n2, 5, 20)

    def run(conj):
        out = gelib.CGproduct_linear(gelib.SO3vec(*xs), gelib.SO3vec(*ys), gelib.SO3weights(*[conj(w) for w in ws]), 2).parts.values()
        mixed = (gelib.SO3vec(*[conj(x) for x in xs]) * gelib.SO3weights(*[conj(w)[:n1].contiguous() for w in ws])).parts.values()
        rs = list(out) + list(mixed)
        gs = [conj(rand(tuple(r.shape), 60 + k)) for k, r in enumerate(rs)]
        return rs + list(torch.autograd.grad(rs, xs + ys + ws, gs))

    near(run(lambda t: t.conj()), run(lambda t: t.conj().resolve_conj()))


def test_graph_of_the_gradients(cabi):
    """A function of the matrices' gradients is differentiated back to the operands and to the gradient of the result; one
    vector is both operands."""
    import gelib_amd as gelib
    xs, _, _ = layer(cabi, 3, 3, 5, 20)
    _, _, ws = layer(cabi, 3, 3, 5, 1)
    gs = [rand((20, 2 * l + 1, 5), 40 + l).requires_grad_() for l in range(3)]
    vs = [rand(tuple(w.shape), 70 + l) for l, w in enumerate(ws)]

    def run(step):
        rs = step(gelib.SO3vec(*xs))
        first = torch.autograd.grad(rs, xs + ws, gs, create_graph=True)
        return list(first) + list(torch.autograd.grad(first[3:], xs + gs, vs))

    mixed = run(lambda x: list(gelib.CGproduct_linear(x, x, gelib.SO3weights(*ws), 2).parts.values()))
    plain = run(lambda x: [torch.matmul(p.as_subclass(torch.Tensor), w) for p, w in zip(x.CGproduct(x, 2).parts.values(), ws)])
    near(mixed, plain)


def test_dispatch_modes_see_the_products(cabi):
    """Counters of operations are shown torch's own products, with the same values."""
    import gelib_amd as gelib
    from torch.utils.flop_counter import FlopCounterMode
    x, w = rand((6, 3, 5), 1), rand((5, 3), 2)
    want = list((gelib.SO3vec(x) * gelib.SO3weights(w)).parts.values())
    with FlopCounterMode(display=False) as counter:
        got = list((gelib.SO3vec(x) * gelib.SO3weights(w)).parts.values())
    assert counter.get_total_flops() > 0
    near(got, want)


# ---- what torch's products part by part give as well ------------------------------------------------------------------


@pytest.mark.parametrize("n,b", [(3, 6), (3, 1100), (4, 6)])
def test_mixed_parts_without_a_gradient(cabi, n, b):
    """A loss of one part of x * W: the other parts and matrices get no gradient, whatever values they hold."""
    import gelib_amd as gelib
    xs, ws = [rand((b, 2 * l + 1, n), l) for l in range(3)], [rand((n, 5), 10 + l).requires_grad_() for l in range(3)]
    xs[2][1, 2, 0] = float("nan")
    xs = [x.requires_grad_() for x in xs]
    g = rand((b, 3, 5), 20)
    for graph in (False, True):
        rs = list((gelib.SO3vec(*xs) * gelib.SO3weights(*ws)).parts.values())
        got = torch.autograd.grad(rs[1], xs + ws, g, allow_unused=True, create_graph=graph)
        assert [t is None for t in got] == [True, False, True] * 2
        near([got[1], got[4]], torch.autograd.grad(torch.matmul(xs[1], ws[1]), [xs[1], ws[1]], g))


@pytest.mark.parametrize("n1,n2", [(3, 3), (4, 2)])
def test_layer_outputs_without_a_gradient(cabi, n1, n2):
    """The same for a layer: the matrices of unused results get none, and what they hold reaches no operand's gradient."""
    import gelib_amd as gelib
    xs, ys, ws = layer(cabi, n1, n2, 5, 20)
    with torch.no_grad():
        ws[2][0, 1] = float("nan")
    g = rand((20, 3, 5), 20)
    P = gelib.SO3vec(*xs).CGproduct(gelib.SO3vec(*ys), 2).parts[1].as_subclass(torch.Tensor)
    want = torch.autograd.grad(torch.matmul(P, ws[1]), xs + ys + [ws[1]], g)
    for graph in (False, True):
        out = gelib.CGproduct_linear(gelib.SO3vec(*xs), gelib.SO3vec(*ys), gelib.SO3weights(*ws), 2)
        got = torch.autograd.grad(out.parts[1], xs + ys + ws, g, allow_unused=True, create_graph=graph)
        assert [t is None for t in got] == [False] * 6 + [True, False, True]
        near(list(got[:6]) + [got[7]], want)


@pytest.mark.parametrize("n,b", [(3, 4), (3, 400), (4, 4)])
def test_classes_of_mixed_parts(cabi, n, b):
    """Odd counts: the class that torch.matmul gives; even ones: a tensor."""
    import gelib_amd as gelib
    make = [lambda t: t, torch.nn.Parameter, lambda t: t.as_subclass(gelib.SO3part), lambda t: t.as_subclass(gelib.SO3partArr)]
    for i, cx in enumerate(make):
        for cw in make[:3]:
            x, w = cx(rand((b, 3, n), 1)), cw(rand((n, 5), 2))
            try:
                want = torch.matmul(x, w)
            except TypeError:   # two classes that know nothing of each other
                if n % 2:
                    with pytest.raises(TypeError):
                        gelib.SO3vec(x) * gelib.SO3weights(w)
                continue
            got = (gelib.SO3vec(x) * gelib.SO3weights(w)).parts[1]
            assert type(got) is (type(want) if n % 2 else torch.Tensor)
            assert got.requires_grad == want.requires_grad and got.is_leaf == want.is_leaf
            near([got], [want])


@pytest.mark.parametrize("L,n,out", [(2, 3, 5), (2, 4, 6), (4, 2, 4), (5, 2, 3)])
def test_layer_of_arrays(cabi, L, n, out):
    """A layer of arrays of vectors is an array of vectors, with parts of the class that the two steps give."""
    import gelib_amd as gelib
    xs, ys = [rand((2, 3, 2 * l + 1, n), l) for l in range(L + 1)], [rand((2, 3, 2 * l + 1, n), 10 + l) for l in range(L + 1)]
    tau = {l: n for l in range(L + 1)}
    for maxl in (L, None):
        ws = [rand((c, out), 20 + l) for l, c in cabi.so3type_product(tau, tau, -1 if maxl is None else maxl).items()]
        x, y, W = gelib.SO3vecArr(*xs), gelib.SO3vecArr(*ys), gelib.SO3weights(*ws)
        two = x.CGproduct(y, maxl) * W
        got = gelib.CGproduct_linear(x, y, W, maxl)
        assert type(got) is gelib.SO3vecArr and got.get_adims() == [3]
        if len(ws) != 5:   # (the kernel of products with the parts l = 0..4 gives tensors)
            assert [type(p) for p in got.parts.values()] == [type(p) for p in two.parts.values()]
        near(got.parts.values(), two.parts.values())


def test_layer_of_an_array_and_a_vector(cabi):
    """Refused, as the product of the two is."""
    import gelib_amd as gelib
    xs, ys, ws = [rand((2, 1, 2 * l + 1, 3), l) for l in range(2)], [rand((2, 1, 2 * l + 1, 3), 9 + l) for l in range(2)], []
    tau = cabi.so3type_product({0: 3, 1: 3}, {0: 3, 1: 3}, 1)
    ws = [rand((c, 5), 20 + l) for l, c in tau.items()]
    with pytest.raises(AssertionError):
        gelib.CGproduct_linear(gelib.SO3vecArr(*xs), gelib.SO3vec(*ys), gelib.SO3weights(*ws), 1)


def test_frozen_matrices_keep_no_product(cabi):
    """Where the matrices learn nothing, the tensors that only their gradients would read are not kept."""
    import gelib_amd as gelib
    xs, ys, ws = layer(cabi, 3, 3, 5, 20)

    def kept(f):
        seen = []
        with torch.autograd.graph.saved_tensors_hooks(lambda t: seen.append(tuple(t.shape)) or t, lambda t: t):
            rs = f()
        return rs, seen
    frozen = [w.detach() for w in ws]
    rs, seen = kept(lambda: list(gelib.CGproduct_linear(gelib.SO3vec(*xs), gelib.SO3vec(*ys), gelib.SO3weights(*frozen), 2).parts.values()))
    assert not [s for s in seen if s in [(20, 2 * l + 1, w.shape[0]) for l, w in enumerate(ws)]]
    P = gelib.SO3vec(*xs).CGproduct(gelib.SO3vec(*ys), 2).parts.values()
    gs = [rand(tuple(r.shape), 30 + k) for k, r in enumerate(rs)]
    near(torch.autograd.grad(rs, xs + ys, gs), torch.autograd.grad([torch.matmul(p.as_subclass(torch.Tensor), w) for p, w in zip(P, frozen)], xs + ys, gs))
    xs, w = [rand((20, 2 * l + 1, 4), 50 + l).requires_grad_() for l in range(3)], [rand((4, 5), 40 + l) for l in range(3)]
    rs, seen = kept(lambda: list((gelib.SO3vec(*xs) * gelib.SO3weights(*w)).parts.values()))
    assert seen and all(s == (4, 5) for s in seen)
    near(torch.autograd.grad(rs, xs, gs), torch.autograd.grad([torch.matmul(x, v) for x, v in zip(xs, w)], xs, gs))
    fixed, learn = [x.detach() for x in xs], [v.requires_grad_() for v in w]
    rs, seen = kept(lambda: list((gelib.SO3vec(*fixed) * gelib.SO3weights(*learn)).parts.values()))
    assert (4, 5) not in seen
    near(torch.autograd.grad(rs, learn, gs), torch.autograd.grad([torch.matmul(x, v) for x, v in zip(fixed, learn)], learn, gs))


def test_parts_on_another_device(cabi, monkeypatch):
    """Parts that are not on the current device, whose stream the library's launches go to, stay with torch's product."""
    import gelib_amd as gelib
    xs, ws = [rand((4, 2 * l + 1, 4), 1 + l) for l in range(2)], [rand((4, 5), 3 + l) for l in range(2)]
    called = []
    monkeypatch.setattr(cabi, "vec_mix_channels", lambda *a: called.append(a))
    with monkeypatch.context() as m:
        m.setattr(torch.cuda, "current_device", lambda: 1)
        got = (gelib.SO3vec(*xs) * gelib.SO3weights(*ws)).parts.values()
    assert not called
    near(list(got), [torch.matmul(x, w) for x, w in zip(xs, ws)])


@pytest.mark.parametrize("counts,b,out,learn,together", [
    ((4,), 50, 5, True, 0), ((2048,), 5, 4, True, 1), ((4, 4), 50, 5, True, 2), ((3, 4, 4), 50, 5, True, 2), ((3, 4), 50, 5, True, 0),
    ((3,), 1024, 5, True, 0), ((3,), 1025, 5, True, 1), ((3, 4), 1025, 5, True, 2), ((3, 3, 3), 204, 5, True, 0), ((3, 3, 3), 205, 5, True, 3),
    ((3, 3, 3), 3000, 5, False, 0), ((501, 3), 4991, 5, False, 2), ((2049,), 4, 4, False, 1)])
def test_which_parts_are_mixed_in_one_call(cabi, monkeypatch, counts, b, out, learn, together):
    """Where the one call takes longer than the parts one after the other they stay apart; the values are the same either way."""
    import gelib_amd as gelib
    xs = [rand((b, 2 * l + 1, n), l).requires_grad_(learn) for l, n in enumerate(counts)]
    ws = [rand((n, out), 10 + l).requires_grad_(learn) for l, n in enumerate(counts)]
    inner, taken = cabi.vec_mix_channels, []
    monkeypatch.setattr(cabi, "vec_mix_channels", lambda rs, *a: (taken.append(len(rs)), inner(rs, *a)))
    got = list((gelib.SO3vec(*xs) * gelib.SO3weights(*ws)).parts.values())
    assert taken == ([together] if together else [])
    want = [torch.matmul(x, w) for x, w in zip(xs, ws)]
    near(got, want)
    if learn:
        gs = [rand(tuple(r.shape), 20 + k) for k, r in enumerate(got)]
        near(torch.autograd.grad(got, xs + ws, gs), torch.autograd.grad(want, xs + ws, gs))
