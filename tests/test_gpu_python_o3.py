"""The O(3) wrappers on the GPU: gelib_amd.O3part / O3vec.  The identities the reference's suite holds for SO(3)
(python/tests/ci_tests/test_SO3part.py, test_SO3vec.py), here under O(3) elements of both determinants, plus
agreement with the CPU oracle: an O(3) product is the SO(3) product of the same tensors, block by block, at the
running channel offset of each output part."""
import numpy as np
import pytest

from oracle import cg_oracle as ora
from tests import gpu_util as U

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def G():
    assert torch.cuda.is_available()
    import gelib_amd
    from gelib_amd import gelib_base  # noqa: F401  (fails loudly if the extension was not built)
    return gelib_amd


def elements(G):
    R = G.O3element.random()
    if R.parity() < 0:
        R = G.O3element(-R)
    return [R, G.O3element(-R), G.O3element(torch.diag(torch.tensor([1.0, 1.0, -1.0])))]   # rotation, improper, mirror


@pytest.mark.parametrize("p1,p2", [(1, 1), (1, -1), (-1, -1)])
@pytest.mark.parametrize("l1,l2,l", [(1, 1, 1), (2, 1, 2), (2, 3, 4)])
@pytest.mark.parametrize("diag", [False, True])
def test_part_equivariance(G, p1, p2, l1, l2, l, diag):
    name = "DiagCGproduct" if diag else "CGproduct"
    x = G.O3part.randn(2, (l1, p1), 4, device="cuda")
    y = G.O3part.randn(2, (l2, p2), 4, device="cuda")
    mu = (l, p1 * p2)
    z = getattr(x, name)(y, mu)
    assert isinstance(z, G.O3part) and z.mu == mu and list(z.shape) == [2, 2 * l + 1, 4 if diag else 16]
    want = ora.cg_fwd(U.host(x), U.host(y), l, diag=diag)
    assert U.gate_excess(U.host(z), want) <= 1.0
    for R in elements(G):
        zr = getattr(x.apply(R), name)(y.apply(R), mu)
        assert torch.allclose(z.apply(R), zr, rtol=1e-3, atol=1e-4)
    with pytest.raises(AssertionError):
        getattr(x, name)(y, (l, -p1 * p2))


def test_part_backprop(G):
    x = G.O3part.randn(3, (2, -1), 4, device="cuda")
    y = G.O3part.randn(3, (1, -1), 4, device="cuda")
    x.requires_grad_()
    y.requires_grad_()
    z = x.CGproduct(y, (2, 1))
    t = G.O3part.randn_like(z)
    loss = z.odot(t)
    loss.backward(torch.tensor(1.0, device="cuda"))
    xeps = G.O3part.randn_like(x)
    assert torch.allclose(G.O3part(x + xeps, x.mu).CGproduct(y, (2, 1)).odot(t) - loss, xeps.odot(x.grad), rtol=1e-3,
                          atol=1e-3)
    yeps = G.O3part.randn_like(y)
    assert torch.allclose(x.CGproduct(G.O3part(y + yeps, y.mu), (2, 1)).odot(t) - loss, yeps.odot(y.grad), rtol=1e-3,
                          atol=1e-3)


TAUS = [({(0, 1): 2, (1, -1): 2, (2, 1): 2}, {(0, 1): 2, (1, -1): 2, (2, 1): 2}),
        ({(0, 1): 3, (1, 1): 3, (1, -1): 3}, {(1, -1): 3, (2, -1): 3})]


def oracle_vec(x, y, diag, maxl):
    """Block by block with the part-level oracle, in the order of O3/O3index.hpp:28-31 and core/Gvec.hpp:311-321."""
    idx = lambda mu: 2 * mu[0] + (mu[1] == -1)
    xm, ym = sorted(x, key=idx), sorted(y, key=idx)
    sizes = {}
    for a in xm:
        for b in ym:
            for l in range(abs(a[0] - b[0]), a[0] + b[0] + 1):
                if maxl >= 0 and l > maxl:
                    continue
                mu = (l, a[1] * b[1])
                sizes[mu] = sizes.get(mu, 0) + (x[a].shape[2] if diag else x[a].shape[2] * y[b].shape[2])
    B = next(iter(x.values())).shape[0]
    out = {mu: np.zeros((B, 2 * mu[0] + 1, n), np.complex64) for mu, n in sizes.items()}
    offs = {mu: 0 for mu in sizes}
    for a in xm:
        for b in ym:
            for l in range(abs(a[0] - b[0]), a[0] + b[0] + 1):
                mu = (l, a[1] * b[1])
                if mu not in out:
                    continue
                ora.part_op(ora.DIAG_FWD if diag else ora.CG_FWD, out[mu], x[a], y[b], offs[mu])
                offs[mu] += x[a].shape[2] if diag else x[a].shape[2] * y[b].shape[2]
    return out


@pytest.mark.parametrize("case", [0, 1])
@pytest.mark.parametrize("diag", [False, True])
@pytest.mark.parametrize("maxl", [-1, 2])
def test_vec_product(G, case, diag, maxl):
    name = "DiagCGproduct" if diag else "CGproduct"
    taux, tauy = (G.O3type(t) for t in TAUS[case])
    x = G.O3vec.randn(3, taux, device="cuda")
    y = G.O3vec.randn(3, tauy, device="cuda")
    z = getattr(x, name)(y, maxl)
    assert dict(z.tau()) == dict(getattr(taux, name)(tauy, maxl))
    want = oracle_vec({mu: U.host(p) for mu, p in x.parts.items()}, {mu: U.host(p) for mu, p in y.parts.items()}, diag,
                      maxl)
    assert set(want) == set(z.parts)
    for mu in want:
        assert U.gate_excess(U.host(z.parts[mu]), want[mu]) <= 1.0, mu
    for R in elements(G):
        zr = getattr(x.apply(R), name)(y.apply(R), maxl)
        rz = z.apply(R)
        for mu in z.parts:
            assert torch.allclose(rz.parts[mu], zr.parts[mu], rtol=1e-3, atol=1e-4), mu


@pytest.mark.parametrize("diag", [False, True])
def test_vec_backprop(G, diag):
    fn = G.DiagCGproduct if diag else G.CGproduct
    taux, tauy = (G.O3type(t) for t in TAUS[1])
    x = G.O3vec.randn(2, taux, device="cuda")
    y = G.O3vec.randn(2, tauy, device="cuda")
    x.requires_grad_()
    y.requires_grad_()
    z = fn(x, y)
    t = G.O3vec.randn_like(z)
    loss = z.odot(t)
    loss.backward(torch.tensor(1.0, device="cuda"))
    xeps = G.O3vec.randn_like(x)
    assert torch.allclose(fn(x + xeps, y).odot(t) - loss, xeps.odot(x.get_grad()), rtol=1e-3, atol=1e-3)
    yeps = G.O3vec.randn_like(y)
    assert torch.allclose(fn(x, y + yeps).odot(t) - loss, yeps.odot(y.get_grad()), rtol=1e-3, atol=1e-3)


@pytest.mark.parametrize("diag", [False, True])
@pytest.mark.parametrize("xmus,ymus", [
    ([(0, 1), (1, -1), (2, 1)], [(1, -1), (1, 1)]),      # every pair of parities somewhere
    ([(1, 1), (2, 1)], [(0, -1), (1, -1), (2, -1)]),     # one parity on each side
    ([(1, -1)], [(0, 1), (1, 1), (1, -1)]),              # a destination first touched by a later product
    ([(7, 1), (2, -1)], [(1, -1), (7, -1)]),             # operands above what the small-l kernels take
])
@pytest.mark.parametrize("accumulate", [False, True])
def test_o3vec_entry_points_match_part_level_calls(G, xmus, ymus, diag, accumulate):
    """The vector calls against one part-level call per (mu1, mu2, mu) at the running channel offset.  Products are bit for
    bit single sums in both (compared to rounding: the families differ); a gradient adds up to a few hundred terms in
    another order, each order within 2^-24 times the terms' moduli per addition of a running sum: 1e-5 of the largest."""
    from gelib_amd import cabi
    from gelib_amd.O3 import _index
    n = 3
    B = 5
    xmus, ymus = sorted(xmus, key=_index), sorted(ymus, key=_index)
    mk = lambda mus, seed: [U.dev(U.seeded(seed + i, B, 2 * mu[0] + 1, n)) for i, mu in enumerate(mus)]
    x, y = mk(xmus, 1), mk(ymus, 30)
    tx, ty = G.O3type({mu: n for mu in xmus}), G.O3type({mu: n for mu in ymus})
    tau = tx.DiagCGproduct(ty, 8) if diag else tx.CGproduct(ty, 8)
    rmus = list(tau)
    start = [U.dev(U.seeded(60 + i, B, 2 * mu[0] + 1, tau[mu])) for i, mu in enumerate(rmus)]
    g = [U.dev(U.seeded(90 + i, B, 2 * mu[0] + 1, tau[mu])) for i, mu in enumerate(rmus)]
    base = (lambda ts: [t.clone() for t in ts]) if accumulate else (lambda ts: [torch.zeros_like(t) for t in ts])
    r0, xg0, yg0 = base(start), base(x), base(y)
    name = "so3part_diagcg_%s" if diag else "so3part_cg_%s"
    fwd, b0, b1 = (getattr(cabi, name % k) for k in ("fwd", "back0", "back1"))
    offs = {mu: 0 for mu in rmus}
    for i, mu1 in enumerate(xmus):
        for j, mu2 in enumerate(ymus):
            for l in range(abs(mu1[0] - mu2[0]), mu1[0] + mu2[0] + 1):
                mu = (l, mu1[1] * mu2[1])
                if mu not in offs:
                    continue
                k = rmus.index(mu)
                fwd(r0[k], x[i], y[j], offs[mu])
                b0(xg0[i], g[k], y[j], offs[mu])
                b1(yg0[j], g[k], x[i], offs[mu])
                offs[mu] += n if diag else n * n
    ps = lambda mus: [mu[1] for mu in mus]
    new = (lambda ts: [t.clone() for t in ts]) if accumulate else (lambda ts: [torch.full_like(t, 7.0) for t in ts])
    r, xg, yg = new(start), new(x), new(y)
    cabi.o3vec_fwd(r, ps(rmus), x, ps(xmus), y, ps(ymus), accumulate=accumulate, diag=diag)
    cabi.o3vec_bwd(xg, yg, g, ps(rmus), x, ps(xmus), y, ps(ymus), accumulate=accumulate, diag=diag)
    only = new(y)
    cabi.o3vec_bwd(None, only, g, ps(rmus), x, ps(xmus), y, ps(ymus), accumulate=accumulate, diag=diag)
    for a, b in list(zip(r, r0)) + list(zip(xg, xg0)) + list(zip(yg, yg0)) + list(zip(only, yg0)):
        assert float((a - b).abs().max()) <= 1e-5 * float(b.abs().max())
    # any order of the parts in the call
    r2 = new(start)
    cabi.o3vec_fwd(r2[::-1], ps(rmus)[::-1], x[::-1], ps(xmus)[::-1], y, ps(ymus), accumulate=accumulate, diag=diag)
    assert all(torch.equal(torch.view_as_real(a), torch.view_as_real(b)) for a, b in zip(r, r2))


@pytest.mark.parametrize("xtau,ytau", [
    ({(0, 1): 0}, {(0, 1): 0}),                                   # nothing at all
    ({(0, 1): 3, (1, 1): 0, (1, -1): 2}, {(0, 1): 0, (1, -1): 2}),
    ({(1, 1): 0, (2, -1): 4}, {(1, 1): 4, (1, -1): 0}),
])
@pytest.mark.parametrize("shared", [False, True])
def test_vec_product_with_parts_without_channels(G, xtau, ytau, shared):
    """A part without channels has no block in a product, its gradient is empty, and the others are as without it."""
    x = {mu: U.dev(U.seeded(3 + i, 3, 2 * mu[0] + 1, n)).requires_grad_() for i, (mu, n) in enumerate(xtau.items())}
    y = {mu: U.dev(U.seeded(30 + i, 1 if shared else 3, 2 * mu[0] + 1, n)).requires_grad_() for i, (mu, n) in enumerate(ytau.items())}
    z = G.CGproduct(G.O3vec(x), G.O3vec(y))
    full = lambda v: {mu: p for mu, p in v.items() if p.size(-1)}
    leaves = list(x.values()) + list(y.values())
    gs = {mu: U.dev(U.seeded(60 + i, *p.shape)) for i, (mu, p) in enumerate(z.parts.items())}
    grads = torch.autograd.grad(list(z.parts.values()), leaves, list(gs.values()))
    for t, g in zip(leaves, grads):
        assert g.shape == t.shape
    if not full(x) or not full(y):
        assert all(p.numel() == 0 or not p.any() for p in z.parts.values()) and not any(g.any() for g in grads)
        return
    w = G.CGproduct(G.O3vec(full(x)), G.O3vec(full(y)))
    for mu, p in z.parts.items():
        if p.size(-1):
            assert torch.equal(torch.view_as_real(p), torch.view_as_real(w.parts[mu]))
    some = list(full(x).values()) + list(full(y).values())
    want = torch.autograd.grad(list(w.parts.values()), some, [gs[mu] for mu in w.parts])
    for t, g in zip(some, want):
        assert torch.equal(torch.view_as_real(g), torch.view_as_real(grads[[t is u for u in leaves].index(True)]))
