"""Sums of slices along a grid dimension (gather) on the GPU, through the C-ABI and through the Python classes.

The reference has no numeric test of gather (python/tests/test_gather_map.py only prints two maps), and the loop it
calls lives in cnine, outside its tree.  What pins the result here is the definition itself: a gather is the product
with the 0/1 incidence matrix of the pairs, computed with torch on the host in float64; the numpy loop of the oracle
adds in the same order as the kernel and must match bit for bit."""
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


def random_pairs(n_in, n_out, k, seed):
    rng = np.random.default_rng(seed)
    return rng.integers(0, n_in, k).tolist(), rng.integers(0, n_out, k).tolist()


def cplx(*shape, seed=0):
    g = torch.Generator().manual_seed(seed)
    return torch.view_as_complex(torch.randn(*shape, 2, generator=g))


@pytest.mark.parametrize("shape,dim,n_out,k", [
    ((3, 7, 5, 4), 1, 6, 20),          # one grid dimension
    ((2, 5, 6, 3, 8), 1, 9, 30),       # first of two
    ((2, 5, 6, 3, 8), 2, 4, 11),       # second of two
    ((40, 3, 16), 0, 17, 100),         # along the batch
    ((1, 300, 7, 16), 1, 70000, 900),  # more targets than one launch takes rows, most of them empty
    ((2, 4, 1, 1), 1, 4, 0),           # no pairs at all
])
@pytest.mark.parametrize("accumulate", [True, False])
def test_cabi_gather_matches_oracle_bit_for_bit(G, shape, dim, n_out, k, accumulate):
    from gelib_amd import cabi
    x = cplx(*shape, seed=1)
    src, tgt = random_pairs(shape[dim], n_out, k, 2)
    rshape = list(shape)
    rshape[dim] = n_out
    r0 = cplx(*rshape, seed=3)
    gm = cabi.GatherMap(src, tgt, shape[dim], n_out)
    r = r0.cuda()
    cabi.part_gather(r, x.cuda(), gm, dim, accumulate=accumulate)
    want = ora.gather(x.numpy(), src, tgt, n_out, dim, r=r0.numpy().copy() if accumulate else None)
    assert np.array_equal(U.host(r), want)
    # the inverse map: sources and targets change places
    g = cplx(*rshape, seed=4)
    xg = torch.zeros(shape, dtype=torch.complex64, device="cuda")
    cabi.part_gather(xg, g.cuda(), gm, dim, inverse=True)
    assert np.array_equal(U.host(xg), ora.gather(g.numpy(), tgt, src, shape[dim], dim))


def test_cabi_gather_is_the_incidence_matrix_product(G):
    from gelib_amd import cabi
    n_in, n_out = 11, 7
    src, tgt = random_pairs(n_in, n_out, 40, 5)
    A = torch.zeros(n_out, n_in, dtype=torch.float64)
    for s, t in zip(src, tgt):
        A[t, s] += 1                      # a repeated pair counts twice
    x = cplx(3, n_in, 5, 4, seed=6)
    r = torch.zeros(3, n_out, 5, 4, dtype=torch.complex64, device="cuda")
    cabi.part_gather(r, x.cuda(), cabi.GatherMap(src, tgt, n_in, n_out), 1)
    want = torch.einsum("ts,bsmc->btmc", A.to(torch.complex128), x.to(torch.complex128))
    assert torch.allclose(r.cpu().to(torch.complex128), want, rtol=1e-5, atol=1e-5)


def test_cabi_gather_strided_and_errors(G):
    from gelib_amd import cabi
    src, tgt = [0, 2, 2, 1], [1, 1, 0, 3]
    gm = cabi.GatherMap(src, tgt, 3, 4)
    big = cplx(2, 3, 5, 12, seed=7).cuda()
    x = big[..., 2:10:2]                  # channel stride 2
    r = torch.zeros(2, 4, 5, 4, dtype=torch.complex64, device="cuda")
    cabi.part_gather(r, x, gm, 1)
    assert np.array_equal(U.host(r), ora.gather(U.host(x), src, tgt, 4, 1))
    with pytest.raises(cabi.GelibHipError) as e:      # wrong extent along the gathered dimension
        cabi.part_gather(torch.zeros(2, 5, 5, 4, dtype=torch.complex64, device="cuda"), x, gm, 1)
    assert e.value.status == 7
    with pytest.raises(cabi.GelibHipError) as e:      # other dimensions must agree
        cabi.part_gather(torch.zeros(2, 4, 5, 3, dtype=torch.complex64, device="cuda"), x, gm, 1)
    assert e.value.status == 5
    with pytest.raises(cabi.GelibHipError) as e:      # index outside the map's range
        cabi.GatherMap([0, 3], [0, 0], 3, 4)
    assert e.value.status == 12
    with pytest.raises(cabi.GelibHipError) as e:      # host memory
        cabi.part_gather(r.cpu(), x, gm, 1)
    assert e.value.status == 8


def test_python_gather_and_its_gradient(G):
    gmap = G.gather_map.random(5, 4, 0.4, seed=3)
    src, tgt = gmap.pairs()
    x = G.SO3partArr.randn(2, [5, 3], 2, 4, device="cuda")
    x.requires_grad_()
    y = x.gather(gmap, 0)
    assert isinstance(y, G.SO3partArr) and list(y.shape) == [2, 4, 3, 5, 4]
    assert np.array_equal(U.host(y), ora.gather(U.host(x), src, tgt, 4, 1))
    t = G.SO3partArr.randn_like(y)
    y.odot(t).backward()
    # the gradient is the gather of t along the same pairs read backwards
    assert np.array_equal(U.host(x.grad), ora.gather(U.host(t), tgt, src, 5, 1))
    # second grid dimension, on a vector; gather commutes with the product when each target has one source
    perm = G.gather_map.sources_targets([2, 0, 1], [0, 1, 2])
    tau = {0: 2, 1: 2, 2: 2}
    u = G.SO3vecArr.randn(2, [2, 3], tau, device="cuda")
    v = G.SO3vecArr.randn(2, [2, 3], tau, device="cuda")
    a = G.CGproduct(u, v, maxl=2).gather(perm, 1)
    b = G.CGproduct(u.gather(perm, 1), v.gather(perm, 1), maxl=2)
    for l in a.parts:
        assert torch.equal(a.parts[l], b.parts[l])
    R = G.SO3element.random()              # gather commutes with rotations
    w = u.gather(G.gather_map.random(3, 5, 0.5, seed=9), 1)
    wr = u.apply(R).gather(G.gather_map.random(3, 5, 0.5, seed=9), 1)
    for l in w.parts:
        assert torch.allclose(w.apply(R).parts[l], wr.parts[l], rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("shape,dim,n_out,k", [
    ((1, 70, 5, 8), 1, 33, 300),       # 16 bytes a thread
    ((1, 70, 5, 3), 1, 33, 300),       # an odd slice: 8 bytes a thread
    ((3, 50, 3, 1), 1, 41, 200),       # an outer dimension, short slices
    ((2, 3, 20, 1, 2), 2, 31, 90),     # two outer dimensions that nest
    ((33, 1, 64), 0, 257, 1100),       # along the batch, several blocks
])
def test_vec_gather_of_parts_with_other_layouts(G, shape, dim, n_out, k):
    """One call for three parts: as it is, 8 bytes past 16-byte alignment, and with strides that nest in no slice."""
    from gelib_amd import cabi
    src, tgt = random_pairs(shape[dim], n_out, k, 12)
    gm = cabi.GatherMap(src, tgt, shape[dim], n_out)
    rshape = list(shape)
    rshape[dim] = n_out
    x = cplx(*shape, seed=7)
    n = x.numel()
    odd = torch.empty(n + 1, dtype=torch.complex64, device="cuda")[1:].reshape(shape)
    odd.copy_(x)
    strided = torch.empty(list(shape[:-1]) + [2 * shape[-1]], dtype=torch.complex64, device="cuda")[..., ::2]
    strided.copy_(x)
    xs = [x.cuda(), odd, strided]
    rs = [torch.full(rshape, 5.0, dtype=torch.complex64, device="cuda") for _ in xs]
    cabi.vec_gather(rs, xs, gm, dim, accumulate=False)
    want = ora.gather(x.numpy(), src, tgt, n_out, dim)
    for r in rs:
        assert np.array_equal(U.host(r), want)
    many = [torch.full(rshape, 5.0, dtype=torch.complex64, device="cuda") for _ in range(11)]   # more parts than a launch takes
    cabi.vec_gather(many, [xs[0]] * 11, gm, dim, accumulate=True)
    for r in many:
        assert np.array_equal(U.host(r), ora.gather(x.numpy(), src, tgt, n_out, dim, r=np.full(rshape, 5.0, np.complex64)))


def test_vec_gather_gradients_of_some_parts(G):
    """Gradients arrive for the parts that are used, as when every part was gathered by itself."""
    x = [cplx(1, 9, 2 * l + 1, 4, seed=l).cuda().requires_grad_(l != 1) for l in range(3)]
    gm = G.gather_map.sources_targets([0, 3, 3, 8], [1, 1, 0, 2], 9, 5)
    for sel in (slice(0, 3), slice(0, 3, 2)):
        v = G.SO3vecArr(*x[sel]).gather(gm)
        assert [p.requires_grad for p in v.parts.values()] == [t.requires_grad for t in x[sel]]
        got = torch.autograd.grad(torch.view_as_real(v.parts[2].as_subclass(torch.Tensor)).sum(), [x[0], x[2]], allow_unused=True)
        assert got[0] is None
        want = torch.zeros(9)
        for s in (0, 3, 3, 8):
            want[s] += 1
        assert torch.equal(got[1].as_subclass(torch.Tensor).real.cpu(), want.reshape(1, 9, 1, 1).expand(1, 9, 5, 4))


def test_gather_function_of_one_part(G):
    """The autograd function of one part takes (x, map, dimension), as the reference's does, and returns the part."""
    from gelib_amd.SO3partArr import SO3partArr_GatherFn
    gmap = G.gather_map.random(6, 4, 0.5, seed=11)
    src, tgt = gmap.pairs()
    x = cplx(2, 3, 6, 5, 4, seed=21).cuda().requires_grad_()
    r = SO3partArr_GatherFn.apply(x, gmap, 1)
    assert isinstance(r, G.SO3partArr) and list(r.shape) == [2, 3, 4, 5, 4]
    assert np.array_equal(U.host(r), ora.gather(U.host(x), src, tgt, 4, 2))
    g = cplx(2, 3, 4, 5, 4, seed=22).cuda()
    (xg,) = torch.autograd.grad(r, x, g)
    assert np.array_equal(U.host(xg), ora.gather(U.host(g), tgt, src, 6, 2))
