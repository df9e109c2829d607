"""The matrix-core kernels for one x part times one y part with channel counts that none of their shapes has exactly (or rows that
are not 16-byte aligned): products and gradients against the CPU oracle, and that what is not a number stays where it belongs."""
import numpy as np
import pytest

from tests import gpu_util as U

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

ONEPAIR = 5


@pytest.fixture(scope="module")
def cabi():
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    from gelib_amd import cabi as c
    c.lib()
    return c


CASES = [
    # (B, l1, n1, l2, n2, maxl): one short of a shape and one channel of it on each side, both halves and all waves of a cell
    (5, 8, 3, 9, 3, -1), (3, 10, 5, 8, 2, -1), (2, 9, 7, 9, 7, -1), (3, 10, 3, 8, 9, -1), (2, 7, 5, 10, 16, 12),
    (2, 10, 9, 10, 5, -1), (1, 9, 16, 9, 6, 10), (2, 8, 9, 8, 9, -1), (1, 10, 16, 10, 15, -1), (1, 10, 13, 11, 11, -1),
    (3000, 7, 3, 9, 3, 8),    # 16 places forward: the any-l kernel from 2049 cells on
]


@pytest.mark.parametrize("B,l1,n1,l2,n2,maxl", CASES)
def test_padded_shapes(cabi, B, l1, n1, l2, n2, maxl):
    xs, ys = [U.seeded(1 + B, B, 2 * l1 + 1, n1)], [U.seeded(2 + B, B, 2 * l2 + 1, n2)]
    O = U.VecOracle(xs, ys, maxl, False, gseed=100 + B)
    dx, dy, dg = [U.dev(a) for a in xs], [U.dev(a) for a in ys], [U.dev(a) for a in O.gs]
    dr = [torch.full(p.shape, 5.0, dtype=torch.complex64, device="cuda") for p in O.r32]
    cabi.so3vec_fwd(dr, dx, dy, accumulate=False)
    N = min(a * b for a, b in [(8, 8), (4, 4), (8, 16), (16, 16), (16, 8), (4, 16), (8, 2)] if n1 <= a and n2 <= b)
    assert (cabi.last_path() == ONEPAIR) == (2 * n1 * n2 > N and (N > 16 or B <= 2048))
    dxg, dyg = [torch.full_like(t, 3.0 - 2j) for t in dx], [torch.full_like(t, 3.0 - 2j) for t in dy]
    cabi.so3vec_bwd(dxg, dyg, dg, dx, dy, accumulate=False)
    assert cabi.last_path() == ONEPAIR
    torch.cuda.synchronize()
    O.check_fwd([U.host(t) for t in dr], "forward")
    O.check_bwd([U.host(dxg[0])], [U.host(dyg[0])], "backward")
    ax, ay = [t.clone() for t in dxg], [t.clone() for t in dyg]
    cabi.so3vec_bwd(ax, ay, dg, dx, dy, accumulate=True)
    torch.cuda.synchronize()
    O.check_bwd_onto([U.host(t) for t in ax], [U.host(t) for t in ay], [U.host(t) for t in dxg], [U.host(t) for t in dyg], "added")


@pytest.mark.parametrize("B,l1,n1,l2,n2,maxl,extra", [(3, 10, 7, 8, 7, -1, 0), (2, 9, 12, 9, 7, 9, 3), (3, 8, 3, 9, 3, -1, 1), (2, 7, 16, 8, 15, 10, 1),
                                                      (2, 9, 16, 8, 8, -1, 1)])
def test_products_added_onto_values(cabi, B, l1, n1, l2, n2, maxl, extra):
    """Adding stores at every width of a row's last piece, and in parts of more channels, which keep what they hold."""
    xs, ys = [U.seeded(1 + B, B, 2 * l1 + 1, n1)], [U.seeded(2 + B, B, 2 * l2 + 1, n2)]
    O = U.VecOracle(xs, ys, maxl, False, gseed=100 + B)
    start = [U.seeded(50 + k, B, p.shape[1], p.shape[2] + extra) for k, p in enumerate(O.r32)]
    r = [U.dev(s) for s in start]
    cabi.so3vec_fwd([t[..., :n1 * n2] for t in r], [U.dev(a) for a in xs], [U.dev(a) for a in ys], accumulate=True)
    assert cabi.last_path() == ONEPAIR
    torch.cuda.synchronize()
    got = [U.host(t) for t in r]
    assert all(np.array_equal(a[..., n1 * n2:], s[..., n1 * n2:]) for a, s in zip(got, start))
    O.check_fwd_onto([a[..., :n1 * n2] for a in got], [s[..., :n1 * n2] for s in start], "added")


@pytest.mark.parametrize("nx,ny", [((5, 7), (7, 5)), ((9, 3), (5, 6))])
def test_vectors_of_several_parts(cabi, nx, ny):
    """Pairs of parts one launch each: blocks at odd channels of parts with row lengths of their own, gradients added up."""
    B = 3
    xs, ys = [U.seeded(k, B, 2 * l + 1, n) for k, (l, n) in enumerate(zip((9, 10), nx))], [U.seeded(5 + k, B, 2 * l + 1, n) for k, (l, n) in enumerate(zip((8, 9), ny))]
    O = U.VecOracle(xs, ys, -1, False, gseed=7)
    assert len({p.shape[2] for p in O.r32}) > 2 and any(p.shape[2] % 2 for p in O.r32)
    dx, dy, dg = [U.dev(a) for a in xs], [U.dev(a) for a in ys], [U.dev(a) for a in O.gs]
    dr = [torch.full(p.shape, 5.0, dtype=torch.complex64, device="cuda") for p in O.r32]
    cabi.so3vec_fwd(dr, dx, dy, accumulate=False)
    dxg, dyg = [torch.full_like(t, 3.0 - 2j) for t in dx], [torch.full_like(t, 3.0 - 2j) for t in dy]
    cabi.so3vec_bwd(dxg, dyg, dg, dx, dy, accumulate=False)
    assert cabi.last_path() == ONEPAIR
    torch.cuda.synchronize()
    O.check_fwd([U.host(t) for t in dr], "forward")
    O.check_bwd([U.host(t) for t in dxg], [U.host(t) for t in dyg], "backward")
    start = [U.host(t) for t in dr]
    cabi.so3vec_fwd(dr, dx, dy, accumulate=True)
    torch.cuda.synchronize()
    O.check_fwd_onto([U.host(t) for t in dr], start, "added")


ROUTES = [
    # (B, l1, n1, l2, n2, maxl, extra channels of the result, taken here?): both sides of the lines that the product is taken along
    (2048, 7, 3, 2, 3, -1, 0, True), (2049, 7, 3, 2, 3, -1, 0, False),                                      # 16 places
    (100, 7, 7, 2, 8, -1, 0, True), (3500, 7, 7, 2, 8, -1, 0, False), (100, 7, 7, 7, 8, 7, 0, False),     # few values of l: small, large, capped
    (20, 4, 15, 8, 15, -1, 0, True), (200, 4, 4, 8, 15, -1, 0, False),                                    # 9 of them: 256 places, 64
    (9, 10, 5, 5, 8, -1, 0, True), (9, 10, 12, 5, 6, -1, 0, False), (9, 8, 12, 8, 6, -1, 0, True),        # more: idle places
    (100, 8, 8, 8, 8, -1, 1, False), (1024, 8, 8, 8, 8, -1, 1, True), (9, 8, 8, 8, 8, -1, 0, True),       # rows that are not aligned
    (9, 8, 16, 8, 8, -1, 1, True), (700, 8, 8, 8, 8, 3, 1, False),
]


@pytest.mark.parametrize("B,l1,n1,l2,n2,maxl,extra,here", ROUTES)
def test_which_products_are_padded(cabi, B, l1, n1, l2, n2, maxl, extra, here):
    """Where the any-l kernel is faster the product stays with it; the two agree to the rounding of sums of at most 31 terms."""
    x, y = U.dev(U.seeded(1, B, 2 * l1 + 1, n1)), U.dev(U.seeded(2, B, 2 * l2 + 1, n2))
    r = [[torch.zeros(B, 2 * l + 1, n + extra, dtype=torch.complex64, device="cuda")[..., :n]
          for l, n in cabi.so3type_product({l1: n1}, {l2: n2}, maxl).items()] for _ in range(2)]
    cabi.so3vec_fwd(r[0], [x], [y], accumulate=False)
    assert (cabi.last_path() == ONEPAIR) == here
    try:
        cabi.set_option("onepair_mfma_fwd", 0)
        cabi.so3vec_fwd(r[1], [x], [y], accumulate=False)
    finally:
        cabi.set_option("onepair_mfma_fwd", 1)
    assert cabi.last_path() != ONEPAIR
    # a term is at most |x| |y|, the squares of a row of coefficients add up to at most 1, and each order of the sum rounds by 31 * 2^-24
    assert all((a - b).norm() <= 2 * 31 * 2.0 ** -24 * 31 ** 0.5 * b.norm() for a, b in zip(*r))


def test_several_parts_stay_in_one_launch_unless_their_counts_are_built(cabi):
    """A vector whose first pair of parts would be padded goes to the any-l kernels as a whole."""
    for n, path in ((7, False), (8, True)):
        xs, ys = [U.dev(U.seeded(l, 5, 2 * l + 1, n)) for l in (8, 9)], [U.dev(U.seeded(l, 5, 2 * l + 1, n)) for l in (4, 5)]
        r = [torch.zeros(5, 2 * l + 1, c, dtype=torch.complex64, device="cuda") for l, c in cabi.so3type_product({8: n, 9: n}, {4: n, 5: n}, -1).items()]
        cabi.so3vec_fwd(r, xs, ys, accumulate=False)
        assert (cabi.last_path() == ONEPAIR) == path


def test_rows_that_are_not_aligned(cabi):
    """8 x 8 channels in parts of 65 channels (an odd row length): eight bytes at a time, the same bits as from aligned rows.  (Enough cells
    for the product of such parts to be taken here.)"""
    B, l = 1027, 9
    x, y = U.dev(U.seeded(1, B, 2 * l + 1, 8)), U.dev(U.seeded(2, B, 2 * l + 1, 8))
    tau = cabi.so3type_product({l: 8}, {l: 8}, -1)
    ref = [torch.empty(B, 2 * k + 1, n, dtype=torch.complex64, device="cuda") for k, n in tau.items()]
    wide = [torch.full((B, 2 * k + 1, n + 1), 7.0, dtype=torch.complex64, device="cuda") for k, n in tau.items()]
    cabi.so3vec_fwd(ref, [x], [y], accumulate=False)
    cabi.so3vec_fwd([w[..., :64] for w in wide], [x], [y], accumulate=False)
    assert cabi.last_path() == ONEPAIR
    assert all(torch.equal(w[..., :64], r) and bool((w[..., 64] == 7).all()) for w, r in zip(wide, ref))
    got = []
    for g in (ref, [w[..., :64] for w in wide]):
        xg, yg = [torch.empty_like(x)], [torch.empty_like(y)]
        cabi.so3vec_bwd(xg, yg, g, [x], [y], accumulate=False)
        assert cabi.last_path() == ONEPAIR
        got.append(xg + yg)
    assert all(torch.equal(a, b) for a, b in zip(*got))


def test_not_a_number_stays_with_its_channels(cabi):
    """One element of g that is not a number reaches the gradients of its own channels of x and y and no other."""
    B, l, n1, n2 = 2, 8, 5, 6
    x, y = U.dev(U.seeded(1, B, 2 * l + 1, n1)), U.dev(U.seeded(2, B, 2 * l + 1, n2))
    tau = cabi.so3type_product({l: n1}, {l: n2}, -1)
    for a, j in ((0, 0), (0, 5), (4, 0), (4, 5), (2, 3)):
        g = [U.dev(U.seeded(9 + k, B, 2 * k + 1, n)) for k, n in tau.items()]
        g[6][1, 3, a * n2 + j] = complex(float("nan"), 0.0)
        xg, yg = [torch.empty_like(x)], [torch.empty_like(y)]
        cabi.so3vec_bwd(xg, yg, g, [x], [y], accumulate=False)
        assert cabi.last_path() == ONEPAIR
        bad_x, bad_y = torch.isnan(torch.view_as_real(xg[0])).any(-1).any(1), torch.isnan(torch.view_as_real(yg[0])).any(-1).any(1)
        assert bad_x.nonzero().tolist() == [[1, a]] and bad_y.nonzero().tolist() == [[1, j]]
