"""Streaming loads and stores change no result: every kernel that has them gives the same bits with and without, at channel counts on
both sides of the lines where the dispatch changes over, and writes nothing beside its own channels."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def cabi():
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    from gelib_amd import cabi as c
    c.lib()
    return c


def rand(shape, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.view_as_complex(torch.randn(*shape, 2, device="cuda", generator=g))


CASES = [
    # (Lx, nx, Ly, ny, maxl, diag): Diag kernels (one and several cells a wave, without gaps, wave form, sets of l2, l above 6), a
    # one-channel operand, products of whole and of partial lines, the kernels for operands above l = 4, one triple
    (6, 64, 6, 64, 6, True), (6, 24, 6, 24, -1, True), (4, 17, 4, 17, 4, True), (2, 8, 2, 8, 2, True), (4, 72, 4, 72, 4, True),
    (3, 24, 2, 1, 3, False), (3, 32, 1, 1, 3, False), (1, 8, 2, 1, 1, False), (4, 16, 3, 1, 4, False),
    (4, 16, 4, 16, 4, False), (3, 4, 3, 4, 3, False), (3, 5, 2, 3, -1, False), (6, 8, 6, 8, -1, False), (6, 4, 6, 4, 6, False),
]


@pytest.mark.parametrize("Lx,nx,Ly,ny,maxl,diag", CASES)
def test_same_bits(cabi, Lx, nx, Ly, ny, maxl, diag):
    B = 37
    xs, ys = [rand((B, 2 * l + 1, nx), l) for l in range(Lx + 1)], [rand((B, 2 * l + 1, ny), 20 + l) for l in range(Ly + 1)]
    tau = cabi.so3type_product({l: nx for l in range(Lx + 1)}, {l: ny for l in range(Ly + 1)}, maxl, diag)
    gs = [rand((B, 2 * l + 1, n), 40 + l) for l, n in tau.items()]
    res = []
    names = ("fwd_stream", "diag6_stream", "bwd_once", "diag6_once")
    try:
        for value in (-1, 0, 1):
            for name in names:
                cabi.set_option(name, value)
            r = [torch.full((B, 2 * l + 1, n + 3), 7.0, dtype=torch.complex64, device="cuda") for l, n in tau.items()]
            cabi.so3vec_fwd([p[..., :-3] for p in r], xs, ys, accumulate=False, diag=diag)
            assert all(bool((p[..., -3:] == 7).all()) for p in r)
            once = [p[..., :-3].clone() for p in r]
            cabi.so3vec_fwd([p[..., :-3] for p in r], xs, ys, accumulate=True, diag=diag)
            xg, yg = [torch.empty_like(x) for x in xs], [torch.empty_like(y) for y in ys]
            cabi.so3vec_bwd(xg, yg, gs, xs, ys, accumulate=False, diag=diag)
            xg1 = [torch.empty_like(x) for x in xs]
            cabi.so3vec_bwd(xg1, None, gs, xs, ys, accumulate=False, diag=diag)
            res.append(once + r + xg + yg + xg1)
    finally:
        for name in names:
            cabi.set_option(name, -1)
    for other in res[1:]:
        assert all(torch.equal(a, b) for a, b in zip(res[0], other))


def parts(tau, B, extra, off):
    return [torch.zeros(B, 2 * l + 1, n + extra, dtype=torch.complex64, device="cuda")[..., off:off + n] for l, n in tau.items()]


SIDES = [
    # (x, y, maxl, diag, MB of product, channels more in its parts, of these in front, streaming stores?, streaming loads?)
    ({l: 64 for l in range(5)}, None, 4, True, 300, 0, 0, 1, 2), ({l: 64 for l in range(5)}, None, 4, True, 40, 0, 0, 0, 2),
    ({l: 64 for l in range(5)}, None, 4, True, 300, 8, 0, 1, 0), ({l: 64 for l in range(5)}, None, 4, True, 300, 16, 8, 1, 0),
    ({l: 64 for l in range(5)}, None, 4, True, 300, 4, 0, 0, 0), ({l: 64 for l in range(5)}, None, 4, True, 300, 16, 1, 0, 0),
    ({l: 64 for l in range(7)}, None, 6, True, 20, 1, 0, 0, 2),
    ({l: 16 for l in range(4)}, {l: 1 for l in range(3)}, 3, False, 300, 0, 0, 1, 2), ({l: 16 for l in range(4)}, {l: 1 for l in range(3)}, 3, False, 300, 1, 0, 0, 0),
    ({l: 8 for l in range(7)}, None, 6, False, 300, 8, 0, 1, 2), ({l: 8 for l in range(7)}, None, 6, False, 300, 1, 0, 0, 2),
    ({l: 8 for l in range(7)}, None, 6, False, 40, 0, 0, 0, 2),
    ({l: 4 for l in range(3)}, None, 2, False, 20, 0, 0, 0, 2), ({l: 4 for l in range(3)}, None, 2, False, 20, 8, 0, 0, 0),
    ({l: 16 for l in range(3)}, None, 2, False, 20, 1, 0, 0, 2),
    ({8: 8}, {3: 8}, -1, False, 300, 0, 0, 1, 2), ({8: 8}, {3: 8}, -1, False, 300, 8, 0, 1, 2), ({8: 8}, {3: 8}, -1, False, 40, 0, 0, 0, 2),
    ({8: 8}, {3: 8}, -1, False, 300, 2, 0, 0, 2), ({7: 4}, {2: 4}, -1, False, 300, 1, 0, 0, 0), ({7: 4}, {2: 4}, -1, False, 300, 0, 0, 1, 2),
]


@pytest.mark.parametrize("tx,ty,maxl,diag,mb,extra,off,stores,loads", SIDES)
def test_where(cabi, tx, ty, maxl, diag, mb, extra, off, stores, loads):
    """Streaming stores where rows start at half-lines and the product is larger than the memory-side cache, streaming loads where rows
    start at lines or are many; results as without."""
    ty = ty or tx
    tau = cabi.so3type_product(tx, ty, maxl, diag)
    B = int(mb * 1e6 / sum(8 * (2 * l + 1) * n for l, n in tau.items()))
    xs, ys = [rand((B, 2 * l + 1, n), l) for l, n in tx.items()], [rand((B, 2 * l + 1, n), 20 + l) for l, n in ty.items()]
    r = parts(tau, B, extra, off)
    cabi.so3vec_fwd(r, xs, ys, accumulate=False, diag=diag)
    assert cabi.last_streaming() == stores
    xg, yg = [torch.empty_like(x) for x in xs], [torch.empty_like(y) for y in ys]
    cabi.so3vec_bwd(xg, yg, r, xs, ys, accumulate=False, diag=diag)
    assert cabi.last_streaming() == loads
    names = ("fwd_stream", "diag6_stream", "onepair_mfma_stream", "bwd_once", "diag6_once", "onepair_mfma_once")
    try:
        for name in names:
            cabi.set_option(name, 0)
        r0, xg0, yg0 = parts(tau, B, extra, off), [torch.empty_like(x) for x in xs], [torch.empty_like(y) for y in ys]
        cabi.so3vec_fwd(r0, xs, ys, accumulate=False, diag=diag)
        assert cabi.last_streaming() == 0
        cabi.so3vec_bwd(xg0, yg0, r, xs, ys, accumulate=False, diag=diag)
        assert cabi.last_streaming() == 0
    finally:
        for name in names:
            cabi.set_option(name, -1)
    assert all(torch.equal(a, b) for a, b in zip(r + xg + yg, r0 + xg0 + yg0))
    cabi.so3vec_fwd(r, xs, ys, accumulate=True, diag=diag)
    assert cabi.last_streaming() == 0
