"""Products of vectors up to l = 5 and 6 in the unrolled forward kernels: what lies above l = 6, and odd channel counts, against the CPU
oracle; destinations inside wider ones, added to what is there."""
import pytest

from tests import gpu_util as U

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

UNROLLED = 2


@pytest.fixture(scope="module")
def cabi():
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    from gelib_amd import cabi as c
    c.lib()
    return c


CASES = [
    # (B, x {l: n}, y {l: n}, maxl): one launch or two, even and odd counts, one channel too many for two a thread, gaps in l, a few l above 6 only, capped
    # there, several tiles of cells
    (3, {6: 4, 5: 2}, {6: 4, 4: 6}, -1), (2, {l: 3 for l in range(7)}, {l: 3 for l in range(7)}, -1),
    (2, {l: 5 for l in range(6)}, {l: 3 for l in range(6)}, 5), (5, {0: 7, 2: 6, 5: 3, 6: 5}, {1: 3, 6: 4}, 8),
    (7, {5: 9, 6: 2}, {2: 3, 3: 5}, -1), (70, {3: 3, 5: 3}, {3: 3, 5: 4}, -1), (3, {6: 5}, {5: 6}, -1), (2, {5: 11, 2: 8}, {5: 12, 6: 1}, 7),
]


@pytest.mark.parametrize("B,tx,ty,maxl", CASES)
def test_forward(cabi, B, tx, ty, maxl):
    tx, ty = dict(sorted(tx.items())), dict(sorted(ty.items()))
    xs = [U.seeded(1 + l, B, 2 * l + 1, n) for l, n in tx.items()]
    ys = [U.seeded(30 + l, B, 2 * l + 1, n) for l, n in ty.items()]
    O = U.VecOracle(xs, ys, maxl, False, gseed=100 + B)
    wide = [torch.full((*p.shape[:-1], p.shape[-1] + 1), 5.0, dtype=torch.complex64, device="cuda") for p in O.r32]
    dr = [w[..., :-1] for w in wide]
    cabi.so3vec_fwd(dr, [U.dev(a) for a in xs], [U.dev(a) for a in ys], accumulate=False)
    few = any(n % 2 for n in tx.values()) and len(tx) * len(ty) <= 4 and len(O.r32) > 7   # these stay with the any-l kernels
    assert few or cabi.last_path() == UNROLLED
    torch.cuda.synchronize()
    O.check_fwd([U.host(t) for t in dr], "forward")
    assert all(bool((w[..., -1] == 5).all()) for w in wide)
    once = [t.clone() for t in dr]
    cabi.so3vec_fwd(dr, [U.dev(a) for a in xs], [U.dev(a) for a in ys], accumulate=True)
    # the same sum again on top of it: doubled, up to the contraction of the last product into the addition
    assert all(torch.allclose(a, 2 * b, rtol=0, atol=2e-6 * float(b.abs().max())) for a, b in zip(dr, once))


@pytest.mark.parametrize("l1,l2,l,n1,n2", [(5, 2, 4, 3, 5), (6, 6, 6, 7, 4), (6, 6, 0, 5, 5), (6, 6, 12, 8, 8), (3, 6, 8, 5, 3), (6, 2, 7, 1, 7)])
def test_one_triple(cabi, l1, l2, l, n1, n2):
    """The same part out of the whole product and by itself, at an offset in a wider one."""
    B = 9
    x, y = U.seeded(1, B, 2 * l1 + 1, n1), U.seeded(2, B, 2 * l2 + 1, n2)
    O = U.VecOracle([x], [y], -1, False, gseed=3)
    k = l - abs(l1 - l2)
    r = torch.full((B, 2 * l + 1, n1 * n2 + 3), 5.0, dtype=torch.complex64, device="cuda")
    cabi.so3part_cg_fwd(r, U.dev(x), U.dev(y), 2, False)
    assert cabi.last_path() == UNROLLED
    torch.cuda.synchronize()
    assert bool((r[..., :2] == 5).all()) and bool((r[..., -1] == 5).all())
    whole = [p if j != k else U.host(r[..., 2:-1].contiguous()) for j, p in enumerate(O.r32)]
    O.check_fwd(whole, "one triple")
