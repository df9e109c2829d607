"""The work that programs give this library, as cases that a benchmark can time and check.

A case goes through the Python classes of ``gelib_amd``, with autograd where it trains, the way an equivariant network
calls them: products of parts and of vectors, the Diag product, products with spherical harmonics on edges, a product
followed by its weight matrices, sums over neighbours, and the O(3) classes.  ``listed()`` names twelve of them,
``draw(rng)`` makes more of the same ranges, ``prepare`` / ``run`` set one up and run one pass, ``work`` counts what a
pass has to move and compute, ``tolerance`` says how far two correct single-precision implementations may lie apart.

Types are written ``"l:n l:n"`` (n channels of degree l); those of O(3) ``"l+:n l-:n"``.
"""
import math

import torch

import gelib_amd as gelib
from gelib_amd import cabi

DEVICE = "cuda"
MAX_BYTES = 1.2e10      # what a drawn case may move at most (the largest listed one moves 51e9)


# ---- types -----------------------------------------------------------------------------------------------------------

def _tau(text):
    return {int(l): int(n) for l, n in (item.split(":") for item in text.split())}


def _tau_text(tau):
    return " ".join("%d:%d" % item for item in tau.items())


def _o3_tau(text):
    out = {}
    for item in text.split():
        mu, n = item.split(":")
        out[(int(mu[:-1]), 1 if mu[-1] == "+" else -1)] = int(n)
    return gelib.O3type(out)


def _uniform(L, n, low=0):
    return _tau_text({l: n for l in range(low, L + 1)})


def _terms(l1, l2, l):
    """Pairs (m1, m2) with |m1 + m2| <= l: the terms of one channel of the block (l1, l2) -> l."""
    return sum(1 for m1 in range(-l1, l1 + 1) for m2 in range(-l2, l2 + 1) if abs(m1 + m2) <= l)


def _product(tx, ty, maxl, diag=False):
    """Type of a product and its terms per cell, over all channels."""
    out, terms = {}, 0
    for l1, n1 in tx.items():
        for l2, n2 in ty.items():
            n = n1 if diag else n1 * n2
            for l in range(abs(l1 - l2), l1 + l2 + 1):
                if maxl < 0 or l <= maxl:
                    out[l] = out.get(l, 0) + n
                    terms += n * _terms(l1, l2, l)
    return dict(sorted(out.items())), terms


def _cell(tau):
    """Complex numbers in one cell of a vector of this type."""
    return sum((2 * l + 1) * n for l, n in tau.items())


# ---- the cases -------------------------------------------------------------------------------------------------------

def listed():
    return [
        # One triple on a small batch, inference: the shape of the unit tests of programs that call parts one by one.
        # A few microseconds on the GPU; what counts is how soon the call is through.
        {"name": "part_1x1to1_n16_b1024_fwd", "op": "part", "l1": 1, "l2": 1, "l": 1, "n1": 16, "n2": 16, "batch": 1024,
         "train": False},
        # A training step on a few samples (one molecule, the end of an epoch): latency of forward and backward.
        {"name": "vec_L4_n16_b64", "op": "vec", "x": _uniform(4, 16), "y": _uniform(4, 16), "maxl": 4, "batch": 64,
         "train": True},
        # O(3) features with both parities, the size of a small batch of molecules.
        {"name": "o3_L2_n8_b1000", "op": "o3", "x": "0+:8 0-:8 1+:8 1-:8 2+:8 2-:8", "y": "0+:8 0-:8 1+:8 1-:8 2+:8 2-:8",
         "maxl": 2, "batch": 1000, "train": True},
        # Sums over the neighbours of a graph's nodes, eight edges a node, and the gradient.
        {"name": "gather_L2_n16_50k", "op": "gather", "x": _uniform(2, 16), "nodes": 50021, "degree": 8, "train": True},
        # Messages on the edges of a graph: node features times the spherical harmonics of the edge directions, which are
        # computed on the way and need no gradient.
        {"name": "edge_L3_n24_b60k", "op": "edge", "x": _uniform(3, 24), "ly": 2, "maxl": 3, "batch": 60013, "train": True},
        # Channel counts that fall with l, different on the two sides and no powers of two; every l of the product.
        {"name": "vec_ragged_b5k", "op": "vec", "x": "0:20 1:12 2:9 3:6 4:3", "y": "0:10 1:7 2:6 3:5", "maxl": -1,
         "batch": 5003, "train": True},
        # The product followed by the weight matrices that mix its channels: a layer of a network, training.
        {"name": "layer_L4_n16_b8192", "op": "layer", "x": _uniform(4, 16), "y": _uniform(4, 16), "maxl": 4, "out": 16,
         "batch": 8192, "train": True},
        # Vectors up to l = 6 and every l up to 12 (the default of CGproduct), an odd batch.
        {"name": "vec_L6_n8_b4099_uncapped", "op": "vec", "x": _uniform(6, 8), "y": _uniform(6, 8), "maxl": -1,
         "batch": 4099, "train": True},
        # One large degree on both sides into every l.
        {"name": "vec_10x10_n8_b16384", "op": "vec", "x": "10:8", "y": "10:8", "maxl": -1, "batch": 16384, "train": True},
        # One triple at throughput, with both gradients.
        {"name": "part_2x3to4_n32_b65536", "op": "part", "l1": 2, "l2": 3, "l": 4, "n1": 32, "n2": 32, "batch": 65536,
         "train": True},
        # The channel-wise product of wide vectors.
        {"name": "diag_L6_n64_b16384", "op": "diag", "x": _uniform(6, 64), "y": _uniform(6, 64), "maxl": 6,
         "batch": 16384, "train": True},
        # The full product at the batch size that the throughput figures are quoted on.
        {"name": "vec_L4_n16_b32768", "op": "vec", "x": _uniform(4, 16), "y": _uniform(4, 16), "maxl": 4, "batch": 32768,
         "train": True},
    ]


def _log_int(rng, low, high):
    """An integer from low to high, spread over its logarithm."""
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(max(low, high))))))))


def _some_tau(rng, L, most):
    """A type of degrees 0..L (now and then one missing) of at most `most` channels each: one count for all, or counts that fall with l."""
    n = _log_int(rng, 1, most)
    if rng.random() < 0.5:
        return {l: n for l in range(L + 1)}
    tau = {l: max(1, int(n * rng.uniform(0.6, 1.0) * (1 - l / (1.5 * (L + 1))))) for l in range(L + 1)}
    if L > 1 and rng.random() < 0.2:
        del tau[rng.randrange(L + 1)]
    return tau


def _sized(rng, case, key, low, high):
    """case with case[key] drawn from low to high, less where it would move more than MAX_BYTES."""
    one = work(dict(case, **{key: 1}))["bytes"]
    case[key] = _log_int(rng, low, max(low, min(high, int(MAX_BYTES / one))))
    return case


def draw(rng):
    op = rng.choice(["part", "vec", "vec", "diag", "high", "edge", "layer", "gather", "o3"])
    train = rng.random() < 0.75
    if op == "part":
        l1, l2 = rng.randint(0, 6), rng.randint(0, 6)
        case = {"op": "part", "l1": l1, "l2": l2, "l": rng.randint(abs(l1 - l2), l1 + l2), "n1": _log_int(rng, 1, 64),
                "n2": _log_int(rng, 1, 48), "train": train}
        return _sized(rng, case, "batch", 16, 131072)
    if op == "vec":
        L = rng.randint(1, 6)
        tx = _some_tau(rng, L, 32 if L < 4 else 16 if L < 5 else 8)
        ty = tx if rng.random() < 0.5 else _some_tau(rng, rng.randint(1, L), 24 if L < 4 else 16 if L < 5 else 8)
        case = {"op": "vec", "x": _tau_text(tx), "y": _tau_text(ty), "maxl": rng.choice([-1, L]), "train": train}
        return _sized(rng, case, "batch", 16, 32768)
    if op == "diag":
        L = rng.randint(1, 6)
        tau = _uniform(L, _log_int(rng, 1, 128))
        return _sized(rng, {"op": "diag", "x": tau, "y": tau, "maxl": rng.choice([-1, L]), "train": train}, "batch", 16, 131072)
    if op == "high":
        n = _log_int(rng, 2, 16)
        case = {"op": "vec", "x": "%d:%d" % (rng.randint(7, 10), n), "y": "%d:%d" % (rng.randint(7, 10), rng.choice([n, n, _log_int(rng, 2, 16)])),
                "maxl": rng.choice([-1, -1, 10]), "train": train}
        return _sized(rng, case, "batch", 64, 16384)
    if op == "edge":
        L = rng.randint(1, 4)
        case = {"op": "edge", "x": _tau_text(_some_tau(rng, L, 64)), "ly": rng.randint(1, 4), "maxl": L, "train": train}
        return _sized(rng, case, "batch", 64, 262144)
    if op == "layer":
        L = rng.randint(2, 4)
        n = _log_int(rng, 2, 16)
        case = {"op": "layer", "x": _uniform(L, n), "y": _uniform(L, rng.choice([n, max(1, n // 2)])), "maxl": L,
                "out": rng.choice([n, 2 * n, _log_int(rng, 4, 32)]), "train": train}
        return _sized(rng, case, "batch", 16, 8192)
    if op == "gather":
        case = {"op": "gather", "x": _tau_text(_some_tau(rng, rng.randint(0, 4), 64)), "degree": rng.randint(2, 12), "train": train}
        return _sized(rng, case, "nodes", 64, 65536)
    L = rng.randint(1, 3)
    n = _log_int(rng, 1, 16)
    tau = " ".join("%d%s:%d" % (l, p, n) for l in range(L + 1) for p in ("+-" if rng.random() < 0.8 else "+"))
    return _sized(rng, {"op": "o3", "x": tau, "y": tau, "maxl": rng.choice([-1, L]), "train": train}, "batch", 16, 16384)


# ---- one pass --------------------------------------------------------------------------------------------------------

class _Source:
    """Standard normal tensors on the GPU, made from a seed."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEVICE).manual_seed(seed)

    def real(self, *shape):
        return torch.randn(*shape, generator=self.g, device=DEVICE)

    def cplx(self, *shape):
        return torch.view_as_complex(self.real(*shape, 2))

    def parts(self, batch, tau):
        return [self.cplx(batch, 2 * l + 1, n) for l, n in tau.items()]

    def whole(self, n, top):
        return torch.randint(top, (n,), generator=self.g, device=DEVICE)


def _leaves(tensors, train):
    return [t.requires_grad_() for t in tensors] if train else tensors


def prepare(case, seed):
    """What a program has in hand before the pass: its tensors, the weights it keeps, the graph's map, and -- where it
    trains -- the gradient that comes back from what follows."""
    src, op, train = _Source(seed), case["op"], case["train"]
    s = {"op": op, "train": train, "maxl": case.get("maxl", -1)}
    if op == "part":
        l1, l2, l, b = case["l1"], case["l2"], case["l"], case["batch"]
        x, y = src.cplx(b, 2 * l1 + 1, case["n1"]), src.cplx(b, 2 * l2 + 1, case["n2"])
        s["leaves"] = _leaves([gelib.SO3part(x), gelib.SO3part(y)], train)
        s["x"], s["y"], s["l"] = s["leaves"] + [l]
        out = [(b, 2 * l + 1, case["n1"] * case["n2"])]
    elif op in ("vec", "diag", "layer"):
        b, tx, ty = case["batch"], _tau(case["x"]), _tau(case["y"])
        xs, ys = _leaves(src.parts(b, tx), train), _leaves(src.parts(b, ty), train)
        s["leaves"] = xs + ys
        s["x"], s["y"] = gelib.SO3vec(*xs), gelib.SO3vec(*ys)
        tr = cabi.so3type_product(tx, ty, case["maxl"], op == "diag")
        if op == "layer":
            ws = _leaves([src.cplx(n, case["out"]) / math.sqrt(n) for n in tr.values()], train)
            s["leaves"] = s["leaves"] + ws
            s["w"] = gelib.SO3weights(*ws)
            tr = {l: case["out"] for l in tr}
        out = [(b, 2 * l + 1, n) for l, n in tr.items()]
    elif op == "edge":
        b, tx = case["batch"], _tau(case["x"])
        s["leaves"] = _leaves(src.parts(b, tx), train)
        s["x"], s["ly"] = gelib.SO3vec(*s["leaves"]), case["ly"]
        s["direction"] = src.real(b, 3, 1)
        tr = cabi.so3type_product(tx, {l: 1 for l in range(case["ly"] + 1)}, case["maxl"])
        out = [(b, 2 * l + 1, n) for l, n in tr.items()]
    elif op == "gather":
        nodes, tx = case["nodes"], _tau(case["x"])
        s["leaves"] = _leaves([src.cplx(1, nodes, 2 * l + 1, n) for l, n in tx.items()], train)
        s["x"] = gelib.SO3vecArr(*s["leaves"])
        edges = torch.stack([src.whole(nodes * case["degree"], nodes), src.whole(nodes * case["degree"], nodes)], 1)
        s["map"] = gelib.gather_map.from_matrix(edges, nodes, nodes)
        out = [tuple(t.shape) for t in s["leaves"]]
    else:
        b, tx, ty = case["batch"], _o3_tau(case["x"]), _o3_tau(case["y"])
        xs = {mu: src.cplx(b, 2 * mu[0] + 1, n) for mu, n in tx.items()}
        ys = {mu: src.cplx(b, 2 * mu[0] + 1, n) for mu, n in ty.items()}
        s["leaves"] = _leaves(list(xs.values()) + list(ys.values()), train)
        s["x"], s["y"] = gelib.O3vec(xs), gelib.O3vec(ys)
        out = [(b, 2 * mu[0] + 1, n) for mu, n in tx.CGproduct(ty, case["maxl"]).items()]
    s["gradients"] = [src.cplx(*shape) for shape in out] if train else None
    return s


def run(s):
    """One pass: the result, and with training the gradients of everything that learns or lies upstream."""
    op = s["op"]
    if op == "part":
        out = [s["x"].CGproduct(s["y"], s["l"])]
    elif op == "vec":
        out = list(gelib.CGproduct(s["x"], s["y"], s["maxl"]).parts.values())
    elif op == "diag":
        out = list(gelib.DiagCGproduct(s["x"], s["y"], s["maxl"]).parts.values())
    elif op == "layer":
        out = list(gelib.CGproduct_linear(s["x"], s["y"], s["w"], s["maxl"]).parts.values())
    elif op == "edge":
        y = gelib.SO3vec(*[gelib.SO3part.spharm(l, s["direction"]) for l in range(s["ly"] + 1)])
        out = list(gelib.CGproduct(s["x"], y, s["maxl"]).parts.values())
    elif op == "gather":
        out = list(s["x"].gather(s["map"]).parts.values())
    else:
        out = list(gelib.CGproduct(s["x"], s["y"], s["maxl"]).parts.values())
    if not s["train"]:
        return out
    return out + list(torch.autograd.grad(out, s["leaves"], s["gradients"]))


# ---- what a pass cannot do without -----------------------------------------------------------------------------------

def work(case):
    """Bytes: operands read and results written once, forward; backward, the incoming gradients and the operands read once
    and the gradients written once.  Flops: eight a term of the product and direction (a complex multiply-add), two
    directions backward; eight a complex multiply-add of the matrices; a complex add a pair of the sums over neighbours."""
    op, train = case["op"], case["train"]
    if op == "gather":
        cell, nodes = _cell(_tau(case["x"])), case["nodes"]
        passes = 2 if train else 1
        return {"bytes": passes * nodes * (16 * cell + 8 * case["degree"]), "flops": passes * 2 * nodes * case["degree"] * cell}
    b = case["batch"]
    if op == "part":
        X, Y = (2 * case["l1"] + 1) * case["n1"], (2 * case["l2"] + 1) * case["n2"]
        R = (2 * case["l"] + 1) * case["n1"] * case["n2"]
        terms = _terms(case["l1"], case["l2"], case["l"]) * case["n1"] * case["n2"]
    elif op == "edge":
        tx, ty = _tau(case["x"]), {l: 1 for l in range(case["ly"] + 1)}
        tr, terms = _product(tx, ty, case["maxl"])
        X, R = _cell(tx), _cell(tr)
        forward, backward = 8 * (X + R) + 12, 8 * (2 * X + R) + 12      # the directions come in, no gradient goes there
        return {"bytes": b * (forward + (backward if train else 0)), "flops": b * terms * (16 if train else 8)}
    elif op == "o3":
        tx, ty = _o3_tau(case["x"]), _o3_tau(case["y"])
        X, Y = (sum((2 * mu[0] + 1) * n for mu, n in t.items()) for t in (tx, ty))
        R = sum((2 * mu[0] + 1) * n for mu, n in tx.CGproduct(ty, case["maxl"]).items())
        _, terms = _product({}, {}, -1)
        for (l1, _), n1 in tx.items():
            for (l2, _), n2 in ty.items():
                terms += _product({l1: n1}, {l2: n2}, case["maxl"])[1]
    else:
        tx, ty = _tau(case["x"]), _tau(case["y"])
        tr, terms = _product(tx, ty, case["maxl"], op == "diag")
        X, Y, R = _cell(tx), _cell(ty), _cell(tr)
        if op == "layer":
            n = case["out"]
            out, mixed = n * sum(2 * l + 1 for l in tr), n * R
            weights = n * sum(tr.values())
            # the product itself need not be stored: operands, matrices and results; backward, their gradients as well
            return {"bytes": 8 * (b * (X + Y + out) + weights + (b * (2 * X + 2 * Y + out) + 2 * weights if train else 0)),
                    "flops": 8 * b * ((terms + mixed) * (3 if train else 1) + (terms if train else 0))}
    return {"bytes": 8 * b * (X + Y + R + (2 * X + 2 * Y + R if train else 0)), "flops": 8 * b * terms * (3 if train else 1)}


def tolerance(case):
    """Four times what the passes differ by from the same pass in complex128: sums of a few dozen terms lie at 0.6e-7 to
    1.9e-7 (largest difference 2e-6), the long sums over m of l1 = l2 = 10 at 3.4e-7 (2.8e-6), the product mixed by
    matrices, sums of up to 4352 channels, at 1.7e-6 (1.3e-5)."""
    if case["op"] == "layer":
        return {"rel": 7e-6, "max": 5e-5}
    if case["op"] == "vec" and max(_tau(case["x"])) > 6:
        return {"rel": 1.4e-6, "max": 1.2e-5}
    return {"rel": 8e-7, "max": 8e-6}
