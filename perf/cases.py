"""Performance cases: what a program that uses this framework has it do.

Functions are sums of Gaussian charge densities, as in the tests and the
benchmark: centres, exponents and weights drawn at random.  A program builds
the projected density and the convolution operator once and keeps them; a pass
is one call on them (an operator application, a batch of applications, a
projection, a sum, a product, an inner product) and the result handed over as
arrays: the node index table, every node's coefficients and its norms.

A case names its sources (`sources`).  The seed of prepare() turns them, by a
mirror image and an exchange of axes, and scales them by a common factor: other
coefficients in other nodes, but as many of them, so that outputs of two seeds
have the same shape.

The ranges: Legendre orders 3, 5, 7 and 9 (all that the device path has),
1 to 32 Gaussians, precisions from 1e-2 to 1e-7, Poisson and Helmholtz kernels,
FP64 and FP32 sweeps, world boxes with and without a scaling factor.
"""
import os

import numpy as np
import torch

import mrcpp_amd as mr
from mrcpp_amd import workloads as W


def listed():
    apply = dict(kind="apply", sources=20240607, mu=0.0, spread=4.0, sweeps="fp64")
    return [
        # an inner product of two trees held on the GPU, <f|Pf>: the smallest call, made at every step of an iteration
        dict(name="dot_k7", kind="dot", sources=11, order=7, box=32, prec=1e-6, gaussians=4, mu=0.0, spread=4.0),
        # a coarse preview: lowest order, loosest precision, one source; eight breadth-first steps of a few nodes
        dict(apply, name="poisson_k3_1", order=3, box=16, prec=1e-3, gaussians=1, spread=0.5),
        # the low-order configuration of the tests and the benchmark (box with a scaling factor)
        dict(apply, name="poisson_k5_1", order=5, box=20, prec=1e-5, gaussians=1, spread=0.5),
        # the benchmark's headline: order 7, 1e-6, 16 sources
        dict(apply, name="poisson_k7_16", order=7, box=32, prec=1e-6, gaussians=16),
        # the same call with the FP32 sweeps that the benchmark chooses
        dict(apply, name="poisson_k7_16_fp32", order=7, box=32, prec=1e-6, gaussians=16, sweeps="fp32"),
        # the largest single application: tight precision, many sources, bound-state Helmholtz kernel
        dict(apply, name="helmholtz_k7_32", order=7, box=32, prec=1e-7, gaussians=32, mu=1.3, spread=6.0),
        # the high-order configuration of the benchmark
        dict(apply, name="helmholtz_k9_1", order=9, box=20, prec=1e-7, gaussians=1, mu=1.0, spread=0.5),
        # uneven trees in one batched call, Poisson and Helmholtz in turn (an orbital update), FP32 sweeps
        dict(apply, name="batch_k7_6_fp32", kind="batch", order=7, box=32, prec=1e-5, gaussians=8, trees=6, sweeps="fp32", mu=0.8, spread=6.0),
        # the density's grid and projection, redone whenever the sources move
        dict(name="project_k7_16", kind="project", sources=20240607, order=7, box=32, prec=1e-6, gaussians=16, spread=4.0),
        # density minus potential on the union of both grids
        dict(name="add_k7_16", kind="add", sources=20240607, order=7, box=32, prec=1e-6, gaussians=16, mu=0.0, spread=4.0),
        # density times potential (the integrand of an energy), low order and high
        dict(name="multiply_k5_8", kind="multiply", sources=12, order=5, box=20, prec=1e-5, gaussians=8, mu=0.0, spread=4.0),
        dict(name="multiply_k9_2", kind="multiply", sources=13, order=9, box=32, prec=1e-6, gaussians=2, mu=0.0, spread=2.0),
    ]


def draw(rng):
    kind = rng.choice(["apply"] * 6 + ["batch", "project", "add", "multiply", "dot"])
    order = rng.choice([3, 5, 7, 9])
    most = {3: 16, 5: 32, 7: 24, 9: 4}[order]
    loose, tight = {3: (1e-2, 1e-4), 5: (1e-3, 1e-6), 7: (1e-4, 1e-7), 9: (1e-5, 1e-7)}[order]

    def log_uniform(lo, hi):
        return lo * (hi / lo) ** rng.random()

    c = dict(kind=kind, sources=rng.randrange(1 << 30), order=order, box=rng.choice([16, 20, 32]), prec=float("%.3g" % log_uniform(tight, loose)),
             gaussians=int(log_uniform(1, most + 0.99)), spread=round(rng.uniform(0.5, 6.0), 3))
    if kind == "project":
        return c
    c["mu"] = 0.0 if rng.random() < 0.5 else round(rng.uniform(0.5, 3.0), 3)
    if kind in ("apply", "batch"):
        c["sweeps"] = rng.choice(["fp64", "fp64", "fp32"])
    if kind == "batch":
        c["trees"] = rng.randint(2, 8)
        c["gaussians"] = min(c["gaussians"], 2 if order == 9 else 8)
        c["prec"] = max(c["prec"], 1e-6)
    return c


# ---------------------------------------------------------------------------
# What a program holds before the call, and the call
# ---------------------------------------------------------------------------


def sources(case, seed, tree, n):
    src = W.random_sources(case["sources"] + 7919 * tree, n, case["spread"])
    rng = W.SplitMix64(1000003 * seed + tree)
    axes = [0, 1, 2]
    axes.sort(key=lambda _: rng.next_u64())
    sign = [1.0 - 2.0 * rng.randint(0, 1) for _ in axes]
    fac = rng.log_uniform(0.5, 2.0)
    centers = [tuple(sign[d] * c[axes[d]] for d in range(3)) for c in src.centers]
    return mr.GaussExp.from_sources(W.GaussianSources([fac * w for w in src.weights], src.exponents, centers))


def density(case, mra, gauss):
    f = mr.FunctionTree(mra)
    mr.build_grid(f, gauss)
    mr.project(case["prec"], f, gauss)
    return f


def operator(case, mra, mu):
    return mr.HelmholtzOperator(mra, mu, case["prec"]) if mu > 0.0 else mr.PoissonOperator(mra, case["prec"])


def prepare(case, seed):
    torch.cuda.init()
    kind, box = case["kind"], case["box"]
    mra = mr.MultiResolutionAnalysis((-box, box), case["order"])
    s = dict(case=case, mra=mra)
    if kind == "project":
        s["gauss"] = sources(case, seed, 0, case["gaussians"])
        return s
    if kind == "batch":
        # uneven trees: 1 to `gaussians` sources each, Poisson and Helmholtz in turn
        most, ops = case["gaussians"], [operator(case, mra, 0.0), operator(case, mra, case["mu"] or 1.0)]
        s["inputs"] = [(ops[t % 2], density(case, mra, sources(case, seed, t, 1 + (t * 5 + 2) % most))) for t in range(case["trees"])]
        return s
    s["f"] = density(case, mra, sources(case, seed, 0, case["gaussians"]))
    s["op"] = operator(case, mra, case["mu"])
    if kind != "apply":
        mr.set_sweep_precision("fp64")
        s["v"] = mr.FunctionTree(mra)
        mr.apply(case["prec"], s["v"], s["op"], s["f"])
    return s


def call(s):
    """The pass itself: the output trees, or the inner product."""
    case, mra = s["case"], s["mra"]
    kind, prec = case["kind"], case["prec"]
    if kind == "dot":
        return mr.dot(s["f"], s["v"])
    if kind == "project":
        return [density(case, mra, s["gauss"])]
    if kind == "batch":
        mr.set_sweep_precision(case["sweeps"])
        outs = [mr.FunctionTree(mra) for _ in s["inputs"]]
        mr.apply_batch([(prec, o, op, f) for o, (op, f) in zip(outs, s["inputs"])])
        return outs
    out = mr.FunctionTree(mra)
    if kind == "apply":
        mr.set_sweep_precision(case["sweeps"])
        s["stats"] = mr.apply(prec, out, s["op"], s["f"])
    elif kind == "add":
        mr.add(prec, out, 1.0, s["f"], -1.0, s["v"])
    else:
        mr.multiply(prec, out, 1.0, s["f"], s["v"])
    return [out]


def run(s):
    out = call(s)
    return out if isinstance(out, float) else [t.export() for t in out]


def work(case):
    """Bytes: the input nodes' coefficients once (an operator application: its
    matrices are far fewer), the output's coefficients and norms once.
    Operations: an application's applied tuples at what they take when every
    tuple shares its x and y sweeps with the most others, (2 + 4 + 8) / 8
    contractions of 2 (k+1)^4; a projection's value products and maps; one
    multiplication and addition per value of a sum or an inner product; the
    maps to and from values and the product of a multiplication."""
    s = prepare(case, 1)
    n1 = case["order"] + 1
    block = 8 * n1 ** 3
    out = call(s)
    kind = case["kind"]
    nout = 0 if kind == "dot" else sum(t.getNNodes() for t in out)
    ins = [f for _, f in s["inputs"]] if kind == "batch" else [s[k] for k in ("f", "v") if k in s]
    nin = sum(t.getNNodes() for t in ins)
    sweep = 2.0 * n1 * block  # one one-dimensional map of a whole node
    if kind == "apply":
        flops = s["stats"]["n_applied"] * 3.5 * n1 ** 4
    elif kind == "batch":
        stats = [mr.apply(case["prec"], mr.FunctionTree(s["mra"]), op, f) for op, f in s["inputs"]]
        flops = sum(st["n_applied"] for st in stats) * 3.5 * n1 ** 4
    elif kind == "project":
        flops = nout * (3.0 * block * case["gaussians"] + 9.0 * sweep)
    elif kind == "multiply":
        flops = nout * (2 * 9.0 * sweep + block + 9.0 * sweep)
    else:
        flops = 2.0 * block * (nout or min(nin, 2 * s["f"].getNNodes()) / 2)
    return {"bytes": 8.0 * (nin * block + nout * (block + 9)), "flops": flops}


def tolerance(case):
    # about four times what is seen: FP64 with the band's partial sums in
    # another order, up to 4.4e-15; FP32 sweeps against FP64 ones, up to 7.7e-8
    # (a single value 3.4e-6 of the root mean square); a projection on the
    # host's cores against the device's, 1.0e-15
    if case.get("sweeps") == "fp32":
        return {"rel": 3e-7, "max": 1.4e-5}
    return {"rel": 2e-14 if case["kind"] != "project" else 1e-14}


# ---------------------------------------------------------------------------
# The same results in plain numpy, 64 bits
# ---------------------------------------------------------------------------
# A node's coefficients as an array [2K, 2K, 2K] over (z, y, x): in each
# direction the scaling half then the wavelet half (or the two children's
# scaling coefficients).


def filters(order):
    """[[H0, H1], [G0, G1]]: two children's scaling coefficients to a parent's
    scaling and wavelet ones (tables of doubles, row by row; the second halves
    follow from the basis' parity)."""
    k = order + 1
    h, g = (np.fromfile(os.path.join(mr.FILTER_DIR, "L_%s0_%d" % (n, order))).reshape(k, k) for n in "HG")
    sign = (-1.0) ** (np.arange(k)[:, None] + np.arange(k)[None, :])
    return np.block([[h, sign * h], [g, (-1.0) ** k * sign * g]])


def legendre(order):
    """Quadrature points and weights on [0, 1] and phi[j, i] = phi_j(x_i)."""
    x, w = np.polynomial.legendre.leggauss(order + 1)
    phi = np.array([np.polynomial.legendre.Legendre.basis(j)(x) * np.sqrt(2.0 * j + 1.0) for j in range(order + 1)])
    return 0.5 * (x + 1.0), 0.5 * w, phi


def along(m, c):
    """The matrix m applied in all three directions of c[n, z, y, x]."""
    for _ in range(3):  # contract the last direction and bring it to the front
        c = np.moveaxis(c @ m.T, 3, 1)
    return c


def to_blocks(c):
    """[n, 2K, 2K, 2K] -> rows of eight blocks, x fastest, as trees are handed over."""
    n, k = c.shape[0], c.shape[1] // 2
    return c.reshape(n, 2, k, 2, k, 2, k).transpose(0, 1, 3, 5, 2, 4, 6).reshape(n, -1)


def from_blocks(c, k):
    n = c.shape[0]
    return c.reshape(n, 2, 2, 2, k, k, k).transpose(0, 1, 4, 2, 5, 3, 6).reshape(n, 2 * k, 2 * k, 2 * k)


class Plain:
    """The adaptive builder: nodes are (scale, x, y, z); `node(keys)` gives
    their coefficients [n, 2K, 2K, 2K]."""

    def __init__(self, case):
        self.k = case["order"] + 1
        self.w = filters(case["order"])
        self.x, self.wt, self.phi = legendre(case["order"])
        mra = mr.MultiResolutionAnalysis((-case["box"], case["box"]), case["order"])
        self.root, self.sf, self.max_scale = mra.root_scale, mra.scaling_factor, mra.max_scale
        r = range(-1, 1)
        self.roots = [(self.root, x, y, z) for z in r for y in r for x in r]
        self.split = {}  # node -> has children

    @staticmethod
    def children(key):
        n, x, y, z = key
        return [(n + 1, 2 * x + (c & 1), 2 * y + (c >> 1 & 1), 2 * z + (c >> 2)) for c in range(8)]

    def listing(self):
        out, stack = [], self.roots[::-1]
        while stack:
            u = stack.pop()
            out.append(u)
            if u in self.split:
                stack += self.children(u)[::-1]
        return out

    def refine(self, first, compute, wants):
        """Breadth-first from the nodes `first`: compute(level), then split
        where wants(key, i) of the level."""
        level = list(first)
        while level:
            compute(level)
            nxt = []
            for i, u in enumerate(level):
                if u not in self.split and u[0] + 2 <= self.max_scale and wants(u, i):
                    self.split[u] = True
                    nxt += self.children(u)
            level = nxt

    def grid_of(self, gauss):
        """A grid as fine as each Gaussian, where it is not zero."""
        for g in gauss.funcs:
            sd = (2.0 * g.alpha) ** -0.5
            visible = int(-np.floor(np.log2(self.k * 0.5 * sd)))

            def wants(u, _):
                lo = [self.sf * 2.0 ** -u[0] * l for l in u[1:]]
                hi = [self.sf * 2.0 ** -u[0] * (l + 1) for l in u[1:]]
                return u[0] < visible and not any(a > p + 5.0 * sd or b < p - 5.0 * sd for a, b, p in zip(lo, hi, g.pos))

            self.refine([u for u in self.listing() if u not in self.split], lambda level: None, wants)

    def build(self, prec, node):
        """Refined by the wavelet test from the grid's end nodes; then parents
        from their children, and the whole tree as arrays."""
        coef, self.total = {}, 0.0
        k = self.k
        first = [u for u in self.listing() if u not in self.split]
        state = {"scaling": None, "wavelet": 0.0}

        def compute(level):
            c = node(level)
            s0 = np.sum(c[:, :k, :k, :k] ** 2, axis=(1, 2, 3))
            self.wave = np.sum(to_blocks(c)[:, k ** 3:] ** 2, axis=1)
            if state["scaling"] is None:
                state["scaling"] = float(np.sum(s0))
            state["wavelet"] += float(np.sum(self.wave))
            self.total = state["scaling"] + state["wavelet"]
            coef.update(zip(level, c))

        def wants(u, i):
            return np.sqrt(self.wave[i]) > max(2.0 * np.finfo(float).eps, prec * np.sqrt(self.total or 1.0) * 2.0 ** (-0.5 * (u[0] + 1)))

        self.refine(first, compute, wants)
        nodes = self.listing()
        for n in sorted({u[0] for u in nodes}, reverse=True):
            at = [u for u in nodes if u[0] == n and u in self.split]
            if at:
                kids = np.array([[coef[v][:k, :k, :k] for v in self.children(u)] for u in at])
                for u, c in zip(at, along(self.w, from_blocks(kids, k))):
                    coef[u] = c
        c = to_blocks(np.array([coef[u] for u in nodes]))
        b = c.reshape(len(nodes), 8, -1)
        norms = np.sqrt(np.sum(b * b, axis=2))
        return None, c, np.concatenate([norms, np.sum(norms * norms, axis=1)[:, None]], axis=1)

    def points(self, level):
        """Quadrature points of the children, per direction: [n, 3, 2K]."""
        two = np.concatenate([self.x, self.x + 1.0])
        return np.array([[self.sf * 2.0 ** -(u[0] + 1) * (2.0 * l + two) for l in u[1:]] for u in level])

    def volume(self, level):
        return np.array([self.sf ** 1.5 * 2.0 ** (-1.5 * (u[0] + 1)) for u in level])[:, None, None, None]

    def from_values(self, level, v):
        half = np.kron(np.eye(2), self.phi * self.wt)
        return along(self.w, along(half, v) * self.volume(level))

    def to_values(self, level, c):
        half = np.kron(np.eye(2), self.phi.T)
        return along(half, along(self.w.T, c)) / self.volume(level)

    def operand(self, tree):
        """Nodes of an input tree; below its leaves, generated from them."""
        idx, c, _ = tree.export()
        known = dict(zip(map(tuple, idx[:, :4].tolist()), from_blocks(c, self.k)))

        def get(key):
            if key not in known:
                up = (key[0] - 1,) + tuple(l >> 1 for l in key[1:])
                kids = to_blocks(along(self.w.T, get(up)[None]))[0].reshape(8, self.k, self.k, self.k)
                for v, s in zip(self.children(up), kids):
                    full = np.zeros((2 * self.k,) * 3)
                    full[:self.k, :self.k, :self.k] = s
                    known.setdefault(v, full)
            return known[key]

        return lambda level: np.array([get(u) for u in level])


def exact(case, seed):
    kind = case["kind"]
    if kind in ("apply", "batch"):
        # millions of three-sweep tensor products behind a tuple-by-tuple
        # screening: many minutes in plain numpy
        return None
    s = prepare(case, seed)
    p = Plain(case)
    if kind == "dot":
        (ia, ca, _), (ib, cb, _) = s["f"].export(), s["v"].export()
        at = {tuple(u): i for i, u in enumerate(ib[:, :4].tolist())}
        total = np.longdouble(0.0)
        for i, u in enumerate(map(tuple, ia[:, :4].tolist())):
            if u in at:
                first = 0 if u[0] == p.root else p.k ** 3
                total += np.sum(ca[i, first:].astype(np.longdouble) * cb[at[u], first:])
        return float(total)
    if kind == "project":
        gauss = s["gauss"]
        p.grid_of(gauss)

        def node(level):
            r = p.points(level)
            v = np.zeros((len(level),) + (2 * p.k,) * 3)
            for g in gauss.funcs:
                e = np.exp(-g.alpha * (r - np.array(g.pos)[None, :, None]) ** 2)
                v += g.coef * e[:, 2, :, None, None] * e[:, 1, None, :, None] * e[:, 0, None, None, :]
            return p.from_values(level, v)

        return [p.build(case["prec"], node)]
    f, v = p.operand(s["f"]), p.operand(s["v"])
    if kind == "add":
        return [p.build(case["prec"], lambda level: f(level) - v(level))]
    return [p.build(case["prec"], lambda level: p.from_values(level, p.to_values(level, f(level)) * p.to_values(level, v(level))))]
