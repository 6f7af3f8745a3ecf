"""Workloads of the pattern-evaluator fit, for timing it through its public
entry points.

A case is a dict of plain values: a "kind" (one use of the framework), a
pattern set, sizes and options.

    leaves    search leaves scored host to host (Evaluator.eval_host)
    score     resident positions scored (Evaluator.__call__)
    extract   row-major pattern indices of positions (Patterns.extract), the
              input of the differentiable evaluator
    products  A x and A^T y of one matrix: a solver's two products
    minibatch forward and backward of the differentiable evaluator through
              autograd (pattern_eval)
    epoch     one epoch of the fused Huber/Adam fit (huber_fit_fused)
    weights   FitWeights: matrix, Jacobi diagonal and a few PCG iterations (in
              64 bits: ten iterations in 32 bits lose all but two digits)
    stages    the stage loop: one system per empty count, fitted in one batch
    fit       the mixed-precision LSQR fit to 1e-10

Positions are random legal play from the seed (their column frequencies are
far from uniform, which is what the gathers and scatters meet), pattern sets
and listed sizes those of bench.py and the reference's evaluators.  The index
matrices are inputs here: exact() takes them as they are and computes the rest
in torch, in 64 bits.
"""
import functools
import math

import torch

from cassandra_amd import capi, names
from cassandra_amd.evaluator import huber_fit_fused, pattern_eval
from cassandra_amd.fit import Context, Patterns, fit_weights

SETS = ("FIT4", "FIT8", "FIT12", "logistello", "edax", "cassandra")


# ------------------------------------------------------------ cases -------
def listed():
    return [
        # the leaves one search thread hands over at a time
        dict(name="leaves_64", kind="leaves", set="FIT4", rows=64, empties=20),
        # scoring a data set with the reference's own 12-pattern evaluator
        dict(name="score_1M", kind="score", set="cassandra", rows=1_000_003, empties=30),
        # the indices of a training set
        dict(name="extract_5M", kind="extract", set="FIT4", rows=5_000_000, empties=30),
        # the products of the reference's own fit: few rows, latency-bound
        dict(name="products_f32_50k", kind="products", set="FIT4", rows=50_001, empties=20, dtype="float32",
             free=False),
        # the products of the large fit
        dict(name="products_f32_5M", kind="products", set="FIT8", rows=5_000_000, empties=24, dtype="float32",
             free=False),
        # the FP64 products of the FP64 solvers and of every refinement
        dict(name="products_f64_1M", kind="products", set="edax", rows=1_234_567, empties=24, dtype="float64",
             free=False),
        # the products of a matrix too large to store
        dict(name="products_free_20M", kind="products", set="FIT12", rows=20_000_000, empties=30, dtype="float32",
             free=True),
        # one step of a user's own training loop
        dict(name="minibatch_65536", kind="minibatch", set="FIT4", rows=65_536, empties=30, dtype="float32"),
        # one epoch of the library's training loop
        dict(name="epoch_5M", kind="epoch", set="FIT4", rows=5_000_000, empties=30, batch=65_536),
        # FitWeights on one stage's positions
        dict(name="weights_100k", kind="weights", set="FIT4", rows=100_000, empties=20, iterations=10),
        # the stage loop over the mid-game
        dict(name="stages_16", kind="stages", set="FIT4", rows=120_000, systems=16, empties=20, iterations=10),
        # the whole fit, to its default tolerance
        dict(name="fit_5M", kind="fit", set="FIT8", rows=5_000_000, empties=24),
    ]


def _between(rng, lo, hi):
    """A whole number of [lo, hi], spread over the logarithm, mostly odd sizes."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(lo, min(hi, n))


def draw(rng):
    kind = rng.choice(("leaves", "score", "extract", "products", "products", "products", "products", "minibatch",
                       "epoch", "weights", "stages", "fit"))
    c = dict(kind=kind, set=rng.choice(SETS), empties=rng.randint(16, 40))
    if kind == "leaves":
        c.update(rows=_between(rng, 1, 8192))
    elif kind == "score":
        c.update(rows=_between(rng, 8192, 1_000_000))
    elif kind == "extract":
        c.update(rows=_between(rng, 50_000, 2_000_000))
    elif kind == "products":
        free = rng.random() < 0.25
        dtype = "float32" if free else rng.choice(("float32", "float32", "float64"))
        c.update(rows=_between(rng, 300_000 if free else 20_000, 8_000_000 if free else 4_000_000), dtype=dtype,
                 free=free)
    elif kind == "minibatch":
        c.update(rows=_between(rng, 4096, 262_144), dtype=rng.choice(("float32", "float32", "float64")))
    elif kind == "epoch":
        c.update(rows=_between(rng, 500_000, 4_000_000), batch=2 ** rng.randint(13, 17))
    elif kind == "weights":
        c.update(rows=_between(rng, 50_000, 1_000_000), iterations=10)
    elif kind == "stages":
        c.update(rows=_between(rng, 30_000, 120_000), systems=rng.randint(2, 16), iterations=10, empties=20)
    else:
        c.update(set=rng.choice(("FIT4", "FIT8")), rows=_between(rng, 2_000_000, 4_000_000), empties=24)
    return c


# ------------------------------------------------------------ inputs ------
@functools.lru_cache(maxsize=None)
def _context():
    return Context(0)


@functools.lru_cache(maxsize=None)
def _patterns(name):
    """A program creates its pattern groups once."""
    return Patterns(_context(), getattr(names, name))


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _positions(case, seed):
    """Random legal play: one empty count, or the systems' rows one after the
    other at rising empty counts (row_begin in the second place)."""
    ctx = _context()
    if case["kind"] == "stages":
        # the stages' row counts fall off over a factor of four
        sizes = [max(1000, int(case["rows"] * 4.0 ** (-s / case["systems"]))) for s in range(case["systems"])]
        parts = [ctx.random_play(seed * 1009 + s, n, case["empties"] + s) for s, n in enumerate(sizes)]
        begin = [0]
        for n in sizes:
            begin.append(begin[-1] + n)
        return torch.cat(parts), begin
    spread = 10 if case.get("free") else 0
    return ctx.random_play(seed, case["rows"], case["empties"] - spread, case["empties"] + spread), [0, case["rows"]]


def _weights(case, seed, dtype=torch.float32):
    n = _patterns(case["set"]).cols
    return 1.5 * torch.randn(n, generator=_generator(seed + 1), device="cuda", dtype=torch.float64).to(dtype)


def _scores(A, seed):
    """Disc differences: a linear evaluation with noise, even, within +-64."""
    return A.make_targets(seed + 2, seed + 3)[1]


def prepare(case, seed):
    kind, P = case["kind"], _patterns(case["set"])
    s = dict(case=case, P=P)
    pos, begin = _positions(case, seed)
    if kind == "leaves":
        s.update(E=P.evaluator(_weights(case, seed)), pos=pos.cpu().numpy().view("uint64"))
    elif kind == "score":
        s.update(E=P.evaluator(_weights(case, seed)), pos=pos)
    elif kind == "extract":
        s.update(pos=pos)
    elif kind == "products":
        dtype = getattr(torch, case["dtype"])
        g = _generator(seed + 4)
        s.update(A=P.matrix_free(pos) if case["free"] else P.matrix(pos), x=_weights(case, seed, dtype),
                 y=torch.randn(case["rows"], generator=g, device="cuda", dtype=dtype))
    elif kind == "minibatch":
        dtype = getattr(torch, case["dtype"])
        s.update(idx=P.extract(pos), w=_weights(case, seed, dtype).requires_grad_(),
                 g=torch.randn(case["rows"], generator=_generator(seed + 4), device="cuda", dtype=dtype))
    elif kind == "epoch":
        s.update(idx=P.extract(pos), target=_scores(P.matrix(pos), seed).float(), seed=seed)
    elif kind == "weights":
        s.update(pos=pos, scores=_scores(P.matrix(pos), seed))
    else:
        A = P.matrix_systems(pos, begin) if kind == "stages" else P.matrix(pos)
        s.update(A=A, b=_scores(A, seed))
    torch.cuda.synchronize()
    return s


# ------------------------------------------------------------ passes ------
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "leaves":
        return s["E"].eval_host(s["pos"])
    if kind == "score":
        return s["E"](s["pos"])
    if kind == "extract":
        return s["P"].extract(s["pos"])
    if kind == "products":
        return s["A"].spmv(s["x"]), s["A"].spmtv(s["y"])
    if kind == "minibatch":
        score = pattern_eval(s["w"], s["idx"], s["P"])
        (grad,) = torch.autograd.grad(score, s["w"], s["g"])
        return score.detach(), grad
    if kind == "epoch":
        model, losses = huber_fit_fused(s["P"], s["idx"], s["target"], epochs=1, batch=case["batch"], seed=s["seed"])
        return model.weight.detach(), losses
    # the weights as the evaluator and the model file take them: floats
    if kind == "weights":
        x, _ = fit_weights(s["P"], s["pos"], s["scores"], case["iterations"], capi.PREC_FP64)
    elif kind == "stages":
        x = s["A"].solve_systems(s["b"], solver=capi.SOLVER_PCG, precision=capi.PREC_FP64, tol=0.0,
                                 max_iterations=case["iterations"], check_every=case["iterations"])[0]
    else:
        x = s["A"].solve(s["b"])[0]
    return x.float()


# ------------------------------------------------------------ work --------
def work(case):
    """Inputs read once, outputs written once.  A stored matrix has 2 bytes an
    entry, an iterative solve reads it twice an iteration (120 iterations reach
    1e-10 in 64 bits) with its row vector, and a gather-sum adds k values."""
    P = _patterns(case["set"])
    kind, n, k, cols = case["kind"], case["rows"], P.k, P.cols
    if kind in ("leaves", "score"):
        return dict(bytes=20 * n + 4 * min(n * k, P.expanded_size()), flops=n * k)
    if kind == "extract":
        return dict(bytes=n * (16 + 4 * k), flops=0)
    if kind == "products":
        v = 8 if case["dtype"] == "float64" else 4
        return dict(bytes=2 * (n * ((16 if case["free"] else 2 * k) + v) + v * cols), flops=2 * n * k)
    if kind == "minibatch":
        v = 8 if case["dtype"] == "float64" else 4
        return dict(bytes=n * (4 * k + 2 * v) + 2 * v * cols, flops=2 * n * k)
    if kind == "epoch":
        steps = -(-n // case["batch"])
        return dict(bytes=n * (4 * k + 12) + steps * 24 * cols, flops=2 * n * k + steps * 12 * cols)
    if kind == "fit":
        return dict(bytes=120 * n * (4 * k + 12), flops=120 * 2 * n * k)
    systems = case.get("systems", 1)
    rows = _positions_count(case)
    its = case["iterations"]
    return dict(bytes=rows * (its * (4 * k + 8) + 2 * k + 24) + its * systems * cols * 40, flops=its * 2 * rows * k)


def _positions_count(case):
    if case["kind"] != "stages":
        return case["rows"]
    return sum(max(1000, int(case["rows"] * 4.0 ** (-s / case["systems"]))) for s in range(case["systems"]))


# ------------------------------------------------------------ 64 bits -----
class _Matrix:
    """A of a case in 64 bits: slot-major indices, products slot by slot."""

    def __init__(self, P, pos):
        self.idx, self.cols, self.rows = P.extract(pos, capi.LAYOUT_SLOT_MAJOR), P.cols, pos.shape[0]

    def times(self, x):
        y = torch.zeros(self.rows, dtype=torch.float64, device="cuda")
        for i in self.idx:
            y += x[i.long()]
        return y

    def transposed_times(self, y):
        return self._column_sums((i, y) for i in self.idx)

    def _column_sums(self, entries, copies=128):
        """z[i[r]] += y[r] for every (i, y), row r adding to one of many copies
        of z: most rows share their commonest columns, and additions to one
        address wait for each other."""
        z = torch.zeros(copies * self.cols, dtype=torch.float64, device="cuda")
        copy = torch.arange(self.rows, device="cuda") % copies * self.cols
        for i, y in entries:
            z.index_add_(0, copy + i, y)
        return z.view(copies, self.cols).sum(0)

    def squares(self):
        """Per column the sum of the squared multiplicities in a row: A^T (its
        row's own count of the column), entry by entry."""
        def count(i):
            n = torch.zeros(self.rows, dtype=torch.float64, device="cuda")
            for j in self.idx:
                n += i == j
            return n

        return self._column_sums((i, count(i)) for i in self.idx)


def _pcg(A, b, iterations):
    """Jacobi-preconditioned CG on A^T A x = A^T b from 0."""
    d = A.squares()
    M = torch.where(d > 0, 1.0 / d.clamp(min=1.0), torch.ones_like(d))
    r = A.transposed_times(b)
    x, z = torch.zeros_like(r), M * r
    p, rz = z.clone(), torch.dot(r, z)
    for _ in range(iterations):
        q = A.transposed_times(A.times(p))
        a = rz / torch.dot(p, q)
        x += a * p
        r -= a * q
        z = M * r
        new = torch.dot(r, z)
        p = z + (new / rz) * p
        rz = new
    return x


def _epoch(case, idx, target, cols, seed, lr=0.05, delta=4.0, b1=0.9, b2=0.999, eps=1e-8):
    """One shuffled epoch of Adam on the mean Huber loss."""
    n, B = case["rows"], case["batch"]
    order = torch.randperm(n, device="cuda", generator=_generator(seed))
    w, m, v = (torch.zeros(cols, dtype=torch.float64, device="cuda") for _ in range(3))
    total, steps = 0.0, 0
    for at in range(0, n, B):
        rows = order[at:at + B]
        i = idx[rows].long()
        d = w[i].sum(1) - target[rows]
        total += torch.where(d.abs() < delta, 0.5 * d * d, delta * (d.abs() - 0.5 * delta)).mean()
        g = torch.zeros_like(w)
        g.index_add_(0, i.reshape(-1), (d.clamp(-delta, delta) / len(rows)).repeat_interleave(i.shape[1]))
        steps += 1
        m = b1 * m + (1 - b1) * g
        v = b2 * v + (1 - b2) * g * g
        w -= lr / (1 - b1 ** steps) * m / (v.sqrt() / math.sqrt(1 - b2 ** steps) + eps)
    return w, [float(total) / steps]


def exact(case, seed):
    """run()'s outputs in 64 bits, in plain torch.  None for the indices (whole
    numbers) and for the whole fit, whose iterations would take too long."""
    kind, P = case["kind"], _patterns(case["set"])
    if kind in ("extract", "fit"):
        return None
    pos, begin = _positions(case, seed)
    if kind in ("leaves", "score"):
        y = _Matrix(P, pos).times(_weights(case, seed).double())
        return y.cpu().numpy() if kind == "leaves" else y
    if kind == "products":
        dtype = getattr(torch, case["dtype"])
        x = _weights(case, seed, dtype).double()
        y = torch.randn(case["rows"], generator=_generator(seed + 4), device="cuda", dtype=dtype).double()
        A = _Matrix(P, pos)
        return A.times(x), A.transposed_times(y)
    if kind == "minibatch":
        dtype = getattr(torch, case["dtype"])
        w = _weights(case, seed, dtype).double()
        g = torch.randn(case["rows"], generator=_generator(seed + 4), device="cuda", dtype=dtype).double()
        A = _Matrix(P, pos)
        return A.times(w), A.transposed_times(g)
    if kind == "epoch":
        target = _scores(P.matrix(pos), seed).float().double()
        return _epoch(case, P.extract(pos), target, P.cols, seed)
    if kind == "weights":
        return _pcg(_Matrix(P, pos), _scores(P.matrix(pos), seed), case["iterations"])
    b = _scores(P.matrix_systems(pos, begin), seed)
    return torch.cat([_pcg(_Matrix(P, pos[lo:hi].contiguous()), b[lo:hi], case["iterations"])
                      for lo, hi in zip(begin, begin[1:])])
