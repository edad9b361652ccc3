"""Workloads of the P1 multigrid path, each called through the public Python classes as a user's program does.

A case is a dict of plain values:

    path       what one pass does (see `run`)
    nx ny nz   sub-cubes of the box [0, nx] x [0, ny] x [0, nz] / max(nx, ny, nz), six macro-tetrahedra each
    level      refinement level the pass works on
    bits       precision of the functions (64 or 32); the solves keep x and b in 64 bits and cycle in 32
    nrhs       right-hand sides, interleaved (1 or 32)
    nu         smoothing steps before and after the coarse correction; sweeps of a `smooth` pass
    omega      SOR relaxation
    symmetric  each smoothing step is a forward and a backward sweep
    wcycle     the coarse correction is visited twice
    graph      the cycle is replayed from a captured graph

The boxes are the unit cube of the benchmark (2 x 2 x 2 sub-cubes, 48 macro-tetrahedra), the cubes that the serving
loop takes (1 to 3 sub-cubes per side, levels 4 to 7) and boxes with unequal sides.  Functions are filled with seeded
Fourier modes: a few smooth ones, as right-hand sides are, and a few that the mesh only just resolves, as the errors
that a smoother works on are.
"""
import math

import numpy as np
import torch

import hyteg_amd as H

SOLVE_TOL = 1e-10       # relative residual of a single solve (the benchmark's)
BATCH_TOL = 1e-8        # of a 32-column solve and of the serving loop


def _case(path, n, level, **more):
    nx, ny, nz = (n, n, n) if isinstance(n, int) else n
    c = {"path": path, "nx": nx, "ny": ny, "nz": nz, "level": level, "bits": 64, "nrhs": 1, "nu": 1, "omega": 1.0,
         "symmetric": False, "wcycle": False, "graph": False}
    c.update(more)
    return c


def listed():
    return [
        # the operator on its own: one stencil apply of a small function (every launch counts), and of the largest
        _case("apply", 1, 3, name="apply-f64-6tets-L3"),
        _case("apply", 2, 8, name="apply-f64-48tets-L8"),
        # the residual of a convergence check in single precision, on the largest mesh of the serving loop
        _case("residual", 3, 6, bits=32, name="residual-f32-162tets-L6"),
        # a smoother called by a user's own loop: one sweep, and symmetric over-relaxation on a box
        _case("smooth", 2, 7, bits=32, name="sor-f32-48tets-L7"),
        _case("smooth", (1, 2, 3), 5, nu=2, omega=1.2, symmetric=True, name="ssor-f64-36tets-L5"),
        # grid transfer, as a multigrid written by the user calls it: fine to coarse and coarse to fine
        _case("restrict", 2, 7, name="restrict-f64-48tets-L7"),
        _case("prolongate", 2, 8, bits=32, name="prolongate-f32-48tets-L8"),
        # one multigrid cycle: the benchmark's FP64 V(3,3), and a small one where latency is all there is
        _case("cycle", 2, 7, nu=3, graph=True, name="v33-f64-48tets-L7"),
        _case("cycle", 1, 4, nu=2, name="v22-f64-6tets-L4-eager"),
        # a Poisson problem from its right-hand side's modes to 1e-10, as the benchmark's headline solves it
        _case("solve", 2, 8, nu=2, name="solve-48tets-L8"),
        # 32 right-hand sides at once, the batch lane of the serving loop
        _case("solve", 2, 5, nu=2, nrhs=32, name="solve-32rhs-48tets-L5"),
        # the whole call of a program that holds its data on the host: right-hand side in, solution out
        _case("host", 2, 6, nu=2, name="host-solve-48tets-L6"),
    ]


def _unknowns(c):
    n = 2 ** c["level"]
    return (c["nx"] * n - 1) * (c["ny"] * n - 1) * (c["nz"] * n - 1)


def draw(rng):
    path = rng.choice(["apply", "residual", "smooth", "restrict", "prolongate", "cycle", "cycle", "solve", "host"])
    # unknowns of the listed range of the path, spread over their logarithm
    low, high, deepest = {"solve": (1e3, 2e7, 7), "host": (1e3, 3e6, 7), "cycle": (1e3, 4e7, 8)}.get(path, (3e2, 1.4e8, 8))
    nrhs = rng.choice([1, 1, 1, 32]) if path in ("residual", "smooth", "cycle", "solve") else 1
    want = math.exp(rng.uniform(math.log(low), math.log(high))) / nrhs
    box = [rng.choice([1, 2, 2, 3]) for _ in range(3)]
    if rng.random() < 0.5:
        box = [box[0]] * 3
    level = round(math.log2((max(want, 27.0) / (box[0] * box[1] * box[2])) ** (1 / 3)))
    c = _case(path, tuple(box), min(max(level, 2), deepest), nrhs=nrhs)
    c["bits"] = rng.choice([64, 32]) if path not in ("solve", "host") else 64
    c["nu"] = rng.choice([1, 2, 2, 3])
    c["omega"] = rng.choice([1.0, 1.0, 1.15, 0.8])
    c["symmetric"] = path in ("smooth", "cycle") and nrhs == 1 and rng.random() < 0.25
    c["wcycle"] = path == "cycle" and rng.random() < 0.2
    c["graph"] = path == "cycle" and rng.random() < 0.6
    while _unknowns(c) * nrhs > high:
        c["level"] -= 1
    return c


# ---- inputs --------------------------------------------------------------------------------------------------


def _modes(c, rng, smooth, rough):
    """(nrhs, smooth + rough, 4) rows (amplitude, k, l, m): wave numbers 1..8, and from a fifth to two fifths of what
    the mesh resolves.  Half wave numbers leave values on the boundary."""
    m = max(c["nx"], c["ny"], c["nz"]) * 2 ** c["level"]
    out = np.zeros((c["nrhs"], smooth + rough, 4))
    out[..., 0] = rng.uniform(0.5, 1.0, out.shape[:2]) * rng.choice([-1.0, 1.0], out.shape[:2])
    out[:, :smooth, 1:] = rng.integers(1, 9, (c["nrhs"], smooth, 3))
    out[:, smooth:, 1:] = rng.integers(max(1, m // 5), max(2, 2 * m // 5) + 1, (c["nrhs"], rough, 3))
    return out


def _inputs(c, seed):
    """Modes of the functions that the pass reads, by name, from the seed alone."""
    rng = np.random.default_rng([int(seed), 20251202])
    if c["path"] in ("solve", "host"):
        return {"f": _modes(c, rng, 8, 0)}
    got = {"x": _modes(c, rng, 3, 3), "b": _modes(c, rng, 3, 3)}
    if c["path"] in ("apply", "residual"):
        got["x"][..., 1:] += 0.5
    return got


def _mesh(c):
    top = max(c["nx"], c["ny"], c["nz"])
    hi = (c["nx"] / top, c["ny"] / top, c["nz"] / top)
    return H.PrimitiveStorage(H.MeshInfo.meshCuboid((0, 0, 0), hi, c["nx"], c["ny"], c["nz"]))


def _multigrid(c, S):
    smoother = H.SymmetricSORSmoother(c["omega"]) if c["symmetric"] else H.SORSmoother(c["omega"])
    return H.GeometricMultigridSolver(S, smoother, H.CGSolver(S, 0, 0), H.P1toP1LinearRestriction(),
                                      H.P1toP1LinearProlongation(), 0, c["level"], c["nu"], c["nu"],
                                      cycleType=H.CycleType.WCYCLE if c["wcycle"] else H.CycleType.VCYCLE)


class Values(dict):
    """Outputs that stay on the device: name -> the values of a function on a level, or a plain value.  A function's
    values are copied to the host where they are looked at, as the user's program would copy them."""

    def __getitem__(self, name):
        v = super().__getitem__(name)
        if not isinstance(v, tuple):
            return v
        function, level = v
        host = function.download(level)
        return host if function.precision == H.F64 else host.astype(np.float32)

    def values(self):
        return [self[k] for k in self]

    def items(self):
        return [(k, self[k]) for k in self]


class State:
    pass


def prepare(case, seed):
    c, s = case, State()
    L, path = c["level"], c["path"]
    prec = H.F64 if c["bits"] == 64 else H.F32
    s.case, s.level, s.S, s.modes = c, L, _mesh(c), _inputs(c, seed)
    lowest = {"apply": L, "residual": L, "smooth": L, "restrict": L - 1, "prolongate": L - 1}.get(path, 0)

    def function(name, level=None):
        f = H.P1Function(name, s.S, lowest, L, precision=prec, nrhs=c["nrhs"])
        if name in s.modes:
            f.interpolate_modes(s.modes[name], L if level is None else level)
        return f

    if path in ("restrict", "prolongate"):
        s.x = function("x", L if path == "restrict" else L - 1)
        s.transfer = H.P1toP1LinearRestriction() if path == "restrict" else H.P1toP1LinearProlongation()
    else:
        s.A = H.P1ConstantLaplaceOperator(s.S, lowest, L)
        s.x, s.b = function("x"), function("b")
        if path in ("apply", "residual"):
            s.r = function("r")
    if path == "smooth":
        s.smoother = H.SymmetricSORSmoother(c["omega"]) if c["symmetric"] else H.SORSmoother(c["omega"])
    if path in ("cycle", "solve", "host"):
        s.gmg = _multigrid(c, s.S)
    if path in ("solve", "host"):
        s.M = H.P1ConstantMassOperator(s.S, lowest, L)
        tol = SOLVE_TOL if path == "solve" and c["nrhs"] == 1 else BATCH_TOL
        s.R = H.MixedPrecisionRefinementSolver(s.S, s.gmg, tolerance=tol, maxOuter=80,
                                               cyclesPerOuter=4 if path == "solve" else 2)
    if path == "host":      # the right-hand side as the program holds it
        s.x.interpolate_modes(s.modes["f"], L)
        s.M.apply(s.x, s.b, L, H.ALL)
        s.values = s.b.download(L)
    return s


def run(s):
    c, L = s.case, s.level
    path = c["path"]
    if path == "apply":
        s.A.apply(s.x, s.r, L, H.INNER)
        return Values(r=(s.r, L))
    if path == "residual":
        s.A.residual(s.x, s.b, s.r, L, H.INNER)
        return Values(r=(s.r, L))
    if path == "smooth":
        for _ in range(c["nu"]):
            s.smoother.solve(s.A, s.x, s.b, L)
        return Values(x=(s.x, L))
    if path == "restrict":
        s.transfer.restrict(s.x, L, H.INNER)
        return Values(coarse=(s.x, L - 1))
    if path == "prolongate":
        s.transfer.prolongate(s.x, L - 1, H.INNER)
        return Values(fine=(s.x, L))
    if path == "cycle":
        if c["graph"]:
            s.gmg.solve_graph(s.A, s.x, s.b, L)
        else:
            s.gmg.solve(s.A, s.x, s.b, L)
        return Values(x=(s.x, L))
    if path == "solve":     # as the serving loop: I_h f into x, b = M I_h f, then the solve from x = 0
        s.x.interpolate_modes(s.modes["f"], L)
        s.M.apply(s.x, s.b, L, H.ALL)
        s.x.interpolate(0.0, L)
        s.R.solve(s.A, s.x, s.b, L)
        return Values(x=(s.x, L), steps=s.R.outerSteps)
    s.b.upload(L, s.values)
    s.x.interpolate(0.0, L)
    s.R.solve(s.A, s.x, s.b, L)
    return {"x": s.x.download(L), "steps": s.R.outerSteps}


def work(case):
    """Bytes: per unknown and value of `size` bytes, an apply reads x and writes y (2), a residual and a sweep read two
    arrays and write one (3), restriction moves 1 + 1/8 and prolongation the same the other way, a cycle's levels add
    up to 8/7 of its finest.  A solve counts its cycles as the contraction of 0.1 to 0.3 a cycle needs them."""
    c = case
    n, size = _unknowns(c) * c["nrhs"], c["bits"] // 8
    sweeps = c["nu"] * (2 if c["symmetric"] else 1)
    per_apply = 29

    def cycle(size):
        visits = sum((2 if c["wcycle"] else 1) ** k / 8 ** k for k in range(c["level"]))
        return (visits * n * size * (2 * sweeps * 3 + 3 + 2 * 1.125),
                visits * n * (2 * sweeps + 1) * (per_apply + 3))

    path = c["path"]
    if path == "apply":
        return {"bytes": 2 * n * size, "flops": per_apply * n}
    if path == "residual":
        return {"bytes": 3 * n * size, "flops": (per_apply + 1) * n}
    if path == "smooth":
        return {"bytes": 3 * n * size * sweeps, "flops": (per_apply + 3) * n * sweeps}
    if path in ("restrict", "prolongate"):
        return {"bytes": 1.125 * n * size, "flops": 2 * n}
    if path == "cycle":
        b, f = cycle(size)
        return {"bytes": b, "flops": f}
    cycles = 32 if path == "solve" and c["nrhs"] == 1 else 26
    steps = cycles // (4 if path == "solve" else 2)
    b, f = cycle(4)
    b, f = cycles * b + (steps + 1) * 3 * n * 8 + steps * 20 * n, cycles * f + (steps + 1) * 30 * n
    return {"bytes": b + (3 + 1 if path == "solve" else 2) * n * 8, "flops": f}


# ---- the same in 64 bits, in plain torch ---------------------------------------------------------------------
# Every micro-vertex of a box lies on one lattice with 2^level points per sub-cube side, so a function is an array
# over the lattice; the micro-tetrahedra of a macro-tetrahedron give operators and transfers element by element.

_SPLIT = [(4, 5, 7, 3), (0, 3, 1, 4), (4, 1, 5, 3), (5, 6, 7, 2), (1, 3, 2, 5), (7, 2, 3, 5)]
_CORNER = [(0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1)]
# micro-tetrahedra at a point (x, y, z) of a macro-tetrahedron's index lattice, and how far from the slanted face
# (x + y + z = 2^level) that point has to be for them to exist
_MICRO = [(1, ((0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1))), (3, ((1, 1, 0), (0, 1, 1), (1, 0, 1), (1, 1, 1)))] + [
    (2, ((0, 1, 0), (1, 0, 1), p, q)) for p, q in (((1, 0, 0), (1, 1, 0)), ((1, 1, 0), (0, 1, 1)),
                                                   ((0, 1, 1), (0, 0, 1)), ((0, 0, 1), (1, 0, 0)))]


class _Lattice:
    def __init__(self, c, level, device):
        self.box, self.N, self.device = (c["nx"], c["ny"], c["nz"]), 2 ** level, device
        self.size = [n * self.N + 1 for n in self.box]
        self.h = 1.0 / (max(self.box) * self.N)
        ids = {}
        self.vertices = []
        for iz in range(self.box[2] + 1):
            for iy in range(self.box[1] + 1):
                for ix in range(self.box[0] + 1):
                    ids[ix, iy, iz] = len(self.vertices)
                    self.vertices.append((ix, iy, iz))
        cells = set()
        for iz in range(self.box[2]):
            for iy in range(self.box[1]):
                for ix in range(self.box[0]):
                    for tet in _SPLIT:
                        cells.add(tuple(ids[ix + _CORNER[k][0], iy + _CORNER[k][1], iz + _CORNER[k][2]] for k in tet))
        self.cells = sorted(cells)

    def flat(self, p):
        """Position of lattice point (or, linearly, of a step) p in the array, x fastest."""
        return p[0] + self.size[0] * (p[1] + self.size[1] * p[2])

    def frame(self, vertices):
        """Flat position of the first vertex and the flat steps towards the others."""
        v = [self.vertices[k] for k in vertices]
        step = [tuple(q[d] - v[0][d] for d in range(3)) for q in v[1:]]
        return self.flat([self.N * k for k in v[0]]), [self.flat(q) for q in step], step

    def simplex(self, dims, first, last):
        """Index points of `dims` coordinates, each at least `first`, their sum at most `last`, first one fastest."""
        r = torch.arange(first, last + 1, device=self.device)
        axes = torch.meshgrid(*[r] * dims, indexing="ij") if dims > 1 else (r,)
        keep = sum(axes) <= last
        return [a[keep] for a in reversed(axes)]

    def owned(self):
        """Flat positions in the order of a function's values: vertices, then the interiors of the edges, faces and
        cells, each class by sorted vertex numbers (cells: by their vertex tuple)."""
        edges, faces = set(), set()
        for t in self.cells:
            edges |= {tuple(sorted((t[a], t[b]))) for a in range(4) for b in range(a)}
            faces |= {tuple(sorted(t[:k] + t[k + 1:])) for k in range(4)}
        parts = [torch.tensor([self.flat([self.N * k for k in v]) for v in self.vertices], device=self.device)]
        for dims, prims in ((1, sorted(edges)), (2, sorted(faces)), (3, self.cells)):
            points = self.simplex(dims, 1, self.N - 1)
            for p in prims:
                o, steps, _ = self.frame(p)
                parts.append(o + sum(a * s for a, s in zip(points, steps)))
        return torch.cat(parts)

    def inner(self):
        m = torch.zeros(self.size[::-1], dtype=torch.bool, device=self.device)
        m[1:-1, 1:-1, 1:-1] = True
        return m.reshape(-1)

    def modes(self, modes):
        """Sum of the modes at every lattice point; one column per right-hand side."""
        axis = [torch.arange(n, device=self.device, dtype=torch.float64) * self.h for n in self.size]
        out = []
        for rhs in modes:
            u = torch.zeros(self.size[::-1], dtype=torch.float64, device=self.device)
            for a, k, l, m in rhs:
                sx, sy, sz = (torch.sin(w * math.pi * t) for w, t in zip((k, l, m), axis))
                u += a * sz[:, None, None] * sy[None, :, None] * sx[None, None, :]
            out.append(u.reshape(-1))
        return torch.stack(out, 1)

    def elements(self):
        """(flat positions of the first points, flat offsets of the four corners, corners in units of h) of the
        micro-tetrahedra, one kind of one macro-tetrahedron at a time."""
        points = {gap: self.simplex(3, 0, self.N - gap) for gap in {g for g, _ in _MICRO} if gap <= self.N}
        for cell in self.cells:
            o, steps, vec = self.frame(cell)
            for gap, corners in _MICRO:
                if gap > self.N:
                    continue
                at = o + sum(a * s for a, s in zip(points[gap], steps))
                offsets = [sum(q * s for q, s in zip(corner, steps)) for corner in corners]
                where = [[sum(q * v[d] for q, v in zip(corner, vec)) for d in range(3)] for corner in corners]
                yield at, offsets, where

    def laplace(self, u):
        y = torch.zeros_like(u)
        for at, off, where in self.elements():
            p = np.array(where, dtype=np.float64) * self.h
            J = (p[1:] - p[0]).T
            grad = np.linalg.inv(J)
            grad = np.vstack([-grad.sum(axis=0), grad])
            K = abs(np.linalg.det(J)) / 6 * grad @ grad.T
            v = [u[at + o] for o in off]
            for i in range(4):
                y.index_add_(0, at + off[i], sum(float(K[i, j]) * v[j] for j in range(4)))
        return y

    def parents(self, coarse):
        """For every point of this lattice the two points of the coarse one (twice its spacing) that it lies halfway
        between; both the same for a coarse point."""
        z, y, x = torch.meshgrid(*[torch.arange(n, device=self.device) for n in coarse.size[::-1]], indexing="ij")
        fine_of = self.flat((2 * x, 2 * y, 2 * z)).reshape(-1)
        both = torch.zeros(2, self.size[0] * self.size[1] * self.size[2], dtype=torch.int64, device=self.device)
        both[:, fine_of] = torch.arange(len(fine_of), device=self.device)
        for at, off, _ in coarse.elements():
            for i in range(4):
                for j in range(i):
                    middle = (fine_of[at + off[i]] + fine_of[at + off[j]]) // 2
                    both[0, middle], both[1, middle] = at + off[i], at + off[j]
        return both


def _stored(u, c):
    return u.float().double() if c["bits"] == 32 else u


def exact(case, seed):
    c = case
    path, L = c["path"], c["level"]
    if path not in ("apply", "residual", "restrict", "prolongate") or _unknowns(c) * c["nrhs"] > 1.5e8:
        return None     # sweeps, cycles and solves follow the framework's own order of updates
    device = "cuda" if torch.cuda.is_available() else "cpu"
    fine, inputs = _Lattice(c, L, device), _inputs(c, seed)
    if path in ("apply", "residual"):
        y = fine.laplace(_stored(fine.modes(inputs["x"]), c))
        if path == "residual":
            y = _stored(fine.modes(inputs["b"]), c) - y
        name, grid, y = "r", fine, torch.where(fine.inner()[:, None], y, 0.0)
    else:
        coarse = _Lattice(c, L - 1, device)
        a, b = fine.parents(coarse)
        if path == "restrict":
            u = _stored(fine.modes(inputs["x"]), c)
            y = torch.zeros(int(np.prod(coarse.size)), c["nrhs"], dtype=torch.float64, device=device)
            y.index_add_(0, a, 0.5 * u)
            y.index_add_(0, b, 0.5 * u)
            name, grid, y = "coarse", coarse, torch.where(coarse.inner()[:, None], y, 0.0)
        else:
            u = _stored(coarse.modes(inputs["x"]), c)
            name, grid, y = "fine", fine, torch.where(fine.inner()[:, None], 0.5 * (u[a] + u[b]), 0.0)
    y = y[grid.owned()].cpu().numpy()
    y = y[:, 0] if c["nrhs"] == 1 else y
    return {name: y if c["bits"] == 64 else y.astype(np.float32)}
