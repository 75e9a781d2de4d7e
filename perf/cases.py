"""The work that programs built on camille_amd have it do, as measurable cases.

Every case builds a solver (or a batch of them) once, and one pass is what
such a program repeats: put the initial state and clock in, advance, take the
fields (or the objective and its gradients) out.  Kinds:

  flow      one 2-D block, fused or plain path, uniform or sheared mean flow,
            sponges, optionally walls
  overset   background grid and cylinder O-grid, holes, receivers, slip wall
  ensemble  a batch of independent 2-D solves of uneven sizes
  flow3d    one 3-D block with a parallel shear flow
  grad2d    objective of observer pressures and its gradients through the
  grad3d    discrete adjoint (torch.autograd), 2-D and 3-D

`exact` advances the same inputs with a plain torch implementation of the
discretization in 64 bits.
"""
import math

import numpy as np
import torch

GAMMA = 1.4
LN2 = math.log(2.0)
CFL = 0.5


def listed():
    return [
        # the small curvilinear fixture problem: launches and latency are all there is
        dict(name="small_97x81_fp64", kind="flow", ni=97, nj=81, mean="uniform", walls=False, prec=64, path="fused",
             sponge=12, steps=60),
        # the reference's first test problem (201 x 201, 200 steps) as a user of the drop-in path runs it:
        # the reference's own arithmetic, bit for bit
        dict(name="plain_201x201", kind="flow", ni=201, nj=201, mean="uniform", walls=False, prec=64, path="plain",
             sponge=20, steps=40),
        # the headline problem: 1025 x 1025 curvilinear monopole, 32-bit bulk and 64 bits
        dict(name="monopole_1025_fp32", kind="flow", ni=1025, nj=1025, mean="uniform", walls=False, prec=32,
             path="fused", sponge=40, steps=1500),
        dict(name="monopole_1025_fp64", kind="flow", ni=1025, nj=1025, mean="uniform", walls=False, prec=64,
             path="fused", sponge=40, steps=1000),
        # a large block out of the last-level cache, odd sizes
        dict(name="monopole_2311x1507_fp32", kind="flow", ni=2311, nj=1507, mean="uniform", walls=False, prec=32,
             path="fused", sponge=24, steps=600),
        # a sheared base flow between slip walls, ragged sizes
        dict(name="channel_701x467_fp32", kind="flow", ni=701, nj=467, mean="shear", walls=True, prec=32,
             path="fused", sponge=20, steps=600),
        # the reference's arithmetic on a sheared base flow between walls, as validation runs use it
        dict(name="plain_channel_461x307", kind="flow", ni=461, nj=307, mean="shear", walls=True, prec=64,
             path="plain", sponge=16, steps=40),
        # scattering by a cylinder on overset grids
        dict(name="cylinder_1025x513_fp32", kind="overset", ni=1025, nj=513, prec=32, sponge=32, steps=300),
        # an ensemble of uneven solves
        dict(name="ensemble_16_fp32", kind="ensemble", solves=16, sizes=5, lo=129, hi_i=1025, hi_j=513, prec=32, sponge=20,
             steps=200),
        # 3-D jet, forward in 64 bits
        dict(name="jet_144x120x112_fp64", kind="flow3d", ni=144, nj=120, nk=112, prec=64, sponge=8, steps=60),
        # source optimisation steps: an objective and its gradients
        dict(name="gradient_385x257_fp64", kind="grad2d", ni=385, nj=257, prec=64, sponge=16, steps=60, every=20),
        dict(name="gradient_112x96x80_fp32", kind="grad3d", ni=112, nj=96, nk=80, prec=32, sponge=8, steps=24,
             every=8),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["flow", "flow", "flow", "plain", "overset", "ensemble", "flow3d", "grad2d", "grad3d"])
    prec = rng.choice([32, 64])
    if kind in ("flow", "plain"):
        plain = kind == "plain"
        ni = _log(rng, 65, 641 if plain else 2049)
        nj = min(_log(rng, 65, 641 if plain else 2049), max(65, int((3.0e5 if plain else 2.4e6) / ni)))
        steps = max(20, min(40, 4_000_000 // (ni * nj))) if plain else max(40, min(800, 800_000_000 // (ni * nj)))
        return dict(kind="flow", ni=ni, nj=nj, mean=rng.choice(["uniform", "shear"]), walls=rng.random() < 0.4,
                    prec=64 if plain else prec, path="plain" if plain else "fused",
                    sponge=rng.randint(8, max(8, min(40, min(ni, nj) // 5))), steps=steps)
    if kind == "overset":
        ni = rng.randint(513, 1025)
        return dict(kind="overset", ni=ni, nj=ni // 2 + rng.randint(0, 7), prec=prec, sponge=rng.randint(16, 32),
                    steps=rng.randint(120, 250))
    if kind == "ensemble":
        return dict(kind="ensemble", solves=rng.randint(4, 16), sizes=rng.randint(1, 10**6), lo=129, hi_i=rng.randint(300, 1025),
                    hi_j=rng.randint(200, 513), prec=prec, sponge=rng.randint(12, 20), steps=rng.randint(60, 200))
    if kind == "flow3d":
        return dict(kind="flow3d", ni=rng.randint(48, 144), nj=rng.randint(40, 120), nk=rng.randint(32, 112),
                    prec=prec, sponge=rng.randint(5, 8), steps=rng.randint(20, 60))
    if kind == "grad2d":
        return dict(kind="grad2d", ni=_log(rng, 97, 385), nj=_log(rng, 81, 257), prec=prec, sponge=rng.randint(8, 16),
                    steps=rng.randint(30, 60), every=rng.choice([10, 20]))
    return dict(kind="grad3d", ni=rng.randint(40, 112), nj=rng.randint(36, 96), nk=rng.randint(32, 80), prec=prec,
                sponge=rng.randint(5, 8), steps=rng.randint(8, 24), every=rng.choice([4, 8]))


# ------------------------------------------------------------------ inputs

_SIDES = {"+xi": (0, 0), "-xi": (0, 1), "+eta": (1, 0), "-eta": (1, 1), "+zeta": (2, 0), "-zeta": (2, 1)}


def _region(block, kind, side, width, dims):
    """A BC-file line of a face region `width` points deep (1: the face)."""
    d, end = _SIDES[side]
    spans = []
    for q in range(3):
        n = dims[q]
        if n == 1:
            spans += ["0", "0"]
        elif q != d:
            spans += ["0", "-0"]
        elif end == 0:
            spans += ["0", str(width - 1)]
        else:
            spans += ["-%d" % (width - 1), "-0"]
    return (block, kind, side) + tuple(spans)


def _pulse(x, y, x0, y0, w, amp):
    return amp * np.exp(-LN2 * ((x - x0) ** 2 + (y - y0) ** 2) / (w * w))


def _block2(case, rng, curved=True):
    """A 2-D block: grid, base flow, initial state, boundary regions, source."""
    ni, nj = case["ni"], case["nj"]
    d = 0.25
    lx, ly = d * (ni - 1), d * (nj - 1)
    xi, eta = np.meshgrid(-0.5 * lx + d * np.arange(ni), -0.5 * ly + d * np.arange(nj))
    L = max(lx, ly)
    walls = case.get("walls", False)
    mean = np.zeros((5, nj, ni))
    mean[4] = 1.0 / GAMMA
    if walls:  # a channel: eta lines follow the walls
        x, y = xi, eta + 0.02 * ly * np.sin(2.0 * np.pi * xi / lx)
    else:
        amp = 0.05 * L if curved else 0.0
        x, y = xi + amp * np.sin(2.0 * np.pi * eta / L), eta + amp * np.sin(2.0 * np.pi * xi / L)
    if case.get("mean") == "shear":
        mean[0] = 0.05 * np.exp(-((y / (0.3 * ly)) ** 2))
        mean[1] = 0.2 * (1.0 + np.tanh(y / (0.1 * ly)))
        mean[4] *= 1.0 + 0.03 * np.exp(-((x / (0.3 * lx)) ** 2 + (y / (0.3 * ly)) ** 2))
    else:
        mean[1] = rng.uniform(0.0, 0.6)
    x0, y0 = rng.uniform(-0.3, 0.3) * lx, rng.uniform(-0.25, 0.25) * ly
    ic = np.zeros((5, nj, ni))
    ic[4] = _pulse(x, y, x0, y0, 6 * d, 1e-3)
    ic[0] = _pulse(x, y, -x0, y0, 5 * d, 2e-4)
    xs, ys = rng.uniform(-0.3, 0.3) * lx, rng.uniform(-0.3, 0.3) * ly
    source = (1e-3, rng.uniform(0.1, 0.5) * math.pi, xs, ys, 0.0, 4 * d)
    dims = (ni, nj, 1)
    if walls:
        bc = [_region(0, "wall_slip_kinematic", s, 1, dims) for s in ("+eta", "-eta")]
        bc += [_region(0, "sponge_freund_ambient", s, case["sponge"], dims) for s in ("+xi", "-xi")]
    else:
        bc = [_region(0, "sponge_freund_ambient", s, case["sponge"], dims) for s in ("+xi", "-xi", "+eta", "-eta")]
    return dict(x=x, y=y, mean=mean, ic=ic, bc=bc, source=source)


def _block3(case, rng):
    """A 3-D Cartesian block with a parallel round shear flow along x."""
    dims = ni, nj, nk = case["ni"], case["nj"], case["nk"]
    d = 5.0 / 95
    z, y, x = np.meshgrid(d * (np.arange(nk) - 0.5 * (nk - 1)), d * (np.arange(nj) - 0.5 * (nj - 1)),
                          d * (np.arange(ni) - 0.5 * (ni - 1)), indexing="ij")
    r = np.sqrt(y * y + z * z)
    mean = np.zeros((5, nk, nj, ni))
    mean[1] = 0.45 * (1.0 - np.tanh((r - 0.5) / 0.15))
    mean[4] = 1.0 / GAMMA
    c = [rng.uniform(-0.2, 0.2) * d * (n - 1) for n in dims]
    r2 = (x - c[0]) ** 2 + (y - c[1]) ** 2 + (z - c[2]) ** 2
    ic = np.zeros((5, nk, nj, ni))
    ic[4] = 1e-3 * np.exp(-LN2 * r2 / (5 * d) ** 2)
    ic[2] = 2e-4 * np.exp(-LN2 * r2 / (6 * d) ** 2)
    bc = [_region(0, "sponge_freund_ambient", s, case["sponge"], dims) for s in ("+xi", "-xi")]
    source = (1e-3, rng.uniform(0.5, 1.0) * math.pi, -c[0], -c[1], -c[2], 4 * d)
    return dict(x=x, y=y, z=z, mean=mean, ic=ic, bc=bc, source=source)


def _sizes(case):
    """The grid sizes of an ensemble."""
    rng = np.random.default_rng(case["sizes"])
    return [(int(rng.integers(case["lo"], case["hi_i"] + 1)), int(rng.integers(case["lo"], case["hi_j"] + 1)))
            for _ in range(case["solves"])]


def _inputs(case, seed):
    """Blocks, regions, sources and tables of a case, as host arrays."""
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind == "flow":
        b = _block2(case, rng)
        return dict(blocks=[b], bc=b["bc"], sim="CASE_MONOPOLE", source=b["source"])
    if kind == "flow3d":
        b = _block3(case, rng)
        return dict(blocks=[b], bc=b["bc"], sim="CASE_MONOPOLE", source=b["source"])
    if kind in ("grad2d", "grad3d"):
        b = _block2(dict(case, mean="shear"), rng) if kind == "grad2d" else _block3(case, rng)
        shape = b["x"].shape
        q = rng.uniform(0.5, 1.5) * np.exp(-LN2 * ((b["x"] - b["source"][2]) ** 2 + (b["y"] - b["source"][3]) ** 2)
                                           / (0.2 * np.ptp(b["y"])) ** 2)
        n = int(np.prod(shape))
        obs = np.sort(rng.choice(n, min(n, 400), replace=False))
        return dict(blocks=[b], bc=b["bc"], sim="SOURCE_FIELD", source=(1e-3, b["source"][1]), q=q, obs=obs)
    if kind == "ensemble":
        blocks = [_block2(dict(ni=ni, nj=nj, sponge=case["sponge"]), rng, curved=False) for ni, nj in _sizes(case)]
        return dict(blocks=blocks, sim="CASE_MONOPOLE")
    from camille_amd import overset_gen as og
    ni, nj = case["ni"], case["nj"]
    geo = og.cylinder(nbg=(ni, nj), extent=(-8.0, 8.0, -4.0, 4.0), nog=(257, 65))
    xp, yp, amp = rng.uniform(-4.0, -2.5), rng.uniform(-1.0, 1.0), rng.uniform(0.5e-3, 1.5e-3)
    blocks = []
    for x, y in geo["blocks"]:
        ic = np.zeros((5,) + x.shape)
        ic[4] = _pulse(x, y, xp, yp, 0.3, amp)
        blocks.append(dict(x=x, y=y, mean=og.potential_flow(x, y, 0.3, 0.5), ic=ic))
    bc = [_region(0, "sponge_freund_ambient", s, case["sponge"], (ni, nj, 1)) for s in ("+xi", "-xi", "+eta", "-eta")]
    bc.append(_region(1, "wall_slip_kinematic", "+eta", 1, (257, 65, 1)))
    return dict(blocks=blocks, bc=bc, sim="CASE_TANNA_TPN49", source=(), tables=og.abi_tables(geo))


def prepare(case, seed):
    """The solver with its geometry, and the initial states a program holds."""
    from camille_amd import FP32, FP64, PATH_FUSED, PATH_PLAIN, Batch, Solver
    inp = _inputs(case, seed)
    prec = FP32 if case["prec"] == 32 else FP64
    geom = [{k: b[k] for k in ("x", "y", "z", "mean") if k in b} for b in inp["blocks"]]
    state = dict(case=case, ics=[b["ic"] for b in inp["blocks"]])
    if case["kind"] == "ensemble":
        state["solver"] = Batch([dict(g, boundaries=b["bc"], simulation=inp["sim"], source_params=b["source"],
                                      mode="FIX_CFL", value=CFL) for g, b in zip(geom, inp["blocks"])], precision=prec)
        return state
    s = Solver(geom, boundaries=inp["bc"], overset=inp.get("tables"), simulation=inp["sim"],
               source_params=inp["source"], precision=prec,
               path=PATH_PLAIN if case.get("path") == "plain" else PATH_FUSED, mode="FIX_CFL", value=CFL,
               num_dim=3 if "z" in geom[0] else 2)
    state["solver"] = s
    if "obs" in inp:
        obs = inp["obs"]
        s.set_observer_points(np.zeros(obs.size), obs, np.full(obs.size, 1.0 / obs.size))
        dtype = torch.float32 if case["prec"] == 32 else torch.float64
        state["q"] = torch.tensor(inp["q"], dtype=dtype, requires_grad=True)
        state["y0"] = torch.tensor(state["ics"][0], dtype=dtype, requires_grad=True)
    return state


def run(state):
    case, s = state["case"], state["solver"]
    if "q" in state:
        from camille_amd.adjoint import observer_energy
        q, y0 = state["q"], state["y0"]
        J = observer_energy(s, q, y0, case["steps"], case["steps"] // 2, case["every"])
        gq, gy = torch.autograd.grad(J, (q, y0))
        return [J.detach().to(q.dtype), gq, gy]
    for ib, ic in enumerate(state["ics"]):
        s.set_solution(ic, ib)
    s.set_time(0, 0.0, 1e-6)
    s.solve(case["steps"], sync=False)
    out = [torch.from_numpy(s.solution(ib)) for ib in range(len(state["ics"]))]
    # the fields of a 32-bit run hold 32-bit values; a program that keeps them keeps them so
    return [o.to(torch.float32) for o in out] if case["prec"] == 32 else out


# -------------------------------------------------------------------- work

def _points(case):
    if case["kind"] == "ensemble":
        return sum(ni * nj for ni, nj in _sizes(case))
    if case["kind"] == "overset":
        return case["ni"] * case["nj"] + 257 * 65
    return case["ni"] * case["nj"] * case.get("nk", 1)


def work(case):
    """Per step the state is read and written once and the geometry (and a
    sheared base flow) read once; the reverse pass recomputes the forward one
    and moves the adjoint state as well.  Operations: the derivative rows, the
    chain rule and the right-hand side of each stage, and the filter sweeps."""
    d3 = "nk" in case
    b = 4 if case["prec"] == 32 else 8
    nv, dim = (5, 3) if d3 else (4, 2)
    sheared = case.get("mean") == "shear" or case["kind"] in ("overset", "flow3d", "grad2d", "grad3d")
    point = 2 * nv * b + 8 * (dim * dim + 1) + (b * (22 if d3 else 14) if sheared else 0)
    flops = 4 * nv * (dim * 7 + dim * (2 * dim + 1) + 3 * dim + 6) + nv * (dim * 17 + 3)
    passes = 4 if case["kind"].startswith("grad") else 1  # forward, recomputed forward, adjoint (twice the fields)
    n = _points(case) * case["steps"] * passes
    return dict(bytes=n * point, flops=n * flops)


# ------------------------------------------------------------- exact values

_FD = {"in": {-2: 1 / 12, -1: -8 / 12, 1: 8 / 12, 2: -1 / 12}, "l0": {0: -1.5, 1: 2.0, 2: -0.5},
       "l1": {-1: -0.5, 1: 0.5}}
_FLT = {"in": [93 / 128, 7 / 32, -7 / 64, 1 / 32, -1 / 256], 0: [1.0], 1: [1.0], 2: [5 / 8, 1 / 4, -1 / 16],
        3: [11 / 16, 15 / 64, -3 / 32, 1 / 64]}


def _codes(shape, dim, nb, iblank):
    """Row of every point along `dim`: 0 interior, 1 none, 2 + k the k-th row
    from a left end, 2 + nb + k from a right end; grid ends first, then the
    ends of the runs between holes, in the order a scan meets them."""
    n = shape[dim]
    line = np.zeros(n, np.int64)
    for k in range(nb):
        line[k], line[n - 1 - k] = 2 + k, 2 + nb + k
    if iblank is None or not (iblank != 0).any():
        return line.reshape([n if q == dim else 1 for q in range(len(shape))])
    ib = np.moveaxis(iblank, dim, 0)
    code = np.repeat(line[:, None], ib.shape[1], 1)
    for c in range(n):
        last, hole = ib[max(c - 1, 0)], ib[c] == 1
        code[c][hole & (last == 1)] = 1
        for k in range(nb):
            if c - 1 - k >= 0:
                m = hole & (last == -1) if c > 0 else np.zeros_like(hole)
                code[c - 1 - k][m] = 2 + nb + k
            if c + k < n:
                code[c + k][~hole & (last == 1)] = 2 + k
    return np.moveaxis(code, 0, dim)


def _weights(code, nb, rows, dev):
    """{offset: weight of the point's row on that neighbour} from row codes."""
    out = {}
    for o in sorted({o for r in rows.values() for o in r[0]}):
        w = np.zeros(code.shape)
        for c, (row, sign) in rows.items():
            if o in row:
                w[code == c] = sign * row[o]
        if w.any():
            out[o] = torch.tensor(w, device=dev)
    return out


def _apply(f, weights, dim):
    """sum_o w_o f(. + o) along `dim` (counted from the end), f zero outside."""
    n = f.shape[dim]
    g = torch.nn.functional.pad(f, [0, 0] * (-1 - dim) + [4, 4])
    out = None
    for o, w in weights.items():
        t = w * g.narrow(dim, 4 + o, n)
        out = t if out is None else out + t
    return out


class _Block:
    """One block of the plain torch implementation."""

    def __init__(self, b, bc, iblank, sponge, dev):
        xs = [b["x"], b["y"]] + ([b["z"]] if "z" in b else [])
        self.D = D = len(xs)
        self.dev, shape = dev, b["x"].shape
        t = lambda a: torch.tensor(a, dtype=torch.float64, device=dev)  # noqa: E731
        X = torch.stack([t(a) for a in xs])
        axes = [-1, -2, -3][:D]
        fd, flt = [], []
        for a in axes:
            c = _codes(shape, len(shape) + a, 2, iblank)
            rev = lambda r: {-o: w for o, w in r.items()}  # noqa: E731
            fd.append((c, {0: (_FD["in"], 1), 2: (_FD["l0"], 1), 3: (_FD["l1"], 1), 4: (rev(_FD["l0"]), -1),
                           5: (rev(_FD["l1"]), -1)}))
            sym = lambda r: {s * o: w for o, w in enumerate(r) for s in (1, -1)}  # noqa: E731
            c8 = _codes(shape, len(shape) + a, 4, iblank)
            rows = {0: (sym(_FLT["in"]), 1)}
            for k in range(4):
                rows[2 + k] = rows[6 + k] = (sym(_FLT[k]), 1)
            flt.append((c8, rows))
        edge = [_weights(_codes(shape, len(shape) + a, 2, None), 2, fd[q][1], dev) for q, a in enumerate(axes)]
        self.axes = axes
        self.fd = [_weights(c, 2, r, dev) for c, r in fd]
        self.flt = [_weights(c, 4, r, dev) for c, r in flt]
        A = [[_apply(X[i], edge[q], axes[q]) for q in range(D)] for i in range(D)]  # d x_i / d xi_q
        if D == 2:
            self.m = [[A[1][1], -A[0][1]], [-A[1][0], A[0][0]]]
            self.J = 1.0 / (A[0][0] * A[1][1] - A[0][1] * A[1][0])
        else:
            cof = lambda l, i: (A[(i + 1) % 3][(l + 1) % 3] * A[(i + 2) % 3][(l + 2) % 3]  # noqa: E731
                                - A[(i + 1) % 3][(l + 2) % 3] * A[(i + 2) % 3][(l + 1) % 3])
            self.m = [[cof(q, i) for i in range(3)] for q in range(3)]
            self.J = 1.0 / sum(A[0][q] * self.m[q][0] for q in range(3))
        mean = t(b["mean"])
        self.u, self.sbar, self.pbar = mean[1:1 + D], mean[0], mean[4]
        self.rhob = (GAMMA * self.pbar) ** (1 / GAMMA) * torch.exp(-self.sbar)
        sheared = any(bool((mean[v] != mean[v].reshape(-1)[0]).any()) for v in range(5))
        self.gm = self.grad(mean) if sheared else None
        self.hole = None if iblank is None else torch.tensor(iblank == 1, device=dev)
        Tb = self.pbar * GAMMA / (GAMMA - 1.0) / self.rhob
        adv = sum((sum(self.m[q][k] * self.u[k] for k in range(D)) * self.m[q][i]).trunc().abs()
                  for q in range(D) for i in range(D))
        fac = sum(self.m[q][i] ** 2 for q in range(D) for i in range(D))
        rate = (adv + torch.sqrt((GAMMA - 1.0) * Tb) * torch.sqrt(fac)) * self.J
        if iblank is not None:
            rate = rate[torch.tensor(iblank == 0, device=dev)]
        self.rate = float(rate.max())
        self.sigma, self.walls = 0.0, []
        for line in bc:
            q, end = _SIDES[line[2]]
            if line[1] == "wall_slip_kinematic":
                self.walls.append((q, end))
                continue
            self.sigma = self.sigma + self._sponge(X, q, end, sponge)

    def _sponge(self, X, q, end, width):
        dim, n = X.dim() - 1 - q, X.shape[X.dim() - 1 - q]
        lo = 0 if end == 0 else n - width
        inner, outer = (width - 1, 0) if end == 0 else (n - width, n - 1)
        pts = X.narrow(dim, lo, width).reshape(self.D, -1).T.contiguous()
        dist = []
        for face in (inner, outer):
            f = X.select(dim, face).reshape(self.D, -1).T.contiguous()
            dist.append(torch.cat([sum((p[:, k, None] - f[None, :, k]) ** 2 for k in range(self.D)).min(1).values.sqrt()
                                   for p in pts.split(max(1, 20_000_000 // f.shape[0]))]))
        out = torch.zeros(X.shape[1:], dtype=X.dtype, device=X.device)
        z = out.narrow(dim - 1, lo, width)
        z.copy_((5.0 * (dist[0] / (dist[0] + dist[1])) ** 2).reshape(z.shape))
        return out

    def grad(self, f):
        """d f / d x_i of stacked fields, a list over i."""
        d = [_apply(f, self.fd[q], self.axes[q]) for q in range(self.D)]
        return [sum(self.m[q][i] * d[q] for q in range(self.D)) * self.J for i in range(self.D)]

    def aux(self, y):
        return self.rhob * (y[4] / (GAMMA * self.pbar) - y[0])

    def rhs(self, y, rho, source):
        D, u, up = self.D, self.u, y[1:1 + self.D]
        g = self.grad(y)
        gp = GAMMA * self.pbar
        out = -sum(u[i] * g[i] for i in range(D))
        vel = [out[1 + k] - g[k][4] / self.rhob for k in range(D)]
        s, p = out[0], out[4] - gp * sum(g[i][1 + i] for i in range(D))
        if self.gm is not None:
            gm = self.gm
            r = rho / self.rhob
            s = s - sum(up[i] * gm[i][0] for i in range(D))
            vel = [vel[k] - sum((up[i] + r * u[i]) * gm[i][1 + k] for i in range(D)) for k in range(D)]
            p = p - sum(up[i] * gm[i][4] for i in range(D)) - GAMMA * y[4] * sum(gm[i][1 + i] for i in range(D))
        if source is not None:
            p = p + source
        vel += [torch.zeros_like(s)] * (3 - D)
        return torch.stack([s] + vel + [p]) - self.sigma * y

    def bcs(self, y):
        for q, end in self.walls:
            dim = y.dim() - 1 - q
            n = y.shape[dim]
            f, s = (0, 1) if end == 0 else (n - 1, -1)
            at = lambda a, k: a.select(a.dim() - 1 - q, f + s * k)  # noqa: E731
            face = ((4.0 * at(y, 1) - at(y, 2)) / 3.0).clone()
            m = [[at(self.m[a][b], 0) for b in range(2)] for a in range(2)]
            v = at(y, 0)
            k = [m[0][0] * v[1] + m[0][1] * v[2], m[1][0] * v[1] + m[1][1] * v[2]]
            k[q] = torch.zeros_like(k[q])
            J = at(self.J, 0)
            face[1], face[2], face[3] = (m[1][1] * k[0] - m[0][1] * k[1]) * J, (m[0][0] * k[1] - m[1][0] * k[0]) * J, v[3]
            y = y.clone()
            y.select(dim, f).copy_(face)
        return y

    def filtered(self, y):
        for w, a in zip(self.flt, self.axes):
            y = _apply(y, w, a)
        return self.clear(y)

    def clear(self, y):
        return y if self.hole is None else torch.where(self.hole, torch.zeros_like(y), y)


def _step(blocks, ys, rhos, t, dt, sources, receive):
    """One RK4 step with the filter; t the clock after the step's increment."""
    b_i, c_i, a_n = (1 / 6, 1 / 3, 1 / 3, 1 / 6), (0.0, 0.5, 0.5, 1.0), (0.5, 0.5, 1.0)
    acc, u, rho = list(ys), list(ys), list(rhos)
    for i in range(4):
        for n, b in enumerate(blocks):
            if i:
                rho[n] = b.aux(u[n])
            k = dt * b.rhs(u[n], rho[n], None if sources[n] is None else sources[n](t + c_i[i] * dt))
            acc[n] = b.clear(acc[n] + b_i[i] * k)
            u[n] = b.clear(ys[n] + a_n[i] * k) if i < 3 else acc[n]
        u = receive([b.bcs(v) for b, v in zip(blocks, u)])
    return [b.filtered(v) for b, v in zip(blocks, u)], [b.aux(v) for b, v in zip(blocks, u)]


def _receiver(inp, dev):
    tb = inp.get("tables")
    if tb is None:
        return lambda ys: ys
    li = lambda k: torch.as_tensor(np.asarray(tb[k], np.int64), device=dev)  # noqa: E731
    rb, rl, db, dl = li("recv_block"), li("recv_l"), li("donor_block"), li("donor_l")
    coef = torch.as_tensor(np.asarray(tb["coef"], np.float64), device=dev)
    coef = coef / coef.sum(1, keepdim=True)
    ni = torch.as_tensor([b["x"].shape[1] for b in inp["blocks"]], device=dev)[db]
    q = torch.arange(25, device=dev)
    at = dl[:, None] + q % 5 + (q // 5) * ni[:, None]

    def receive(ys):
        flat = [y.reshape(5, -1) for y in ys]
        val = torch.zeros(5, rb.numel(), dtype=torch.float64, device=dev)
        for n, f in enumerate(flat):
            val[:, db == n] = (f[:, at[db == n]] * coef[db == n]).sum(-1)
        out = []
        for n, (f, y) in enumerate(zip(flat, ys)):
            f = f.clone()
            f[:, rl[rb == n]] = val[:, rb == n]
            out.append(f.reshape(y.shape))
        return out
    return receive


def _shape_of(b, src, dev):
    """A monopole's p-source as a function of time."""
    amp, omega, x0, y0, z0, w = src
    r2 = (b["x"] - x0) ** 2 + (b["y"] - y0) ** 2 + ((b["z"] - z0) ** 2 if "z" in b else 0.0)
    g = torch.tensor(np.exp(-LN2 * r2 / (w * w)), device=dev)
    return lambda t: amp * math.sin(omega * t) * g


def exact(case, seed):
    """What run() returns, from a plain torch implementation in 64 bits."""
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    inp = _inputs(case, seed)
    iblank = [None] * len(inp["blocks"])
    if "tables" in inp:
        tb = inp["tables"]
        for n, b in enumerate(inp["blocks"]):
            ib = np.zeros(b["x"].size, np.int64)
            ib[np.asarray(tb["hole_l"])[np.asarray(tb["hole_block"]) == n]] = 1
            ib[np.asarray(tb["recv_l"])[np.asarray(tb["recv_block"]) == n]] = -1
            iblank[n] = ib.reshape(b["x"].shape)
    together = case["kind"] == "overset"
    groups = [list(range(len(inp["blocks"])))] if together else [[n] for n in range(len(inp["blocks"]))]
    out = []
    for group in groups:
        raw = [inp["blocks"][n] for n in group]
        blocks = [_Block(b, b["bc"] if "bc" in b else [ln for ln in inp["bc"] if ln[0] == n], iblank[n],
                         case["sponge"], dev) for n, b in zip(group, raw)]
        dt = CFL / max(b.rate for b in blocks)
        ys = [torch.tensor(b["ic"], device=dev) for b in raw]
        if "q" in inp:
            return _gradients(case, inp, blocks[0], ys[0], dt, dev)
        sources = [_shape_of(b, b.get("source", inp.get("source")), dev) if inp["sim"] == "CASE_MONOPOLE" else None
                   for b in raw]
        receive = _receiver(inp, dev)
        rhos = [b.aux(y) for b, y in zip(blocks, ys)]
        for k in range(case["steps"]):
            ys, rhos = _step(blocks, ys, rhos, (k + 1) * dt, dt, sources, receive)
        out += [y.cpu() for y in ys]
    return out


def _gradients(case, inp, block, y0, dt, dev):
    from torch.utils.checkpoint import checkpoint
    dtype = torch.float32 if case["prec"] == 32 else torch.float64
    # the inputs as the program holds them
    q = torch.tensor(inp["q"], dtype=dtype).to(dev, torch.float64).requires_grad_(True)
    y0 = y0.to(dtype).double().requires_grad_(True)
    amp, omega = inp["source"]
    obs = torch.as_tensor(inp["obs"], device=dev)

    def step(y, rho, q, k):
        source = lambda t: amp * math.sin(omega * t) * q  # noqa: E731
        ys, rhos = _step([block], [y], [rho], (k + 1) * dt, dt, [source], lambda v: v)
        return ys[0], rhos[0]
    y, rho, J = y0, block.aux(y0), 0.0
    for k in range(case["steps"]):
        y, rho = checkpoint(step, y, rho, q, k, use_reentrant=False)
        if k + 1 > case["steps"] // 2:
            J = J + (y[4].reshape(-1)[obs] ** 2).sum() / obs.numel()
    gq, gy = torch.autograd.grad(J, (q, y0))
    return [J.detach().cpu(), gq.cpu(), gy.cpu()]
