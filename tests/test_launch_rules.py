"""Kernel forms that the launch rules pick by size, at the edges of the
rules: against plain formulas, the CPU oracle, or the form they replace."""
import numpy as np
import pytest

import boundary_tables
from camille_amd import FP32, FP64, PATH_PLAIN, Batch, LeeError, Solver
from test_zz_no_alloc import _noalloc

pytestmark = pytest.mark.gpu

GAMMA = 1.4


def _rel(a, b):
    return float(np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300))


def _box3(ni, nj, nk, seed, flow="general"):
    """A stretched 3-D box with a rough state and a base flow: "general" varies
    in every field, "jet" only in u(y, z), "rotor" in u and p."""
    rng = np.random.default_rng(seed)
    k, j, i = np.meshgrid(np.arange(nk), np.arange(nj), np.arange(ni), indexing="ij")
    x, y, z = (0.25 * a + 0.05 * np.sin(0.3 * a) for a in (i, j, k))
    mean = np.zeros((5, nk, nj, ni))
    mean[0] = 0.1 * np.sin(0.2 * x)
    mean[1] = 0.3 * np.tanh(0.4 * (y - y.mean()))
    mean[2] = 0.1 * np.cos(0.3 * z)
    mean[3] = 0.05 * np.sin(0.25 * x + 0.2 * y)
    mean[4] = (1.0 + 0.1 * np.cos(0.2 * z + 0.1 * x)) / GAMMA
    if flow != "general":
        mean[0], mean[2], mean[3] = 0.0, 0.1, 0.0
        mean[1] = 0.3 * np.tanh(0.4 * (y - y.mean())) * np.cos(0.2 * z)
    if flow == "jet":
        mean[4] = 1.0 / GAMMA
    return x, y, z, mean, rng.standard_normal((5, nk, nj, ni)), rng.standard_normal((5, nk, nj, ni))


# (131, 61, 45) takes chunks of 2 or 4 planes forwards and 3 or 4 backwards,
# with one plane left over; (70, 13, 9) and (9, 9, 14) take single planes
@pytest.mark.parametrize("dims", [(131, 61, 45), (70, 13, 9), (9, 9, 14)])
@pytest.mark.parametrize("flow", ["general", "jet", "rotor"])
@pytest.mark.parametrize("prec,tol", [(FP64, 1e-12), (FP32, 2e-5)])
def test_3d_stage_chunks(dims, flow, prec, tol):
    """The 3-D right-hand side equals its definition, built from the FP64
    derivative entry point, and its transpose satisfies <L y, k> = <y, L^T k>.
    FP32: some 40 terms of size 1 to 10, each rounded at 6e-8, relative to
    the largest value; the dot products gather random signs and stay below.
    The flows differ in which mean coefficient fields are constant and so read
    at one point."""
    x, y, z, mean, q, kap = _box3(*dims, seed=3, flow=flow)
    s = Solver([dict(x=x, y=y, z=z, mean=mean)], precision=prec, mode="FIX_DT", value=0.01, num_dim=3)
    d = [[s.take_derivative_xyz(f, i) for i in range(3)] for f in q]
    g = [[s.take_derivative_xyz(f, i) for i in range(3)] for f in mean]
    rhob = (GAMMA * mean[4]) ** (1 / GAMMA) * np.exp(-mean[0])
    rho = rhob * (q[4] / (GAMMA * mean[4]) - q[0])
    ub, up = mean[1:4], q[1:4]
    ref = np.zeros_like(q)
    for i in range(3):
        ref[0] -= ub[i] * d[0][i] + up[i] * g[0][i]
        ref[4] -= ub[i] * d[4][i] + up[i] * g[4][i] + GAMMA * (mean[4] * d[1 + i][i] + q[4] * g[1 + i][i])
        for v in range(3):
            ref[1 + v] -= ub[i] * d[1 + v][i] + (up[i] + rho / rhob * ub[i]) * g[1 + v][i]
        ref[1 + i] -= d[4][i] / rhob
    r = s.compute_rhs(q, 0.0)
    assert max(_rel(r[v], ref[v]) for v in range(5)) <= tol
    lk = s.compute_rhs_adjoint(kap)
    a, b = float(np.sum(r * kap)), float(np.sum(q * lk))
    assert abs(a - b) <= tol * np.linalg.norm(r) * np.linalg.norm(kap)
    s.close()


# a last column tile of 1, 4 and 1 points (11-point closure rows reach 8 back
# into the tile before) and of 62
@pytest.mark.parametrize("shape", [(65, 11), (68, 13), (129, 12), (126, 17)])
@pytest.mark.parametrize("order", [4, 11])
def test_plain_stage_tile_edges(shape, order):
    """The plain path equals the oracle bit for bit where its tiles end in
    slivers, with a sheared mean flow, a carried w', sponges and walls."""
    from oracle.pyoracle import Oracle
    ni, nj = shape
    rng = np.random.default_rng(7)
    i, j = np.meshgrid(np.arange(ni), np.arange(nj))
    x, y = 0.5 * i + 0.1 * np.sin(0.7 * j), 0.5 * j + 0.1 * np.sin(0.4 * i)
    mean = np.zeros((5, nj, ni))
    mean[0] = 0.05 * np.cos(0.3 * x)
    mean[1] = 0.2 * np.tanh(0.5 * (y - y.mean()))
    mean[4] = (1.0 + 0.05 * np.sin(0.2 * x + 0.3 * y)) / GAMMA
    ic = 1e-4 * rng.standard_normal((5, nj, ni))
    bc = [(0, "sponge_freund_ambient", "+xi", "0", "4", "0", "-0", "0", "0"),
          (0, "sponge_freund_ambient", "-xi", "-3", "-0", "0", "-0", "0", "0"),
          (0, "wall_slip_kinematic", "+eta", "0", "-0", "0", "0", "0", "0"),
          (0, "neumann", "-eta", "0", "-0", "-0", "-0", "0", "0")]
    scheme = dict(fd_order=order, filter_order=8 if order == 4 else 11, filter_blend=0.9, filter_strength=0.6, rk=4,
                  sponge_order=2, sponge_constant=5.0)
    o = Oracle([dict(x=x, y=y, mean=mean, ic=ic)], scheme, bc, None, "FIX_CFL", 0.4)
    o.run(6)
    s = Solver([dict(x=x, y=y, mean=mean)], boundaries=bc, precision=FP64, path=PATH_PLAIN, mode="FIX_CFL", value=0.4,
               fd_order=order, filter_order=scheme["filter_order"], filter_blend=0.9, filter_strength=0.6)
    s.set_solution(ic)
    s.solve(6)
    assert np.array_equal(s.solution(), o.solution(0)[:, 0])
    s.close()


def _pair_case(ni, nj, kind, seed):
    """A 2-D block whose sponges overlap in the corners, with a source inside
    one of them; kind: "sponges" (uniform mean), "sheared", "faces" (a BC on
    every side, meeting in the corners) or "wave" (a harmonic face and zone)."""
    rng = np.random.default_rng(seed)
    i, j = np.meshgrid(np.arange(ni), np.arange(nj))
    x, y = 0.5 * i + 0.1 * np.sin(0.7 * j), 0.5 * j + 0.1 * np.sin(0.4 * i)
    mean = np.zeros((5, nj, ni))
    mean[1], mean[2] = 0.3, -0.1
    mean[4] = 1.0 / GAMMA
    if kind in ("sheared", "faces"):
        mean[0] = 0.05 * np.cos(0.3 * x)
        mean[1] = 0.2 * np.tanh(0.5 * (y - y.mean()))
        mean[4] = (1.0 + 0.05 * np.sin(0.2 * x + 0.3 * y)) / GAMMA
    ic = 1e-4 * rng.standard_normal((5, nj, ni))
    ic[3] = 0.0
    bc = [(0, "sponge_freund_ambient", "+xi", "0", "6", "0", "-0", "0", "0"),
          (0, "sponge_freund_ambient", "+eta", "0", "-0", "0", "5", "0", "0"),
          (0, "sponge_freund_ambient", "-eta", "0", "-0", "-4", "-0", "0", "0")]
    harmonic = None
    if kind == "faces":
        bc = [(0, "wall_slip_kinematic", "+eta", "0", "-0", "0", "0", "0", "0"),
              (0, "neumann", "+xi", "0", "0", "0", "-0", "0", "0"),
              (0, "dirichlet_allzero", "-xi", "-0", "-0", "2", "-3", "0", "0"),
              (0, "wall_slip_kinematic", "-eta", "0", "-0", "-0", "-0", "0", "0")]
    if kind == "wave":
        bc = [(0, "dirichlet_harmonicwave", "+xi", "0", "0", "0", "-0", "0", "0"),
              (0, "sponge_freund_harmonicwave", "+xi", "0", "6", "0", "-0", "0", "0"),
              (0, "sponge_freund_ambient", "-eta", "0", "-0", "-4", "-0", "0", "0")]
        harmonic = dict(wave="WAVE_ENTROPY", shape="WAVEFORM_GAUSSIAN_ROUNDJET", direction="X", amplitude=0.02,
                        wavelength=5.0, halfwidth=1.5)
    src = (1e-3, 0.6, float(x[2, 3]), float(y[2, 3]), 0.0, 1.0)
    return dict(x=x, y=y, mean=mean), ic, dict(boundaries=bc, harmonic=harmonic, simulation="CASE_MONOPOLE",
                                               source_params=src, mode="FIX_CFL", value=0.4)


# tiles of 60 x 4 and 60 x 12 points: one point past a tile, one short of it,
# blocks narrower than a tile's halo, and one with tiles inside the block
@pytest.mark.parametrize("shape", [(61, 13), (60, 12), (59, 25), (9, 9), (9, 131), (181, 121), (721, 500)])
@pytest.mark.parametrize("kind", ["sponges", "sheared", "faces", "wave"])
@pytest.mark.parametrize("prec", [FP64, FP32])
def test_paired_stages_bit_identical(shape, kind, prec):
    """Two RK stages a launch, as the tuner picks them, against one stage a
    launch (a pinned tile shape), bit for bit after 5 steps."""
    block, ic, kw = _pair_case(*shape, kind, seed=11)
    out = []
    for pinned in (False, True):
        s = Solver([block], precision=prec, **kw)
        s.set_solution(ic)
        if pinned:
            s.set_tile_shape(1, 4)
        else:
            s.autotune()
            s.set_kernel_timing(True)
        s.solve(5)
        if not pinned:
            print(shape, kind, prec, "launches", {k: v[1] for k, v in s.kernel_timing().items()}, flush=True)
        out.append((s.solution(), s.clock()))
        s.close()
    assert np.all(np.isfinite(out[0][0]))
    assert np.array_equal(out[0][0], out[1][0]) and out[0][1] == out[1][1]


def _launched(s, steps):
    """Stage launches of `steps` steps: (first, middle, last class)."""
    s.set_kernel_timing(True)
    s.solve(steps)
    n = {k: v[1] for k, v in s.kernel_timing().items()}
    s.set_kernel_timing(False)
    return tuple(n["stage_" + k] for k in ("first", "mid", "last"))


@pytest.mark.parametrize("shape", [(61, 13), (60, 12), (59, 25), (9, 9), (9, 12), (9, 131), (181, 121)])
@pytest.mark.parametrize("kind", ["sponges", "sheared", "faces", "wave"])
@pytest.mark.parametrize("prec", [FP64, FP32])
def test_both_paired_forms_bit_identical(shape, kind, prec):
    """Two RK stages a launch, with tiles of one and of two rows per wave,
    against one stage a launch, bit for bit after 5 steps; the launches of
    every run are counted."""
    block, ic, kw = _pair_case(*shape, kind, seed=11)
    s = Solver([block], precision=prec, **kw)
    if shape == (9, 9) and kind in ("sponges", "sheared"):  # its three sponges meet
        with pytest.raises(LeeError, match="no three"):
            s.set_stage_pairs(1)
        return
    out = []
    for rows in (0, 1, 2):
        s.set_stage_pairs(rows)
        assert s.stage_pairs() == rows
        s.set_solution(ic)
        s.set_time(0, 0.0, 1e-6)
        assert _launched(s, 5) == ((5, 10, 5) if rows == 0 else (5, 0, 5))
        out.append((s.solution(), s.clock()))
    s.set_tile_shape(*s.tile_shape())
    assert s.stage_pairs() == 0
    s.close()
    assert np.all(np.isfinite(out[0][0]))
    for o in out[1:]:
        assert np.array_equal(o[0], out[0][0]) and o[1] == out[0][1]


@pytest.mark.parametrize("kind", ["sponges", "sheared"])
@pytest.mark.parametrize("prec", [FP64, FP32])
def test_both_paired_forms_of_a_batch(kind, prec):
    """The same for a batch of uneven solves, against one stage a launch."""
    cases = [_pair_case(*shape, kind, seed=3 + k) for k, shape in
             enumerate([(61, 13), (9, 12), (120, 24), (59, 131), (181, 121)])]
    b = Batch([dict(block, **{k: v for k, v in kw.items() if k != "harmonic"}) for block, _, kw in cases], precision=prec)
    out = []
    for rows in (0, 1, 2):
        b.set_tile_shape(1, 4)
        b.set_stage_pairs(rows)
        assert b.stage_pairs() == rows
        for k, (_, ic, _) in enumerate(cases):
            b.set_solution(ic, k)
        b.set_time(0, 0.0, 1e-6)
        b.solve(3)  # replays of the captured step
        assert _launched(b, 2) == ((2, 4, 2) if rows == 0 else (2, 0, 2))
        out.append([b.solution(k) for k in range(len(cases))])
    b.close()
    for o in out[1:]:
        assert all(np.all(np.isfinite(q)) and np.array_equal(p, q) for p, q in zip(o, out[0]))


def test_paired_form_is_searched_for_on_the_device():
    """On a small block a launch takes the host longer than the device, and the
    paired forms as long as each other there: the search has to see that one
    row per wave takes the device a third less than two, every time."""
    block, ic, kw = _pair_case(97, 81, "sponges", seed=2)
    s = Solver([block], precision=FP32, **kw)
    s.set_solution(ic)
    picks = []
    for _ in range(16):
        s.autotune()
        picks.append(s.stage_pairs())
    s.close()
    assert picks == [1] * 16


def test_stage_pairs_are_refused_where_they_cannot_run():
    block, _, kw = _pair_case(61, 33, "sponges", seed=1)
    for bad in (dict(kw, rk=2), dict(kw, fd_order=11), dict(kw, path=PATH_PLAIN),
                dict(kw, boundaries=[(0, "sponge_freund_ambient", "+xi", "0", "4", str(5 * q), str(5 * q + 3), "0", "0")
                                     for q in range(5)])):
        s = Solver([block], precision=FP64, **bad)
        for rows in (1, 2):
            with pytest.raises(LeeError, match="two RK stages"):
                s.set_stage_pairs(rows)
        s.set_stage_pairs(0)
        assert s.stage_pairs() == 0
        with pytest.raises(LeeError, match="1 or 2 rows"):
            s.set_stage_pairs(3)
        s.close()


_FACES = {
    "none": [],
    "walls": [(0, "wall_slip_kinematic", "+eta", "0", "-0", "0", "0", "0", "0"),
              (1, "neumann", "-xi", "-0", "-0", "0", "-0", "0", "0")],
    "meeting": [(0, "neumann", "+xi", "0", "0", "0", "-0", "0", "0"),
                (0, "wall_slip_kinematic", "+eta", "0", "-0", "0", "0", "0", "0"),
                (1, "dirichlet_allzero", "-eta", "0", "-0", "-0", "-0", "0", "0")],
}


# receivers that other sums and faces read, that faces write, and whose
# stencils read what faces write; "twice" names points twice, which has no order
@pytest.mark.parametrize("nrecv", [1, 25, 26, 51, 700])
@pytest.mark.parametrize("faces", list(_FACES))
@pytest.mark.parametrize("twice", [False, True])
def test_boundary_phase_in_one_launch(nrecv, faces, twice):
    """The faces and the interpolation in one launch against the launch per
    face, gather and scatter, bit for bit, over three applications in a row."""
    rng = np.random.default_rng(nrecv)
    dims = [(41, 31), (67, 23)]
    blocks = []
    for ni, nj in dims:
        i, j = np.meshgrid(np.arange(ni), np.arange(nj))
        mean = np.zeros((5, nj, ni))
        mean[4] = 1.0 / GAMMA
        blocks.append(dict(x=i + 0.1 * np.sin(0.5 * j), y=j + 0.1 * np.sin(0.4 * i), mean=mean))
    pts = np.array([(b, p) for b, (ni, nj) in enumerate(dims) for p in range(ni * nj)])
    recv = pts[rng.permutation(len(pts))[:nrecv]]
    db = rng.integers(0, 2, nrecv)
    dl = np.array([rng.integers(0, dims[b][1] - 4) * dims[b][0] + rng.integers(0, dims[b][0] - 4) for b in db])
    coef = rng.uniform(0.1, 1.0, (nrecv, 25))
    if twice:
        recv[-1], db[-1], dl[-1], coef[-1] = recv[0], db[0], dl[0], coef[0]
    tables = dict(recv_block=recv[:, 0], recv_l=recv[:, 1], donor_block=db, donor_l=dl,
                  widths=np.array([[5, 5, 1], [5, 5, 1]]), coef=coef, hole_block=np.zeros(0, int),
                  hole_l=np.zeros(0, int))
    s = Solver(blocks, overset=tables, boundaries=_FACES[faces], precision=FP64, mode="FIX_DT", value=0.01)
    ys = [rng.standard_normal((5, nj, ni)) for ni, nj in dims]
    for _ in range(3):
        want = _noalloc(s, ys)
        ys = s.update_boundary(ys)
        for got, ref in zip(ys, want):
            assert np.all(np.isfinite(got)) and np.array_equal(got, ref)
    s.close()


@pytest.mark.parametrize("shear", [False, True])
@pytest.mark.parametrize("prec", [FP64, FP32])
@pytest.mark.parametrize("nscalar", [0, 2])
def test_boundary_phase_forms_agree_over_a_run(shear, prec, nscalar):
    """Steps of an overset run whose boundary phase is one launch against the
    same run with a receiver named twice, which takes a launch per face, gather
    and scatter (test_host_runs pins both for these tables), bit for bit: with
    the aux density refreshed (sheared mean), in both precisions and with
    scalars, of which fewer receivers fit a workgroup."""
    rng = np.random.default_rng(5)
    blocks, ics = [], []
    for ni, nj in boundary_tables.DIMS:
        i, j = np.meshgrid(np.arange(ni), np.arange(nj))
        x, y = i + 0.1 * np.sin(0.5 * j), j + 0.1 * np.sin(0.4 * i)
        mean = np.zeros((5 + nscalar, nj, ni))
        mean[1], mean[4] = 0.2, 1.0 / GAMMA
        if shear:
            mean[1] = 0.2 * np.tanh(0.1 * (y - y.mean()))
            mean[4] = (1.0 + 0.05 * np.sin(0.1 * x)) / GAMMA
        for z in range(nscalar):
            mean[5 + z] = 0.1 * np.cos(0.05 * x + z)
        ic = 1e-3 * rng.standard_normal(mean.shape)
        ic[3] = 0.0
        blocks.append(dict(x=x, y=y, mean=mean))
        ics.append(ic)
    out = []
    for twice in (False, True):
        s = Solver(blocks, overset=boundary_tables.tables(20, 10, 200, 30, 8, twice=twice), precision=prec,
                   boundaries=[boundary_tables.WALL], mode="FIX_DT", value=0.05, num_scalar=nscalar)
        for ib, ic in enumerate(ics):
            s.set_solution(ic, ib)
        s.solve(6)
        out.append([s.solution(ib) for ib in range(2)])
        s.close()
    for a, b in zip(*out):
        assert np.all(np.isfinite(a)) and np.array_equal(a, b)


@pytest.mark.parametrize("dims", [(150, 70), (90, 21, 19)])
def test_transposed_rows_round_their_smallest_product(dims):
    """FP32 adjoint of the right-hand side under a uniform mean flow, inside the
    block, against the same sums in numpy: each direction's row rounds its
    first product, weight 1/12, and fuses the others onto it.  Sums formed in
    64 bits and rounded once stand for the fused ones, and fluxes that are
    rounded from 64 bits may fall on the other side of a tie: 1 point in 1000
    may differ; with another order of the fusions 90 to 250 do."""
    d3 = len(dims) == 3
    axes = np.meshgrid(*[np.arange(n) for n in dims[::-1]], indexing="ij")[::-1]
    if d3:
        xyz = [0.25 * a + 0.05 * np.sin(0.3 * a) for a in axes]
    else:
        xyz = [0.5 * axes[0] + 0.1 * np.sin(0.7 * axes[1]), 0.5 * axes[1] + 0.1 * np.sin(0.4 * axes[0])]
    mean = np.zeros((5,) + axes[0].shape)
    ub = [0.3, -0.2, 0.1][:len(dims)]
    for d, u in enumerate(ub):
        mean[1 + d] = u
    mean[4] = 1.0 / GAMMA
    s = Solver([dict(zip("xyz", xyz), mean=mean)], precision=FP32, mode="FIX_DT", value=0.01, num_dim=len(dims))
    met, jac = s.metrics()
    kap = np.random.default_rng(3).standard_normal(mean.shape).astype(np.float32)
    if not d3:
        kap[3] = 0
    got = s.compute_rhs_adjoint(kap.astype(np.float64))
    s.close()
    f32, k = np.float32, kap.astype(np.float64)
    w = [f32(-1.0 / 12.0), f32(8.0 / 12.0), -f32(8.0 / 12.0), -f32(-1.0 / 12.0)]
    lam = [np.zeros(axes[0].shape, f32) for _ in range(5)]
    gp, irb = GAMMA * (1.0 / GAMMA), 1.0 / (GAMMA * (1.0 / GAMMA)) ** (1.0 / GAMMA)
    for q in range(len(dims)):
        m = [met[q][i] for i in range(len(dims))]
        U = sum(m[i] * ub[i] for i in range(len(dims)))
        F = [U * k[v] for v in range(5)]
        for i in range(len(dims)):
            F[1 + i] = F[1 + i] + m[i] * (gp * k[4])
        F[4] = F[4] + sum(m[i] * k[1 + i] for i in range(len(dims))) * irb
        for v in range(5):
            f = (F[v] * -jac).astype(f32)
            at = [np.roll(f, -o, axis=axes[0].ndim - 1 - q) for o in (-2, -1, 1, 2)]
            acc = w[0] * at[0]
            for e in range(1, 4):
                acc = (np.float64(w[e]) * at[e] + acc.astype(np.float64)).astype(f32)
            lam[v] = lam[v] + acc
    inner = tuple([slice(4, -4)] * len(dims))
    for v in [0, 1, 2, 4] + ([3] if d3 else []):
        off = np.mean(got[v][inner] != lam[v][inner].astype(np.float64))
        assert off <= 1e-3, (v, off)


@pytest.mark.parametrize("prec", [FP64, FP32])
@pytest.mark.parametrize("end", [0, 1])
def test_closure_rows_keep_infinities(prec, end):
    """An infinite value two points from a face, which the first two closure
    rows read once, gives the infinities and NaNs that the rows' definition
    gives: two RK stages a launch as one a launch, and the 3-D right-hand side
    as its formula from the derivative entry point."""
    ni, nj = 90, 41
    i, j = np.meshgrid(np.arange(ni), np.arange(nj))
    mean = np.zeros((5, nj, ni))
    mean[1], mean[2], mean[4] = 0.3, 0.2, 1.0 / GAMMA
    ic = 1e-3 * np.random.default_rng(4).standard_normal((5, nj, ni))
    ic[3] = 0.0
    ic[4, 20, 2 if end == 0 else ni - 3] = np.inf
    s = Solver([dict(x=0.5 * i + 0.1 * j, y=0.4 * j - 0.1 * i, mean=mean)], precision=prec, filter_order=0, mode="FIX_DT",
               value=0.01)
    out = []
    for rows in (0, 1, 2):
        s.set_stage_pairs(rows)
        s.set_solution(ic)
        s.solve(1)
        out.append(s.solution())
    s.close()
    assert np.isinf(out[0]).any()
    for o in out[1:]:
        assert np.array_equal(o, out[0], equal_nan=True)

    dims = (40, 19, 11)
    k, j, i = np.meshgrid(*[np.arange(n) for n in dims[::-1]], indexing="ij")
    xyz = dict(x=0.5 * i - 0.1 * j - 0.05 * k, y=0.5 * j - 0.1 * k - 0.1 * i, z=0.4 * k - 0.1 * i - 0.05 * j)
    mean = np.zeros((5,) + i.shape)
    ub = (0.3, 0.2, 0.1)
    for d in range(3):
        mean[1 + d] = ub[d]
    mean[4] = 1.0 / GAMMA
    y = 1e-3 * np.random.default_rng(5).standard_normal(mean.shape)
    y[0, 5, 9, 2 if end == 0 else dims[0] - 3] = np.inf
    y[0, 5, 2 if end == 0 else dims[1] - 3, 20] = np.inf
    s = Solver([dict(mean=mean, **xyz)], precision=prec, mode="FIX_DT", value=0.01, num_dim=3)
    ref = -sum(ub[d] * s.take_derivative_xyz(y[0], d) for d in range(3))
    r = s.compute_rhs(y, 0.0)[0]
    s.close()
    assert np.isinf(ref).sum() >= 4
    assert np.array_equal(np.isnan(r), np.isnan(ref)) and np.array_equal(np.isinf(r), np.isinf(ref))


@pytest.mark.parametrize("prec", [FP64, FP32])
@pytest.mark.parametrize("dims,at", [((70, 40), (33, 20)), ((70, 40), (6, 9)), ((40, 19, 15), (20, 9, 7)),
                                     ((40, 19, 15), (5, 5, 5))])
def test_transposed_rows_leave_out_their_own_point(prec, dims, at):
    """An infinite adjoint value inside the block reaches the neighbours whose
    rows read it and not its own point, which no row but a line's first and
    last reads, under a uniform mean without sponges."""
    d3 = len(dims) == 3
    axes = np.meshgrid(*[np.arange(n) for n in dims[::-1]], indexing="ij")[::-1]
    xyz = dict(zip("xyz", [0.5 * axes[0] - 0.1 * axes[1], 0.4 * axes[1] + 0.1 * axes[0]]
                   + ([0.3 * axes[2] - 0.05 * axes[0]] if d3 else [])))
    mean = np.zeros((5,) + axes[0].shape)
    mean[1], mean[2], mean[4] = 0.3, 0.2, 1.0 / GAMMA
    s = Solver([dict(mean=mean, **xyz)], precision=prec, mode="FIX_DT", value=0.01, num_dim=len(dims))
    kap = np.random.default_rng(6).standard_normal(mean.shape)
    if not d3:
        kap[3] = 0
    kap[(0,) + at[::-1]] = np.inf
    lam = s.compute_rhs_adjoint(kap)
    s.close()
    assert np.isfinite(lam[(0,) + at[::-1]])
    assert np.isinf(lam[0]).sum() == 4 * len(dims) and not np.isnan(lam).any()
