"""viscosity() on the GPU (bmg_viscosity, viscosity.h:163-178) against the
oracle's restatement (oracle/viscosity.py): with the reference's default
in-place Gauss-Seidel (hyperplanes on the GPU, the serial loop in the
oracle), the Jacobi relax_viscosity (the reference's JACOBI variant) and
the red-black Gauss-Seidel extension, the solver statistics and every velocity component equal the
oracle's bit for bit, for variable and constant mu and rho, the default wall
BCs and no slip, periodic dimensions, in 2D and 3D.  The oracle is pinned
by test_viscosity_oracle.py."""
import numpy as np
import pytest

import basilisk_amd as bmg
from oracle.viscosity import Viscosity

pytestmark = pytest.mark.gpu


def _problem(dim, depth, seed, variable):
    rng = np.random.default_rng(seed)
    n = 1 << depth
    u = [np.ascontiguousarray(rng.standard_normal((n,) * dim)) for _ in range(dim)]
    if variable:
        mu = [np.ascontiguousarray(rng.uniform(0.2, 3.0, tuple(n + (1 if e == d else 0) for e in range(dim))))
              for d in range(dim)]
        rho = np.ascontiguousarray(np.where(rng.uniform(size=(n,) * dim) < 0.3, 10.0, 1.0))
    else:
        mu, rho = 0.8, 1.5
    return u, mu, rho


@pytest.mark.parametrize("dim,depth", [(2, 6), (2, 7), (3, 4), (3, 5)])
@pytest.mark.parametrize("variable", [True, False])
@pytest.mark.parametrize("noslip", [False, True])
@pytest.mark.parametrize("smoother", ["jacobi", "rbgs"])
def test_viscosity_bitexact(dim, depth, variable, noslip, smoother):
    print("case viscosity", dim, depth, variable, noslip, smoother, flush=True)
    u, mu, rho = _problem(dim, depth, 100 * dim + depth, variable)
    dt = 0.004
    sigma = -np.ones((dim, 2 * dim), np.int64) if noslip else None
    g = bmg.Grid(dim, depth, smoother=smoother)
    g.set_tolerance(1e-8)
    o = Viscosity(dim, depth)
    o.smoother = smoother
    o.TOLERANCE = 1e-8
    if noslip:
        o.sigma = sigma
    o.set_coefficients(mu, rho)
    uo, so, _ = o.solve(u, dt)
    ug = [x.copy() for x in u]
    sg = g.viscosity(ug, mu=mu, rho=rho, dt=dt, sigma=sigma)
    for k in ("i", "resb", "resa", "nrelax", "minlevel"):
        assert sg[k] == so[k], (k, sg, so)
    assert abs(sg["sum"] - so["sum"]) <= 1e-9 * (1.0 + abs(so["sum"]))
    for c in range(dim):
        assert np.array_equal(ug[c], uo[c]), c


def test_viscosity_device_tensors():
    torch = pytest.importorskip("torch")
    print("case viscosity tensors", flush=True)
    dim, depth = 3, 5
    u, mu, rho = _problem(dim, depth, 7, True)
    g = bmg.Grid(dim, depth)
    g.set_tolerance(1e-9)
    uh = [x.copy() for x in u]
    sh = g.viscosity(uh, mu=mu, rho=rho, dt=0.01)
    ud = [torch.tensor(x, device="cuda:0") for x in u]
    md = [torch.tensor(m, device="cuda:0") for m in mu]
    rd = torch.tensor(rho, device="cuda:0")
    sd = g.viscosity(ud, mu=md, rho=rd, dt=0.01)
    assert sh == sd
    for c in range(dim):
        assert np.array_equal(ud[c].cpu().numpy(), uh[c])


def test_viscosity_zero_dt_is_identity_and_errors():
    print("case viscosity errors", flush=True)
    g = bmg.Grid(2, 5)
    u, mu, rho = _problem(2, 5, 3, True)
    ug = [x.copy() for x in u]
    s = g.viscosity(ug, mu=mu, rho=rho, dt=0.0)
    assert s["i"] == 1 and s["resb"] == 0.0
    for c in range(2):
        assert np.array_equal(ug[c], u[c])
    with pytest.raises(bmg.BMGError):
        g.viscosity([x.copy() for x in u], mu=mu, rho=rho, dt=0.1, sigma=[[2, 1, 1, 1], [1, 1, 1, 1]])
    with pytest.raises(bmg.BMGError):
        g.viscosity([x.copy() for x in u], mu=1.0, rho=-1.0, dt=0.1)


@pytest.mark.parametrize("dim,depth,periodic", [(2, 6, (True, False)), (2, 6, (False, True)), (2, 5, (True, True)),
                                                (3, 4, (True, False, True)), (3, 4, (True, True, True)),
                                                (2, 1, (True, True)), (3, 2, (False, True, False))])
@pytest.mark.parametrize("variable", [True, False])
@pytest.mark.parametrize("smoother", ["jacobi", "rbgs"])
def test_viscosity_periodic_bitexact(dim, depth, periodic, variable, smoother):
    """Periodic dimensions (grid/multigrid.h:600-701): wrapped ghosts, the
    level-0 root rule, and face n of mu replaced by face 0 (random values
    are given for face n, so reading it would show)."""
    print("case viscosity periodic", dim, depth, periodic, variable, smoother, flush=True)
    u, mu, rho = _problem(dim, depth, 31 * dim + depth + 7 * sum(periodic), variable)
    dt = 0.004
    g = bmg.Grid(dim, depth, smoother=smoother)
    for d in range(dim):
        if periodic[d]:
            g.set_periodic(d)
    g.set_tolerance(1e-8)
    o = Viscosity(dim, depth)
    o.smoother = smoother
    o.TOLERANCE = 1e-8
    o.periodic = list(periodic)
    o.set_coefficients(mu, rho)
    uo, so, _ = o.solve(u, dt)
    ug = [x.copy() for x in u]
    sg = g.viscosity(ug, mu=mu, rho=rho, dt=dt)
    for k in ("i", "resb", "resa", "nrelax", "minlevel"):
        assert sg[k] == so[k], (k, sg, so)
    for c in range(dim):
        assert np.array_equal(ug[c], uo[c]), c


@pytest.mark.parametrize("dim,depth", [(2, 1), (2, 2), (3, 1), (3, 2)])
@pytest.mark.parametrize("smoother", ["jacobi", "rbgs"])
def test_viscosity_tiny_grids_bitexact(dim, depth, smoother):
    """Grids of 2 and 4 cells per side: the single-cell level 0 and pairs
    that touch both walls."""
    print("case viscosity tiny", dim, depth, smoother, flush=True)
    u, mu, rho = _problem(dim, depth, 7 * dim + depth, True)
    g = bmg.Grid(dim, depth, smoother=smoother)
    g.set_tolerance(1e-10)
    o = Viscosity(dim, depth)
    o.smoother = smoother
    o.TOLERANCE = 1e-10
    o.set_coefficients(mu, rho)
    uo, so, _ = o.solve(u, 0.05)
    ug = [x.copy() for x in u]
    sg = g.viscosity(ug, mu=mu, rho=rho, dt=0.05)
    for k in ("i", "resb", "resa", "nrelax"):
        assert sg[k] == so[k], (k, sg, so)
    for c in range(dim):
        assert np.array_equal(ug[c], uo[c]), c


@pytest.mark.parametrize("depth", [5, 7])
@pytest.mark.parametrize("smoother", ["jacobi", "rbgs"])
@pytest.mark.parametrize("y0", [0.0, 0.5])
def test_viscosity_axi_bitexact(depth, smoother, y0):
    """The AXI form (viscosity.h:12-14; pinned in test_viscosity_oracle.py
    by second-order convergence to the axisymmetric operator): mu times the
    metric (the cell's y on x faces, the face's y on y faces, with a random
    variation), rho times the cell's y, no slip on the walls; statistics and
    both components equal the oracle's bit for bit, the box from y0."""
    print("case viscosity axi", depth, smoother, y0, flush=True)
    rng = np.random.default_rng(17 + depth)
    n = 1 << depth
    D = 1.0 / n
    yc = (np.arange(n) + 0.5) * D + y0
    yf = np.arange(n + 1) * D + y0
    mux = np.ascontiguousarray(np.tile(yc[None, :], (n + 1, 1)) * rng.uniform(0.5, 2.0, (n + 1, n)))
    muy = np.ascontiguousarray(np.tile(yf[None, :], (n, 1)) * rng.uniform(0.5, 2.0, (n, n + 1)))
    rho = np.ascontiguousarray(np.tile(yc[None, :], (n, 1)) * np.where(rng.uniform(size=(n, n)) < 0.3, 5.0, 1.0))
    u = [np.ascontiguousarray(rng.standard_normal((n, n))) for _ in range(2)]
    sigma = -np.ones((2, 4), np.int64)
    dt = 0.02
    g = bmg.Grid(2, depth, origin=(0.0, y0, 0.0), smoother=smoother)
    g.set_axi(True)
    g.set_tolerance(1e-9)
    o = Viscosity(2, depth, Y0=y0, axi=True)
    o.smoother = smoother
    o.TOLERANCE = 1e-9
    o.sigma = sigma
    o.set_coefficients([mux, muy], rho)
    uo, so, _ = o.solve(u, dt)
    ug = [x.copy() for x in u]
    sg = g.viscosity(ug, mu=[mux, muy], rho=rho, dt=dt, sigma=sigma)
    for k in ("i", "resb", "resa", "nrelax", "minlevel"):
        assert sg[k] == so[k], (k, sg, so)
    for c in range(2):
        assert np.array_equal(ug[c], uo[c]), c
    # AXI off again: the plain operator (a different solution)
    g.set_axi(False)
    ug2 = [x.copy() for x in u]
    g.viscosity(ug2, mu=[mux, muy], rho=rho, dt=dt, sigma=sigma)
    assert not np.array_equal(ug2[1], ug[1])
    with pytest.raises(bmg.BMGError):
        bmg.Grid(3, 3).set_axi(True)


@pytest.mark.parametrize("dim,depth,case", [(2, 5, "walls"), (2, 4, "noslip"), (2, 4, "periodic"), (2, 4, "axi"),
                                            (3, 3, "walls"), (3, 3, "periodic"), (2, 1, "walls"), (3, 2, "noslip")])
def test_viscosity_gauss_seidel_bitexact(dim, depth, case):
    """relax_viscosity without -DJACOBI, the reference's default: each cell
    overwritten as the i-major loop visits it.  The GPU sweeps hyperplanes
    (4i + 2j + k, or 2i + j); the oracle runs the serial loop.  Statistics
    and every component equal bit for bit (sizes the serial loop finishes
    in seconds)."""
    print("case viscosity gs", dim, depth, case, flush=True)
    u, mu, rho = _problem(dim, depth, 53 * dim + depth, True)
    dt = 0.004
    g = bmg.Grid(dim, depth, smoother="gs")
    g.set_tolerance(1e-8)
    o = Viscosity(dim, depth, axi=case == "axi")
    o.smoother = "gs"
    o.TOLERANCE = 1e-8
    sigma = None
    if case == "noslip" or case == "axi":
        sigma = -np.ones((dim, 2 * dim), np.int64)
        o.sigma = sigma
    if case == "periodic":
        o.periodic = [True] + [False] * (dim - 1)
        g.set_periodic(0)
        mu = [m.copy() for m in mu]
        mu[0][-1] = mu[0][0]
    if case == "axi":
        g.set_axi(True)
    o.set_coefficients(mu, rho)
    uo, so, _ = o.solve(u, dt)
    ug = [x.copy() for x in u]
    sg = g.viscosity(ug, mu=mu, rho=rho, dt=dt, sigma=sigma)
    for k in ("i", "resb", "resa", "nrelax", "minlevel"):
        assert sg[k] == so[k], (k, sg, so)
    for c in range(dim):
        assert np.array_equal(ug[c], uo[c]), c


@pytest.mark.parametrize("dim,depth,axi", [(2, 6, False), (2, 6, True), (3, 5, False)])
def test_viscosity_explicit_bitexact(dim, depth, axi):
    """viscosity_explicit(): u += residual_viscosity (u, u), resb."""
    print("case viscosity explicit", dim, depth, axi, flush=True)
    u, mu, rho = _problem(dim, depth, 71 * dim + depth, True)
    dt = 0.003
    g = bmg.Grid(dim, depth)
    if axi:
        g.set_axi(True)
    o = Viscosity(dim, depth, axi=axi)
    o.set_coefficients(mu, rho)
    uo, so = o.explicit(u, dt)
    ug = [x.copy() for x in u]
    sg = g.viscosity(ug, mu=mu, rho=rho, dt=dt, explicit=True)
    assert sg["resb"] == so["resb"] and sg["i"] == 0
    for c in range(dim):
        assert np.array_equal(ug[c], uo[c]), c


@pytest.mark.parametrize("dim,depth", [(2, 3), (2, 4), (2, 5), (3, 3), (3, 6)])
def test_viscosity_coarse_workgroup_bitexact(dim, depth):
    """Grids below, at and above the size whose levels all run in one
    workgroup, periodic along x, with large coefficient jumps."""
    print("case viscosity coarse", dim, depth, flush=True)
    u, mu, rho = _problem(dim, depth, 31 * dim + depth, True)
    for c in range(dim):  # face n is face 0 along a periodic dimension
        if c == 0:
            mu[c][-1] = mu[c][0]
    g = bmg.Grid(dim, depth)
    g.set_periodic(0)
    g.set_tolerance(1e-7)
    o = Viscosity(dim, depth)
    o.smoother = "rbgs"
    o.TOLERANCE = 1e-7
    o.periodic = tuple([True] + [False] * (dim - 1))
    o.set_coefficients(mu, rho)
    uo, so, _ = o.solve(u, 0.003)
    ug = [x.copy() for x in u]
    sg = g.viscosity(ug, mu=mu, rho=rho, dt=0.003)
    assert (sg["i"], sg["resb"], sg["resa"]) == (so["i"], so["resb"], so["resa"])
    for c in range(dim):
        assert np.array_equal(ug[c], uo[c]), c


@pytest.mark.parametrize("dim,depth,at", [(2, 2, (0, 3)), (2, 6, (17, 40)), (3, 4, (3, 4, 5)), (3, 5, (31, 0, 7))])
@pytest.mark.parametrize("cycles", [0, 1])
def test_viscosity_counts_nan(dim, depth, at, cycles):
    """The NaN values of every residual of a solve are counted, over all
    components and blocks: one NaN of the velocity against the residuals of
    the oracle's cycle."""
    print("case viscosity nan", dim, depth, cycles, flush=True)
    u, mu, rho = _problem(dim, depth, 5, True)
    u[1][at] = np.nan
    o = Viscosity(dim, depth)
    o.smoother = "rbgs"
    o.set_coefficients(mu, rho)
    res, _ = o.residual(u, u, 0.01)
    count = sum(int(np.isnan(x).sum()) for x in res)
    assert 0 < count < sum(x.size for x in res) or depth == 2
    if cycles:
        res, _ = o.residual(o.mg_cycle(u, res, 0.01, 4), u, 0.01)
        count += sum(int(np.isnan(x).sum()) for x in res)
    g = bmg.Grid(dim, depth)
    g.set_niter(cycles, cycles)
    with pytest.raises(bmg.BMGError, match=r"viscous residual is NaN \(%d values\)" % count) as e:
        g.viscosity([x.copy() for x in u], mu=mu, rho=rho, dt=0.01)
    assert e.value.code == 5
