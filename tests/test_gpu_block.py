"""The red-black kernels that keep a level or its tiles on chip (k_coarse_rb,
k_rb_tile) against the in-place kernel and the coarse kernel that work from
memory (BMG_RB_KERNEL=inplace), bit for bit in both precisions: residual
norms, the solution, and res and da of every level.  The in-place kernels
equal the oracle's sweeps (test_gpu_parity.py)."""
import numpy as np
import pytest

import basilisk_amd as bmg
from tests import cases

pytestmark = pytest.mark.gpu

D, N, S, P = cases.BC_DIRICHLET, cases.BC_NEUMANN, cases.BC_SYMMETRY, cases.BC_PERIODIC
BOXES = {
    2: {"walls": [D, N, S, D], "periodic": [P] * 4, "channel": [P, P, D, S]},
    3: {"walls": [D, N, S, D, N, D], "periodic": [P] * 6, "channel": [D, N, P, P, S, D]},
}


def _grid(dim, depth, box, coef, precision, kind="multigrid"):
    g = bmg.Grid(dim, depth, precision=precision, smoother="rbgs", kind=kind)
    n = 1 << depth
    lam = np.random.default_rng(8).uniform(-2.0, -0.5, (n,) * dim) if "lam" in coef else -0.7
    cases.random_problem(g, 31 + depth, lam=lam, alpha="alpha" in coef, bcs=BOXES[dim][box])
    g.restriction_alpha_lambda()
    return g


def _same(dim, depth, box, coef, precision, nrelax, minlevels, monkeypatch, kind="multigrid"):
    print("block", dim, depth, box, coef, precision, nrelax, minlevels, kind, flush=True)
    monkeypatch.setenv("BMG_RB_KERNEL", "inplace")
    one = _grid(dim, depth, box, coef, precision, kind)
    monkeypatch.delenv("BMG_RB_KERNEL")
    two = _grid(dim, depth, box, coef, precision, kind)
    assert one.residual() == two.residual()
    for m in minlevels:
        for g in (one, two):
            g.mg_cycle(nrelax, m)
        for l in range(m, depth + 1):
            assert np.array_equal(one.get_da(l), two.get_da(l)), l
            if l < depth:
                assert np.array_equal(one.get_res(l), two.get_res(l)), l
        assert one.residual() == two.residual()
    assert np.array_equal(one.get_a(), two.get_a())


# every level size up to one where each kernel variant has whole, cut and
# wrapped tiles: 2D regions of 32, 48 and 64 cells per side, 3D of 16
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("box", ["walls", "periodic", "channel"])
@pytest.mark.parametrize("dim,depth", [(2, 1), (2, 4), (2, 6), (2, 8), (2, 9), (2, 10), (3, 1), (3, 2), (3, 4), (3, 5),
                                       (3, 6)])
def test_levels_bitexact(dim, depth, box, precision, monkeypatch):
    _same(dim, depth, box, "alpha lam", precision, 4, (0, 1), monkeypatch)


# levels of several hundred tiles of 64^2 cells
@pytest.mark.parametrize("depth,box,coef,precision", [(11, "walls", "alpha", "fp64"), (11, "periodic", "lam", "mixed"),
                                                      (11, "channel", "alpha lam", "fp64"),
                                                      (12, "channel", "alpha", "mixed")])
def test_large_2d_levels_bitexact(depth, box, coef, precision, monkeypatch):
    _same(2, depth, box, coef, precision, 4, (1,), monkeypatch)


@pytest.mark.parametrize("coef", ["alpha", "lam", ""])
@pytest.mark.parametrize("dim,depth", [(2, 7), (3, 5)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_coefficients_bitexact(dim, depth, coef, precision, monkeypatch):
    _same(dim, depth, "channel", coef, precision, 3, (0, 1), monkeypatch)


@pytest.mark.parametrize("nrelax", [0, 1, 2, 3, 5, 9])
@pytest.mark.parametrize("dim,depth", [(2, 7), (3, 5)])
def test_sweep_counts_and_coarsest_levels(dim, depth, nrelax, monkeypatch):
    _same(dim, depth, "walls", "alpha", "fp64", nrelax, (0, depth - 2, depth), monkeypatch)


@pytest.mark.parametrize("dim,depth", [(2, 7), (3, 5)])
def test_tree_corner_rule(dim, depth, monkeypatch):
    _same(dim, depth, "walls", "alpha", "mixed", 4, (0,), monkeypatch, kind="tree")


def test_affine_side_without_reflection(monkeypatch):
    """sigma 0: the ghost of the correction is zero."""
    out = []
    for kernel in ("inplace", None):
        if kernel:
            monkeypatch.setenv("BMG_RB_KERNEL", kernel)
        else:
            monkeypatch.delenv("BMG_RB_KERNEL")
        g = _grid(2, 7, "walls", "alpha", "fp64")
        g.set_bc_affine(bmg.TOP, 0, np.linspace(0.0, 1.0, 128))
        g.set_a(np.zeros(g.shape()))
        out.append((g.poisson(tolerance=1e-8), g.get_a()))
    assert out[0][0] == out[1][0] and np.array_equal(out[0][1], out[1][1])


def test_graph_replays_of_a_correcting_cycle():
    """mg_cycle's last launch adds the correction itself: replays of its
    graph, with eager work between them, equal launches without graphs."""
    print("block replays", flush=True)
    grids = []
    for graphs in ("0", "1"):
        import os
        os.environ["BMG_GRAPHS"] = graphs
        try:
            grids.append(_grid(2, 7, "walls", "alpha lam", "fp64"))
        finally:
            del os.environ["BMG_GRAPHS"]
    for _ in range(4):
        r = [g.residual() for g in grids]
        assert r[0] == r[1]
        for g in grids:
            g.mg_cycle(3, 1)
            g.synchronize()
    assert np.array_equal(grids[0].get_a(), grids[1].get_a())


def _coarse_launches(dim, depth, top, nrelax):
    """launches of the coarse levels of a cycle: one workgroup for the levels
    up to top, then per level a launch for every sweep (4^dim and 8^dim cells)
    or for up to 4 (2D) or 2 (3D) sweeps"""
    n = 1
    for l in range(top + 1, depth):
        n += nrelax if l < 4 else -(-nrelax // (4 if dim == 2 else 2))
    return n


@pytest.mark.parametrize("dim,depth,box,coef,precision,default,top",
                         [(2, 7, "walls", "alpha", "fp64", 5, t) for t in (0, 2, 6)]
                         + [(2, 7, "channel", "lam", "mixed", 5, 4), (2, 7, "periodic", "alpha", "fp64", 5, 2)]
                         + [(3, 5, "walls", "alpha", "fp64", 3, t) for t in (1, 4)]
                         + [(3, 5, "walls", "", "fp64", 4, 3), (3, 5, "channel", "alpha", "mixed", 4, 2),
                            (3, 5, "periodic", "", "mixed", 4, 2)])
def test_coarse_top_switch(dim, depth, box, coef, precision, default, top, monkeypatch):
    """BMG_COARSE_TOP moves the level up to which a cycle runs in one
    workgroup, also beyond what k_coarse_rb takes (tiles then run levels down
    to 16 cells across, smaller than their region), with the same values."""
    print("block coarse top", dim, depth, box, coef, precision, top, flush=True)
    out = []
    for t in (None, top):
        monkeypatch.delenv("BMG_COARSE_TOP", raising=False)
        if t is not None:
            monkeypatch.setenv("BMG_COARSE_TOP", str(t))
        g = _grid(dim, depth, box, coef, precision)
        g.residual()
        g.mg_cycle(4, 0)
        g.profile(True)
        g.mg_cycle(4, 0)
        g.synchronize()
        assert g.profile_get("relax_coarse")[1] == _coarse_launches(dim, depth, default if t is None else t, 4)
        out.append((g.residual(), g.get_a()))
    assert out[0][0] == out[1][0] and np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("threads", [64, 320])
def test_coarse_block_switch(threads, monkeypatch):
    """BMG_COARSE_BLOCK takes the coarse kernel whose threads it sets: on a
    grid that ends there the correction is then a launch of its own."""
    print("block coarse threads", threads, flush=True)
    out = []
    for t in (None, threads):
        if t is not None:
            monkeypatch.setenv("BMG_COARSE_BLOCK", str(t))
        g = _grid(2, 5, "channel", "alpha lam", "fp64")
        g.residual()
        g.profile(True)
        g.mg_cycle(3, 0)
        g.synchronize()
        assert g.profile_get("correction")[1] == (0 if t is None else 1)
        out.append((g.residual(), g.get_a()))
    assert out[0][0] == out[1][0] and np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("dim,depth,kernel,kind,launches",
                         [(2, 7, None, "relax_fine_tile", 2), (3, 5, None, "relax_fine_tile", 3),
                          (2, 7, "inplace", "relax_fine", 5), (3, 7, None, "relax_fine", 5)])
def test_profile_kinds_of_the_finest_level(dim, depth, kernel, kind, launches, monkeypatch):
    """relax_fine counts launches of one sweep; tiles, which run several and
    interpolate and correct as well, are a kind of their own."""
    print("block profile", dim, depth, kernel, flush=True)
    if kernel:
        monkeypatch.setenv("BMG_RB_KERNEL", kernel)
    g = _grid(dim, depth, "walls", "", "fp64")
    g.residual()
    g.profile(True)
    g.mg_cycle(5, 0)
    g.synchronize()
    count = {k: g.profile_get(k)[1] for k in bmg.PROFILE_KINDS}
    fine = {k: count[k] for k in ("relax_fine", "relax_fine2", "relax_fine_tile")}
    assert fine == dict.fromkeys(fine, 0) | {kind: launches}
    assert count["correction"] == (0 if kind == "relax_fine_tile" else 1)
