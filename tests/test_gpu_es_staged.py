"""The staged state-based passes at the sizes where their tile and split
change (slices of 64 nodes: 400, 2500), in 2D and 3D, on ragged and empty
rows and over mesh sizes: against the oracle, and bit for bit between the FP64
modes' tiles.

Bars, relative to the displacement norm.  Exact mode: the oracle's operations
in its order, each node's update rounded alike: 1e-13.  FP64: the oracle's
extension |Y| - |X| cancels (about 2^-53 |X| in an extension of 1e-7 |X| here,
1e-9; the steps' share of the displacement makes it smaller).  FP32-force:
1e-5, that mode's target.
"""
import numpy as np
import pytest

from conftest import progress
from nlmech_amd import problems as pr
from nlmech_amd.capi import (NLM_PREC_FP32_FORCE, NLM_PREC_FP64,
                             NLM_PREC_FP64_EXACT)

pytestmark = pytest.mark.gpu
MODES = [NLM_PREC_FP64_EXACT, NLM_PREC_FP64, NLM_PREC_FP32_FORCE]
BAR = {NLM_PREC_FP64_EXACT: 1e-13, NLM_PREC_FP64: 1e-9,
       NLM_PREC_FP32_FORCE: 1e-5}


def plate(nx, ny, jitter=0.02, h=1e-3):
    x, vol = pr.grid2d(nx, ny, h, jitter, 3)
    v0 = np.zeros_like(x)
    v0[:, :2] = np.random.default_rng(1).normal(size=(x.shape[0], 2))
    return pr.Problem(name="plate", dim=2, x=x, vol=vol, horizon=3 * h, h=h,
                      dt=1e-4 * h, nsteps=1, material=pr.es_material(dim=2),
                      v0=v0)


def run(p, mode, steps, tile=None):
    from nlmech_amd.engine import GpuFD
    with GpuFD(p, precision=mode) as g:
        if tile:
            g.set_tile(tile)
        g.init()
        g.step(steps)
        return g.get_state() + (g.node_fields()[0], g.get_bonds())


def check(p, mode, steps, oracle):
    o = oracle.OracleES(p)
    o.init()
    o.step(steps)
    got = run(p, mode, steps)
    ref = o.get_state()[0]
    assert np.linalg.norm(got[0] - ref) <= BAR[mode] * np.linalg.norm(ref)
    if mode != NLM_PREC_FP32_FORCE:
        assert np.array_equal(got[4], o.get_bonds())
    return got


@pytest.mark.parametrize("mode", MODES, ids=["exact", "fp64", "fp32"])
@pytest.mark.parametrize("shape", [(8, 8), (5, 13), (160, 159), (161, 160),
                                   (400, 399), (401, 400)],
                         ids=["64", "65", "398", "403", "2494", "2507"])
def test_plate(oracle, mode, shape):
    progress(f"[gpu] staged state-based plate {shape} mode {mode}")
    got = check(plate(*shape), mode, 4, oracle)
    assert shape[0] < 100 or got[4].sum() > 0


@pytest.mark.parametrize("mode", MODES, ids=["exact", "fp64", "fp32"])
@pytest.mark.parametrize("shape", [(4, 4, 4), (29, 29, 30), (30, 29, 30),
                                   (54, 54, 54), (54, 54, 55)],
                         ids=["64", "395", "408", "2461", "2506"])
def test_block(oracle, mode, shape):
    progress(f"[gpu] staged state-based block {shape} mode {mode}")
    p = pr.cube3d(shape[0], 1e-3, 3, 1e-7, 1, ny=shape[1], nz=shape[2],
                  sigma_v=1.0, jitter=0.02)
    got = check(p, mode, 3, oracle)
    if mode != NLM_PREC_FP32_FORCE and shape[0] in (29, 54):
        for tile in (128, 256, 512):
            for a, b in zip(got, run(p, mode, 3, tile)):
                assert np.array_equal(a, b), tile


@pytest.mark.parametrize("mode", MODES, ids=["exact", "fp64", "fp32"])
def test_ragged_and_empty_rows(oracle, mode):
    progress(f"[gpu] staged state-based ragged rows mode {mode}")
    p = plate(30, 30, jitter=0.3)
    rng = np.random.default_rng(5)
    extra = np.zeros((100, 3))
    extra[:, :2] = 0.010 + 0.004 * rng.random((100, 2))  # a dense cluster
    # pairs of nodes far from the plate, one bond each
    far = np.zeros((128, 3))
    far[:, 0] = 1.0 + np.repeat(np.arange(64), 2) * 0.1
    far[1::2, 0] += 1e-3
    x = np.concatenate([p.x, extra, far])
    v0 = np.concatenate([p.v0, np.zeros((228, 3))])
    p = pr.with_(p, x=x, v0=v0, vol=np.concatenate([p.vol, np.full(228, 5e-7)]))
    check(p, mode, 5, oracle)


@pytest.mark.parametrize("mode", MODES, ids=["exact", "fp64", "fp32"])
@pytest.mark.parametrize("dim", [1, 2, 3])
def test_nodes_without_neighbors(oracle, mode, dim):
    """Nodes with no neighbor at all (their weighted volume is 0, 1/m infinite)
    in slices with nodes that have some: they keep their velocity, the others
    the oracle's motion."""
    progress(f"[gpu] staged state-based nodes without neighbors {dim}D {mode}")
    h = 1e-3
    if dim == 3:
        x, vol = pr.grid3d(6, 5, 7, h, jitter=0.05, seed=3)
    else:
        x, vol = pr.grid2d(21, 1 if dim == 1 else 10, h, 0.05, 3)
    # along a line far away: two bonded nodes, one alone, two bonded, ...
    far = np.zeros((150, 3))
    far[:, 0] = 1.0 + np.arange(150) // 3 * 0.1 + np.tile([0., h, 0.05], 50)
    x = np.concatenate([x, far])
    vol = np.concatenate([vol, np.full(150, h ** dim)])
    if dim == 1:
        x[:, 1] = 0.
    v0 = np.zeros_like(x)
    v0[:, :dim] = np.random.default_rng(1).normal(size=(x.shape[0], dim))
    mat = pr.es_material(dim=dim, E=4e9 if dim == 1 else -1.0)
    p = pr.Problem(name="alone", dim=dim, x=x, vol=vol, horizon=3 * h, h=h,
                   dt=1e-7, nsteps=1, material=mat, v0=v0)
    got = check(p, mode, 5, oracle)
    alone = x.shape[0] - 150 + np.arange(2, 150, 3)
    assert np.all(np.isfinite(got[0])) and np.all(got[2][alone] == 0.)
    assert np.allclose(got[0][alone], 5 * p.dt * v0[alone], rtol=1e-14)


@pytest.mark.parametrize("mode", MODES, ids=["exact", "fp64", "fp32"])
@pytest.mark.parametrize("h", [1.0, 1e-5, 1e-6])
def test_mesh_size(oracle, mode, h):
    """The force coefficients go with h^-4: the same strains at other mesh
    sizes, rows of odd length included."""
    progress(f"[gpu] staged state-based mesh size {h} mode {mode}")
    check(plate(23, 17, h=h), mode, 4, oracle)
    p = pr.cube3d(9, h, 3, 1e-4 * h, 1, ny=8, nz=7, sigma_v=1.0, jitter=0.02)
    check(p, mode, 3, oracle)


@pytest.mark.parametrize("mode", MODES, ids=["exact", "fp64", "fp32"])
@pytest.mark.parametrize("shape", [(5, 13), (161, 160), (9, 8, 7)],
                         ids=["65", "25760", "3d"])
def test_force(oracle, mode, shape):
    """The force itself at strains of about 1e-3, without broken bonds.  Exact:
    the sum's order and operations, a few ulp from the IEEE root of a sum of
    another length: 1e-13.  FP64: the oracle's extension cancels, 2^-53 |X| in
    1e-3 |X|, a few of them: 1e-11.  FP32-force: about 25 roundings of 2^-24
    a bond: 2e-6."""
    from nlmech_amd.engine import GpuFD
    progress(f"[gpu] staged state-based force {shape} mode {mode}")
    h = 1e-3
    if len(shape) == 2:
        p = pr.with_(plate(*shape), material=pr.es_material(dim=2, sc=-1.0))
    else:
        p = pr.cube3d(shape[0], h, 3, 1e-7, 1, ny=shape[1], nz=shape[2],
                      jitter=0.02, sc=-1.0)
    u = np.zeros((p.n, 3))
    d = len(shape)
    u[:, :d] = np.random.default_rng(6).normal(scale=1e-6, size=(p.n, d))
    o = oracle.OracleES(p)
    o.set_state(u=u, v=np.zeros_like(u), f=np.zeros_like(u))
    o.compute_forces()
    ref = o.get_state()[2]
    with GpuFD(p, precision=mode) as g:
        g.set_state(u=u, v=np.zeros_like(u), f=np.zeros_like(u))
        g.compute_forces()
        f = g.get_state()[2]
    bar = {NLM_PREC_FP64_EXACT: 1e-13, NLM_PREC_FP64: 1e-11,
           NLM_PREC_FP32_FORCE: 2e-6}[mode]
    assert np.linalg.norm(f - ref) <= bar * np.linalg.norm(ref)


@pytest.mark.parametrize("dim", [2, 3])
def test_coincident_nodes(oracle, dim):
    """Exact mode, no breaking: two nodes at one place that move apart.  The
    bond's reference length 0 is exact, its force that of the oracle."""
    from nlmech_amd.engine import GpuFD
    progress(f"[gpu] staged state-based coincident nodes {dim}D")
    h = 1e-3
    if dim == 2:
        p = pr.with_(plate(9, 8), material=pr.es_material(dim=2, sc=-1.0))
    else:
        p = pr.cube3d(7, h, 3, 1e-7, 1, ny=6, nz=5, jitter=0.02, sc=-1.0)
    p.x[31] = p.x[30]
    u = np.zeros((p.n, 3))
    u[:, :dim] = np.random.default_rng(6).normal(scale=1e-6, size=(p.n, dim))
    o = oracle.OracleES(p)
    o.set_state(u=u, v=np.zeros_like(u), f=np.zeros_like(u))
    o.compute_forces()
    ref = o.get_state()[2]
    assert np.all(np.isfinite(ref))
    with GpuFD(p, precision=NLM_PREC_FP64_EXACT) as g:
        g.set_state(u=u, v=np.zeros_like(u), f=np.zeros_like(u))
        g.compute_forces()
        f = g.get_state()[2]
    assert np.linalg.norm(f - ref) <= 1e-13 * np.linalg.norm(ref)


def test_time_of_uneven_halos():
    """3D FP64: a block that the Morton order cuts unevenly (70^3) costs no
    more a node than one it cuts evenly, 64^3 (on tiles of 256 nodes, one a
    CU: 1.33 times), and takes the same steps at every tile."""
    from nlmech_amd.engine import GpuFD
    progress("[gpu] time of uneven halos")
    us, state = [], []
    for n in (64, 70):
        p = pr.cube3d(n, 1e-3, 3, 1e-7, 1, jitter=0.0, sigma_v=1e-3)
        with GpuFD(p, precision=NLM_PREC_FP64) as g:
            g.init()
            us.append(min(g.timed_steps(21)[1] for _ in range(8)) * 1e6 / p.n)
    for tile in (None, 128, 256):
        state.append(run(p, NLM_PREC_FP64, 3, tile))
    progress(f"[gpu]   {us[0]:.3f} {us[1]:.3f} ns a node")
    assert us[1] <= 1.2 * us[0]
    for other in state[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(state[0], other))


def test_short_rows_are_not_split():
    """3D FP32-force above 2500 slices: rows of 25 bonds keep one wavefront (two
    cost more than they gain), rows of 81 have two."""
    from nlmech_amd.engine import GpuFD
    progress("[gpu] short rows are not split")
    for ratio, parts in ((2, 1), (3, 2)):
        p = pr.cube3d(56, 1e-3, ratio, 1e-7, 1, jitter=0.0)
        with GpuFD(p, precision=NLM_PREC_FP32_FORCE) as g:
            assert g.get_tile() == (256, parts)
