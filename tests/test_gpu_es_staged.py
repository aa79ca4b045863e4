"""The staged state-based passes at the sizes where their tile and split
change (slices of 64 nodes: 400, 2500), in 2D and 3D, and on ragged and empty
rows: against the oracle, and bit for bit between the FP64 modes' tiles.

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


def plate(nx, ny, jitter=0.02):
    h = 1e-3
    x, vol = pr.grid2d(nx, ny, h, jitter, 3)
    v0 = np.zeros_like(x)
    v0[:, :2] = np.random.default_rng(1).normal(size=(x.shape[0], 2))
    return pr.Problem(name="plate", dim=2, x=x, vol=vol, horizon=3 * h, h=h,
                      dt=1e-7, nsteps=1, material=pr.es_material(dim=2),
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
