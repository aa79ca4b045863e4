"""Node fields returned to the host: reordered on the device into the
context's staging (sizes around one workgroup, 2D and 3D, partial calls and
calls that follow a larger one)."""
import ctypes as C

import numpy as np
import pytest

from conftest import progress
from nlmech_amd import capi
from nlmech_amd import problems as pr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 1), (15, 17), (16, 16), (7, 5, 9)],
                         ids=["1", "255", "256", "3d"])
def test_state_round_trip(shape):
    from nlmech_amd.engine import GpuFD
    progress(f"[gpu] state round trip {shape}")
    h = 1e-3
    grid = pr.grid2d if len(shape) == 2 else pr.grid3d
    x, vol = grid(*shape, h, jitter=0.1, seed=3)
    p = pr.Problem(name="p", dim=len(shape), x=x, vol=vol, horizon=3 * h, h=h,
                   dt=1e-7, nsteps=1, material=pr.rnp_material(dim=len(shape)))
    rng = np.random.default_rng(1)
    want = [rng.normal(size=x.shape) for _ in range(3)]
    if len(shape) == 2:
        for a in want:
            a[:, 2] = 0.0
    with GpuFD(p) as g:
        g.set_state(*want)
        for _ in range(2):
            for a, b in zip(g.get_state(), want):
                assert np.array_equal(a, b)
        # one vector alone
        v = np.full(x.shape, 7.0)
        rc = g.lib.nlm_fd_get_state(g.ctx, None, capi.ptr(v, C.c_double), None)
        assert rc == 0 and np.array_equal(v, want[1])
        # the energy alone, from the same staging
        z, phi, e = g.postproc()
        e2 = np.full(p.n, 7.0)
        rc = g.lib.nlm_fd_postproc(g.ctx, None, None, capi.ptr(e2, C.c_double))
        assert rc == 0
        assert np.array_equal(e, e2, equal_nan=True)


def test_dilatation_alone():
    from nlmech_amd.engine import GpuFD
    progress("[gpu] dilatation alone")
    p = pr.cube3d(7, 1e-3, 3, 1e-8, 1)
    with GpuFD(p) as g:
        g.init()
        g.step(3)
        th, mw = g.node_fields()
        t2 = np.full(p.n, 7.0)
        rc = g.lib.nlm_fd_get_node_fields(g.ctx, capi.ptr(t2, C.c_double), None)
        assert rc == 0 and np.array_equal(th, t2) and np.all(mw > 0)
