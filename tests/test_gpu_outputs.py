"""Node fields returned to the host: reordered on the device into the
context's staging (sizes around one workgroup, 2D and 3D, partial calls and
calls that follow a larger one; 1.9e6 nodes, beyond its 128 MiB with three
vectors, and 5.8e6, beyond it with one)."""
import ctypes as C

import numpy as np
import pytest

from conftest import progress
from nlmech_amd import capi
from nlmech_amd import problems as pr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 1), (15, 17), (16, 16), (7, 5, 9),
                                   (1400, 1350), (2401, 2400)],
                         ids=["1", "255", "256", "3d", "1890000", "5762400"])
def test_state_round_trip(shape):
    from nlmech_amd.engine import GpuFD
    progress(f"[gpu] state round trip {shape}")
    h = 1e-3
    grid = pr.grid2d if len(shape) == 2 else pr.grid3d
    x, vol = grid(*shape, h, jitter=0.1, seed=3)
    ratio = 3 if x.shape[0] < 10 ** 6 else 1.2  # (4 neighbors will do)
    p = pr.Problem(name="p", dim=len(shape), x=x, vol=vol, horizon=ratio * h,
                   h=h,
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


def test_node_fields_of_a_large_model():
    """9e6 nodes: two fields beyond the staging's 128 MiB."""
    from nlmech_amd.engine import GpuFD
    progress("[gpu] node fields of a large model")
    h = 1e-3
    x, vol = pr.grid2d(3001, 2999, h, jitter=0.0)
    vol *= 1.0 + np.random.default_rng(1).random(x.shape[0])
    p = pr.Problem(name="p", dim=2, x=x, vol=vol, horizon=1.2 * h, h=h,
                   dt=1e-7, nsteps=1, material=pr.es_material(dim=2))
    with GpuFD(p) as g:
        th, mw = g.node_fields()
    # m_i = sum_j |X|^2 c V_j over the four neighbors at a distance h
    w = np.pad(vol.reshape(2999, 3001), 1)
    s = w[:-2, 1:-1] + w[2:, 1:-1] + w[1:-1, :-2] + w[1:-1, 2:]
    ratio = mw.reshape(2999, 3001) / s
    assert np.all(th == 0.0)
    assert np.allclose(ratio, ratio[0, 0], rtol=1e-9)


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


def test_time_of_small_outputs():
    """Three vectors of 810 nodes cost little more than one (a copy each to
    pageable memory: more than twice)."""
    import time

    from nlmech_amd.engine import GpuFD
    progress("[gpu] time of small outputs")
    p = pr.plate2d(30, 27, 1e-3, 3, 1e-7, 1)
    us = []
    with GpuFD(p) as g:
        out = [np.zeros((p.n, 3)) for _ in range(3)]
        ptrs = [o.ctypes.data_as(C.POINTER(C.c_double)) for o in out]
        for args in ([ptrs[0], None, None], ptrs):
            best = 1e9
            for _ in range(200):
                t = time.perf_counter()
                g._call("nlm_fd_get_state", *args)
                best = min(best, time.perf_counter() - t)
            us.append(1e6 * best)
    progress(f"[gpu]   {us[0]:.0f} {us[1]:.0f} us")
    assert us[1] <= 1.8 * us[0]
