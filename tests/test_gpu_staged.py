"""The LDS-staged bond-based step kernel (fd_staged.h) against the oracle at
the sizes and options where its paths part: slices just below, at and above
64 nodes, the short and the general form of the softening exponential
(critical-stretch factor 1, 10 and bonds that never break), no-fail nodes.

Bars, per node, relative to sum_j |F_ij| of the oracle's bond forces:
  FP64 exact: the same operations in the same order except exp, whose device
    and host values differ by at most 2 ulp in each bond force, and the
    rounding of the running sum that follows from it (half an ulp per
    addition, up to 24 slots): 2 + 12 ulp, taken as 16 x 2^-52;
  FP64: about 20 roundings of half an ulp per bond force (fused operations,
    the third-order reciprocal root below one ulp entering three times) and
    the same sum: 64 x 2^-52.
"""
import numpy as np
import pytest

from conftest import progress
from nlmech_amd import problems as pr
from nlmech_amd.capi import NLM_PREC_FP64, NLM_PREC_FP64_EXACT

pytestmark = pytest.mark.gpu

ULP = 2.0 ** -52
BAR = {NLM_PREC_FP64_EXACT: 16 * ULP, NLM_PREC_FP64: 64 * ULP}


def specimen(shape, **mat):
    p = pr.plate2d(shape[0], shape[1], 1e-3, 3, 1e-7, 1, notch_len=2e-3,
                   layers=0, jitter=0.05, **mat)
    return p


def force_of(p, precision, u, bonds=None):
    from nlmech_amd.engine import GpuFD
    with GpuFD(p, precision=precision) as g:
        g.set_state(u=u, f=np.zeros((p.n, 3)))
        g.compute_forces()
        return g.get_state()[2], g.get_bonds()


@pytest.mark.parametrize("precision", [NLM_PREC_FP64_EXACT, NLM_PREC_FP64],
                         ids=["exact", "fp64"])
@pytest.mark.parametrize("mat", [dict(), dict(check_sc=10.0),
                                 dict(irreversible=False)],
                         ids=["sc1", "sc10", "never"])
@pytest.mark.parametrize("shape", [(7, 9), (8, 8), (5, 13), (33, 31)],
                         ids=["63", "64", "65", "1023"])
def test_staged_force(oracle, precision, mat, shape):
    progress(f"[gpu] staged force {shape} {mat} mode {precision}")
    p = specimen(shape, **mat)
    if shape == (33, 31):  # some nodes that must not break
        p.interior = np.ones(p.n, np.uint8)
        p.interior[::7] = 0
    rng = np.random.default_rng(2)
    u = np.zeros((p.n, 3))
    # stretches up to several times the critical one
    u[:, :2] = rng.normal(scale=6e-6, size=(p.n, 2))
    o = oracle.OracleFD(p)
    o.set_state(u=u, v=np.zeros_like(u), f=np.zeros_like(u))
    b0 = o.get_bonds().sum()
    scale = o.force_abs_sum()
    o.compute_forces()
    f, bonds = force_of(p, precision, u)
    assert np.array_equal(bonds, o.get_bonds())
    if not mat:
        assert bonds.sum() > b0
    err = np.abs(f - o.get_state()[2]).max(1)
    assert np.all(err <= BAR[precision] * scale), (err / scale).max() / ULP
