"""Conjugate gradients of the quasi-static solver: against a dense solve at
sizes around a slice and a 256-node block, on both tangents and both forms of
their products; a softening tangent (not positive) and a bond broken in one
direction only (not self-adjoint) end in BiCGSTAB's answer.

Bar: the solver stops at ||r|| <= 1e-10 ||b||; the true residual adds the
recursion's rounding, n iterations of a few ulp: 2e-10 for these sizes.
"""
import numpy as np
import pytest

from conftest import progress
from nlmech_amd import problems as pr
from nlmech_amd.capi import NLM_PREC_FP64_EXACT

pytestmark = pytest.mark.gpu


def dense(g, p):
    blk, dg = g.qs_tangent()
    rp, col = g.neighbors()
    A = np.zeros((2 * p.n, 2 * p.n))
    for i in range(p.n):
        A[2 * i:2 * i + 2, 2 * i:2 * i + 2] = dg[i]
        for k in range(rp[i], rp[i + 1]):
            j = col[k]
            A[2 * i:2 * i + 2, 2 * j:2 * j + 2] = blk[k]
    return A


def check(g, p, precond, max_iter=4000, tol=1e-10):
    fix = g.get_fixity()
    free = np.stack([fix & 1, fix >> 1 & 1], 1).reshape(-1) == 0
    b = np.zeros((p.n, 3))
    b[:, :2] = np.random.default_rng(4).standard_normal((p.n, 2))
    x, it, rr = g.qs_linear_solve(b, precond=precond, tol=tol,
                                  max_iter=max_iter)
    A = dense(g, p)[np.ix_(free, free)]
    xf = x[:, :2].reshape(-1)
    assert np.all(xf[~free] == 0)
    bf = b[:, :2].reshape(-1)[free]
    return it, rr, np.linalg.norm(A @ xf[free] - bf) / np.linalg.norm(bf)


@pytest.mark.parametrize("nx", [8, 9, 16, 17])
@pytest.mark.parametrize("tangent", [0, 1])
@pytest.mark.parametrize("precond", [0, 1])
def test_dense(nx, tangent, precond):
    from nlmech_amd.engine import GpuFD
    progress(f"[gpu] cg {nx} tangent {tangent} precond {precond}")
    p = pr.qs_plate(nx, jitter=0.05, layers=1)
    with GpuFD(p, precision=NLM_PREC_FP64_EXACT) as g:
        g.qs_assemble(tangent)
        for scalar in (True, False):
            g.qs_set_launch(True, scalar)
            it, rr, res = check(g, p, precond)
            assert 0 < it < 4000 and rr <= 1e-10 and res <= 2e-10


@pytest.mark.parametrize("kind", ["softening", "one_way"])
def test_falls_back(kind):
    from nlmech_amd.engine import GpuFD
    progress(f"[gpu] cg fallback {kind}")
    p = pr.qs_plate(12, jitter=0.05, layers=1, check_sc=10.0)
    with GpuFD(p, precision=NLM_PREC_FP64_EXACT) as g:
        if kind == "softening":
            # strains past the force's maximum on many bonds
            u = np.zeros((p.n, 3))
            u[:, :2] = np.random.default_rng(1).normal(scale=1.2e-5,
                                                       size=(p.n, 2))
            g.set_state(u=u)
        else:
            bonds = g.get_bonds()
            bonds[::5] = 1
            g.set_bonds(bonds)
        g.qs_assemble(0)
        if kind == "softening":
            w = np.linalg.eigvalsh(dense(g, p) * np.repeat(p.vol, 2)[:, None])
            assert w[0] < -1e-3 * w[-1]
        it, rr, res = check(g, p, 1, max_iter=20000, tol=1e-8)
        # (BiCGSTAB may stop at its limit on an indefinite tangent; what it
        # reports as solved is solved)
        assert rr > 1e-8 or res <= 1e-7
        if kind == "one_way":
            assert rr <= 1e-8


def setup_again(g, p):
    """Another problem set up on the context of g (which is used up)."""
    from nlmech_amd import capi
    from nlmech_amd.engine import GpuFD

    class Lib:  # hands out the context there is
        def __getattr__(self, name):
            return getattr(g.lib, name)

        def nlm_ctx_create(self, h, device):
            h._obj.value, g.ctx = g.ctx.value, None
            return 0

    load = capi.load
    capi.load = Lib
    try:
        return GpuFD(p, precision=NLM_PREC_FP64_EXACT)
    finally:
        capi.load = load


def solves(g, p):
    """Every solver's answers, on the model as it stands."""
    b = np.zeros((p.n, 3))
    b[:, :2] = np.random.default_rng(4).standard_normal((p.n, 2))
    g.qs_assemble(0)
    out = [g.qs_linear_solve(b, precond=pc, tol=1e-10, max_iter=300)
           for pc in (1, 1 | 16, 0)]
    st = g.qs_solve(2, lin_max_iter=600)
    out.append((st["linear_iters"], st["newton_iters"], st["residual"]))
    return [v for o in out for v in o] + list(g.get_state())


@pytest.mark.parametrize("kind", ["smaller", "more_nodes_fewer_bonds"])
def test_second_model_on_a_context(kind):
    """A context set up again gives a fresh context's answers, bit for bit: a
    smaller model (fewer partial sums), one with more nodes and slices but
    fewer bonds (buffers larger than the first model's although the tangent
    is smaller); what the first model left is not solved with."""
    from nlmech_amd.capi import NLM_QS_PRECOND_COARSE, NlmError
    from nlmech_amd.engine import GpuFD
    progress(f"[gpu] second model on a context: {kind}")
    assert NLM_QS_PRECOND_COARSE == 16
    if kind == "smaller":
        first, second = pr.qs_plate(40, jitter=0.05), pr.qs_plate(12)
    else:
        first = pr.qs_plate(20, ratio=6, jitter=0.05)
        second = pr.qs_plate(36, ratio=2, jitter=0.05)
    with GpuFD(second, precision=NLM_PREC_FP64_EXACT) as g:
        nnz2 = g.nnz
        want = solves(g, second)
    g = GpuFD(first, precision=NLM_PREC_FP64_EXACT)
    assert (g.nnz > nnz2) and (first.n > second.n) == (kind == "smaller")
    solves(g, first)
    g = setup_again(g, second)
    with pytest.raises(NlmError):
        g.qs_linear_solve(np.zeros((second.n, 3)))
    for a, b in zip(want, solves(g, second)):
        assert np.array_equal(a, b)
    g.close()
