"""Conjugate gradients of the quasi-static solver: against a dense solve at
sizes around a slice and a 256-node block, on both tangents and both forms of
their products; a softening tangent (not positive) and bonds broken in one
direction only (not self-adjoint) end in BiCGSTAB's answer; the iteration
limit; a context set up for a second model.

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


def cg_end(A, W, b, tol, limit):
    """How conjugate gradients in the inner product W, point Jacobi, end:
    (iterations, True where they converge)."""
    z = b / np.diag(A)
    r, p, rho = b.copy(), z.copy(), W @ (b * z)
    for it in range(limit):
        if np.linalg.norm(r) <= tol * np.linalg.norm(b):
            return it, True
        q = A @ p
        pq = W @ (p * q)
        if not (rho > 0 and pq > 0):
            return it, False
        r -= rho / pq * q
        z = r / np.diag(A)
        rho, beta = W @ (r * z), rho
        p = z + rho / beta * p
    return limit, False


@pytest.mark.parametrize("kind", ["softening", "one_way"])
def test_falls_back(kind):
    """Where conjugate gradients end without convergence (restated here), the
    answer is BiCGSTAB's."""
    from nlmech_amd.engine import GpuFD
    progress(f"[gpu] cg fallback {kind}")
    p = pr.qs_plate(12, jitter=0.05, layers=1, check_sc=10.0)
    limit = 2000
    with GpuFD(p, precision=NLM_PREC_FP64_EXACT) as g:
        if kind == "softening":
            # strains past the force's maximum on some bonds
            u = np.zeros((p.n, 3))
            u[:, :2] = np.random.default_rng(1).normal(scale=3e-6,
                                                       size=(p.n, 2))
            g.set_state(u=u)
        else:
            bonds = g.get_bonds()
            bonds[::5] = 1
            g.set_bonds(bonds)
        g.qs_assemble(0)
        fix = g.get_fixity()
        free = np.stack([fix & 1, fix >> 1 & 1], 1).reshape(-1) == 0
        A = dense(g, p)[np.ix_(free, free)]
        W = np.repeat(p.vol, 2)[free]
        b = np.random.default_rng(4).standard_normal((p.n, 2)).reshape(-1)
        ends, conv = cg_end(A, W, b[free], 1e-8, limit)
        assert not conv and (ends == limit) == (kind == "one_way")
        if kind == "softening":
            w = np.linalg.eigvalsh(dense(g, p) * np.repeat(p.vol, 2)[:, None])
            assert w[0] < -1e-3 * w[-1]
        it, rr, res = check(g, p, 1, max_iter=limit, tol=1e-8)
        assert 0 < it < limit and rr <= 1e-8 and res <= 2e-8


def test_converged_at_the_limit():
    """Convergence in the last iteration allowed is convergence; one iteration
    less goes to BiCGSTAB."""
    from nlmech_amd.engine import GpuFD
    progress("[gpu] cg converged at the iteration limit")
    p = pr.qs_plate(17, jitter=0.05, layers=1)
    b = np.zeros((p.n, 3))
    b[:, :2] = np.random.default_rng(4).standard_normal((p.n, 2))
    with GpuFD(p, precision=NLM_PREC_FP64_EXACT) as g:
        g.qs_assemble(0)
        for graph in (True, False):
            g.qs_set_graph(graph)
            x, it, rr = g.qs_linear_solve(b, tol=1e-10)
            x1, it1, rr1 = g.qs_linear_solve(b, tol=1e-10, max_iter=it)
            assert it1 == it and rr1 == rr and np.array_equal(x, x1)
            _, it2, rr2 = g.qs_linear_solve(b, tol=1e-10, max_iter=it - 1)
            assert it2 < it and rr2 <= 1e-10


def test_failure_is_remembered_in_a_load_step():
    """A limit that neither method reaches convergence in: conjugate gradients
    are tried once a load step, BiCGSTAB in every Newton iteration."""
    from nlmech_amd.engine import GpuFD
    progress("[gpu] cg failure within a load step")
    p = pr.qs_plate(40, jitter=0.05, pull=2e-5)
    with GpuFD(p, precision=NLM_PREC_FP64_EXACT) as g:
        st = g.qs_solve(2, lin_max_iter=60)
    newton = st["newton_iters"]
    assert newton >= 4 and st["linear_failures"] == newton
    assert st["linear_iters"] == 60 * (2 + newton)


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
