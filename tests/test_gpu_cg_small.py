"""Conjugate gradients in two kernels an iteration (small lowest-order W0 problems) against the form over the
colour-ordered apply in separate kernels, whose sums run in another order: the same iterates up to rounding
after a fixed number of iterations (the recurrences' error grows by the condition of B B^T + 0.1 I elements, below
100: 1e4 eps of the norm), counts within one to a tolerance, and the ends of a solve.  Sizes of one block, several, a
partial one, both sides of the loads ahead (256 and 512 blocks of 256 dofs, FP64 and FP32) and of the largest it
takes (512 and 768 blocks), and beyond."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _cg(hip, op, b, P, form, **kw):
    hip.set_apply_form(form)
    try:
        x = hip.FieldVector(op.fs_to, P)
        x.set_scalar(0.0)
        res = hip.ConjugateGradient(op, hip.DiagonalPreconditioner.from_operator(op), **kw).apply(x, b)
        return res, x.export_field()
    finally:
        hip.set_apply_form(1)


@pytest.mark.parametrize("prec", ["R64", "R32"])
@pytest.mark.parametrize("n,nl", [(2, 2), (3, 4), (5, 7), (12, 20), (20, 26), (20, 27), (24, 36), (24, 37),
                                  (28, 40), (28, 41), (25, 48), (25, 49), (32, 60)])
def test_two_kernel_iteration(hip, n, nl, prec):
    P, eps = (hip.R64, np.finfo(np.float64).eps) if prec == "R64" else (hip.R32, np.finfo(np.float32).eps)
    fs = hip.FunctionSpace.cubedsphere(n, nl)
    op = hip.LmaOperator(fs).generate_spd(n + nl)
    op = op if P == hip.R64 else op.convert(P)
    b = hip.FieldVector(fs, P).fill_uniform(n, 3)
    for iters in (1, 2, 6):
        kw = dict(r_tol=1e-30, a_tol=0.0, max_iter=iters, monitor_convergence=False, check_every=4)
        (r1, x1), (r0, x0) = (_cg(hip, op, b, P, form, **kw) for form in (1, 0))
        assert r1.iterations == r0.iterations == iters
        assert np.linalg.norm(x1 - x0) <= 1e4 * eps * np.linalg.norm(x0)
    kw = dict(r_tol=1e-8 if P == hip.R64 else 1e-4, a_tol=0.0, max_iter=100, check_every=8)
    (r1, x1), (r0, x0) = (_cg(hip, op, b, P, form, **kw) for form in (1, 0))
    assert r1.status == r0.status == 0 and abs(r1.iterations - r0.iterations) <= 1


def test_ends_of_a_solve(hip):
    fs = hip.FunctionSpace.cubedsphere(6, 9)
    op = hip.LmaOperator(fs).generate_spd(1)
    zero = hip.FieldVector(fs)
    zero.set_scalar(0.0)
    res, x = _cg(hip, op, zero, hip.R64, 1, r_tol=1e-10, a_tol=0.0, max_iter=50)
    assert res.status == 0 and res.iterations == 0 and not x.any()
    bad = hip.FieldVector(fs).import_field(np.full(fs.undf, np.nan))
    with pytest.raises(hip.LfricError):
        _cg(hip, op, bad, hip.R64, 1, r_tol=1e-10, a_tol=0.0, max_iter=50)
    b = hip.FieldVector(fs).fill_uniform(1, 3)
    res, _ = _cg(hip, op, b, hip.R64, 1, r_tol=1e-12, a_tol=0.0, max_iter=3)
    assert res.status == 1 and res.iterations == 3


@pytest.mark.parametrize("prec", ["R64", "R32"])
@pytest.mark.parametrize("n,nl,order", [(2, 2, 0), (12, 20, 0), (25, 48, 0), (48, 60, 0), (6, 5, 1)])
def test_breakdown_leaves_x_as_it_was(hip, n, nl, order, prec):
    """A = 0: p.(A p) is 0 in the first iteration, which ends the solve before x is stepped, in the two-kernel
    iteration and (beyond 512 or 768 blocks, order 1) in the separate kernels."""
    P = getattr(hip, prec)
    fs = hip.FunctionSpace.cubedsphere(n, nl, hip.W0, order)
    op = hip.LmaOperator(fs, precision=P)
    b, x = hip.FieldVector(fs, P).fill_uniform(n, 3), hip.FieldVector(fs, P).fill_uniform(nl, 4)
    before = x.export_raw()
    cg = hip.ConjugateGradient(op, hip.NullPreconditioner(), 1e-8, 0.0, 50)
    with pytest.raises(hip.LfricError):
        cg.apply(x, b)
    assert cg.result.status == 3 and cg.result.iterations == 0
    np.testing.assert_array_equal(x.export_raw(), before)
