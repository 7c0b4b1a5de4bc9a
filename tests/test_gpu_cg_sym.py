"""Conjugate gradients over the symmetric-packed copy, whose iteration forms p.(A p) from the units and
updates the residual where it gathers A p, against the same solve over the element layout: the operators are
the same and only the order of a sum changes, so the iteration counts agree within one and the solutions to
what a residual of r_tol leaves (condition of B B^T + 0.1 I elements below 100: 100 r_tol).  Sizes with one
block and several, partial blocks and wavefronts; and the ends of a solve: no iteration (b = 0 and an exact
initial guess), the iteration limit, monitoring off."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["R64", "R32"])
@pytest.mark.parametrize("n,nl", [(2, 2), (3, 2), (5, 7), (4, 62), (24, 30)])
def test_cg_over_the_symmetric_copy(hip, n, nl, prec):
    P = getattr(hip, prec)
    r_tol = 1e-10 if prec == "R64" else 1e-5
    fs = hip.FunctionSpace.cubedsphere(n, nl)
    op64 = hip.LmaOperator(fs).generate_spd(n)
    b = hip.FieldVector(fs, P).fill_uniform(n, 3)
    out = []
    for copy in (False, True):
        op = op64.convert(P)
        if copy:
            op.prepare_symmetric()
        x = hip.FieldVector(fs, P)
        x.set_scalar(0.0)
        res = hip.ConjugateGradient(op, hip.DiagonalPreconditioner.from_operator(op), r_tol, 0.0, 200).apply(x, b)
        assert res.status == 0
        out.append((res.iterations, x.export_field()))
    (i0, x0), (i1, x1) = out
    assert abs(i0 - i1) <= 1
    assert np.linalg.norm(x1 - x0) <= 100 * r_tol * np.linalg.norm(x0)


def test_ends_of_a_solve(hip):
    fs = hip.FunctionSpace.cubedsphere(6, 9)
    op = hip.LmaOperator(fs).generate_spd(1)
    plain = op.convert(hip.R64)
    op.prepare_symmetric()
    prec = hip.DiagonalPreconditioner.from_operator(op)
    b, x = hip.FieldVector(fs).fill_uniform(2, 3), hip.FieldVector(fs)
    zero = hip.FieldVector(fs)
    zero.set_scalar(0.0)
    x.set_scalar(0.0)
    res = hip.ConjugateGradient(op, prec, 1e-10, 0.0, 50).apply(x, zero)  # r0 = 0
    assert res.status == 0 and res.iterations == 0 and not x.export_field().any()
    for iters in (1, 2, 5, 9):  # the limit, on both sides of the host's reads
        xs = []
        for A in (op, plain):
            y = hip.FieldVector(fs)
            y.set_scalar(0.0)
            res = hip.ConjugateGradient(A, prec, 1e-30, 0.0, iters, monitor_convergence=False, check_every=4).apply(y, b)
            assert res.iterations == iters
            xs.append(y.export_field())
        # the same iterates up to rounding: 1e-12 of the norm after at most 9 iterations
        assert np.linalg.norm(xs[0] - xs[1]) <= 1e-12 * np.linalg.norm(xs[1])
    bad = hip.FieldVector(fs).import_field(np.full(fs.undf, np.nan))
    x.set_scalar(0.0)
    with pytest.raises(hip.LfricError):
        hip.ConjugateGradient(op, prec, 1e-10, 0.0, 50).apply(x, bad)
