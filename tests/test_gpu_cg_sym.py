"""Conjugate gradients over the symmetric-packed copy.

* Against the same solve over the element layout: the operators are the same and only the order of a sum
  changes, so the iteration counts agree within one and the solutions to what a residual of r_tol leaves
  (condition of B B^T + 0.1 I elements below 100: 100 r_tol).  Sizes with one block and several, partial blocks
  and wavefronts; and the ends of a solve: no iteration (b = 0 and an exact initial guess), the iteration limit,
  monitoring off.
* Against the iteration written out in the public vector operations, bit for bit, over systems whose columns
  are scaled by 10^U(-2, 2): hundreds of FP32 iterations carry one rounding of alpha to another stopping
  point, so the products have to be those of the vectors themselves (p . (A p) of the gathered A p).  Up to
  2048 blocks of 256 dofs a dot's partial sums are the apply's.
* The apply itself against the colour-ordered one, bit for bit, on both sides of the size (524288 points)
  from which a thread of its second kernel takes several points.
* The scaled mixed-precision solve against its refinement written out the same way, and its residual in
  the oracle's assembled matrix."""
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


def _scaled_system(hip, n, nl, copy, prec):
    fs = hip.FunctionSpace.cubedsphere(n, nl)
    op64 = hip.LmaOperator(fs).generate_spd(n + nl, scaled=True)
    ops = [op64, op64.convert(hip.R32)] if prec == "mixed" else [op64 if prec == "R64" else op64.convert(hip.R32)]
    for op in ops:
        if copy == "rows":
            op.prepare_rows()
        elif copy == "symmetric":
            op.prepare_symmetric()
    return (fs, *ops)


def _cg_by_vector_operations(hip, op, diag, b, iterations):
    """x after each iteration from x = 0 (cg_solve without a convergence test)."""
    A = hip.LinearOperator.from_lma(op)
    x, r, z, p, q = (b.duplicate() for _ in range(5))
    x.set_scalar(0.0)
    r.copy(b)
    z.divide(r, diag)
    p.copy(z)
    rz = r.dot(z)
    for _ in range(iterations):
        A.apply(p, q)
        alpha = rz / p.dot(q)
        x.axpy(alpha, p)
        r.axpy(-alpha, q)
        z.divide(r, diag)
        rz, old = r.dot(z), rz
        p.aypx(rz / old, z)
    return x


@pytest.mark.parametrize("prec", ["R64", "R32"])
@pytest.mark.parametrize("copy", ["none", "rows", "symmetric"])
@pytest.mark.parametrize("n,nl", [(4, 62), (12, 20), (32, 60)])
def test_scaled_cg_equals_the_vector_operations(hip, n, nl, copy, prec):
    P = getattr(hip, prec)
    fs, op = _scaled_system(hip, n, nl, copy, prec)
    diag = op.mm_diagonal(hip.FieldVector(fs, P))
    b = hip.FieldVector(fs, P).fill_uniform(n, 3)
    for iters in (7, 60):
        x = hip.FieldVector(fs, P)
        x.set_scalar(0.0)
        res = hip.ConjugateGradient(op, hip.DiagonalPreconditioner(diag), 1e-30, 0.0, iters, monitor_convergence=False,
                                    check_every=16).apply(x, b)
        assert res.iterations == iters
        np.testing.assert_array_equal(x.export_raw(), _cg_by_vector_operations(hip, op, diag, b, iters).export_raw())


@pytest.mark.parametrize("copy", ["none", "rows", "symmetric"])
def test_scaled_mixed_precision_solve(hip, orc, copy):
    fs, op, op32 = _scaled_system(hip, 8, 12, copy, "mixed")
    prec = hip.DiagonalPreconditioner.from_operator(op32)
    b, x = hip.FieldVector(fs).fill_uniform(1, 3), hip.FieldVector(fs)
    A, want = hip.LinearOperator.from_lma(op), np.zeros(fs.undf)
    for outer in range(2):
        # r = b - A x, its inner solve to the remaining reduction, and x + ||r|| d
        xw, r = hip.FieldVector(fs).import_field(want), hip.FieldVector(fs)
        A.apply(xw, r)
        r.import_field(b.export_field() - r.export_field())
        nr = r.norm()
        nr0 = nr if outer == 0 else nr0
        b32, d32 = hip.FieldVector(fs, hip.R32), hip.FieldVector(fs, hip.R32)
        b32.import_raw((r.export_field() * (1.0 / nr)).astype(np.float32))
        d32.set_scalar(0.0)
        hip.ConjugateGradient(op32, prec, max(1e-4, 0.5 * 1e-8 * nr0 / nr), 0.0, 2000).apply(d32, b32)
        want = want + nr * d32.export_raw().astype(np.float64)
        x.set_scalar(0.0)
        res = hip.MixedPrecisionCG(op, op32, prec, 1e-8, 0.0, 2000, max_outer=outer + 1).apply(x, b)
        assert res.outer_iterations == outer + 1
        got = x.export_field()
        # the device adds nr d to x with or without rounding the product first
        assert np.all(np.abs(got - want) <= np.finfo(np.float64).eps * (np.abs(got) + np.abs(want)))
        want = got
    x.set_scalar(0.0)
    res = hip.MixedPrecisionCG(op, op32, prec, 1e-8, 0.0, 2000).apply(x, b)
    assert res.status == 0
    m = orc.Mesh(8, 12)
    S = orc.assembled_csr(m, orc.gen_spd(m.ndf, m.ncell_3d, 20, scaled=True))
    bb = b.export_field()
    assert np.linalg.norm(bb - S @ x.export_field()) <= 1e-8 * np.linalg.norm(bb)


@pytest.mark.parametrize("prec", ["R64", "R32"])
@pytest.mark.parametrize("nl,points", [(36, 511562), (37, 525388)])
def test_apply_beside_the_several_points_limit(hip, nl, points, prec):
    P = getattr(hip, prec)
    fs = hip.FunctionSpace.cubedsphere(48, nl)
    assert fs.undf == points
    op = hip.LmaOperator(fs).generate_spd(nl)
    op = op if P == hip.R64 else op.convert(P)
    x, y, z = hip.FieldVector(fs, P).fill_uniform(1), hip.FieldVector(fs, P), hip.FieldVector(fs, P)
    op.apply(x, y)
    op.prepare_symmetric()
    z.set_scalar(7.0)
    hip.LinearOperator.from_lma(op).apply(x, z)
    np.testing.assert_array_equal(z.export_raw(), y.export_raw())
