"""The W2 applies over the tables of columns and neighbours.

The 6 x 6 apply in both orders of sums equals the multi-RHS kernels that walk the column lists and the colours,
bit for bit.

The transpose apply of 1 x 6 (W3 <- W2) operators over the neighbour table, and enforce_bc inside the
W2 mass apply, against numpy on the element matrices, bit for bit up to the order of two terms: a side-face
dof is fl(D1 x1) + fl(D2 x2) (commutative), a bottom/top-face dof fma(D5, x', fl(D4 x)).  numpy has no fma, so
the second is compared within one rounding of the product (2 eps of |D||x|)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["R64", "R32"])
@pytest.mark.parametrize("n,nl", [(2, 1), (3, 2), (4, 16), (5, 51), (9, 7)])
def test_table_apply_equals_the_list_kernels(hip, n, nl, prec):
    P, T = getattr(hip, prec), np.float64 if prec == "R64" else np.float32
    w2 = hip.FunctionSpace.cubedsphere(n, nl, hip.W2, 0)
    op = hip.LmaOperator(w2).generate_spd(n + nl, shift=1.0)
    op = op if P == hip.R64 else op.convert(P)
    X = np.random.default_rng(nl).uniform(-1, 1, (w2.undf, 2)).astype(T)
    xm, ym = hip.FieldVector(w2, P, 2).import_raw(X.ravel()), hip.FieldVector(w2, P, 2)
    for variant, method in ((2, "apply"), (1, "apply_gather")):
        op.apply_mrhs(xm, ym, variant)
        ref = ym.export_raw().reshape(w2.undf, 2)
        x, y = hip.FieldVector(w2, P).import_raw(X[:, 1].copy()), hip.FieldVector(w2, P)
        y.set_scalar(5.0)
        getattr(op, method)(x, y)
        np.testing.assert_array_equal(y.export_raw(), ref[:, 1], err_msg=method)


@pytest.mark.parametrize("prec", ["R64", "R32"])
@pytest.mark.parametrize("n,nl", [(2, 1), (3, 2), (4, 16), (5, 51), (9, 7)])
def test_transpose_over_the_neighbour_table(hip, n, nl, prec):
    P, T = getattr(hip, prec), np.float64 if prec == "R64" else np.float32
    w2 = hip.FunctionSpace.cubedsphere(n, nl, hip.W2, 0)
    w3 = w2.sibling(hip.W3, 0)
    D = hip.LmaOperator(w3, w2).generate_uniform(n, 5, 0.5, 1.5, (-1.0, -1.0, 1.0, 1.0, -1.0, 1.0))
    D = D if P == hip.R64 else D.convert(P)
    x = np.random.default_rng(nl).uniform(-1, 1, w3.undf).astype(T)
    xv, y = hip.FieldVector(w3, P).import_raw(x), hip.FieldVector(w2, P)
    y.set_scalar(9.0)
    D.apply_transpose(xv, y)
    lay = np.arange(nl)[None, :, None]
    d3 = ((w3.dofmap() - 1)[:, None, :] + lay).reshape(-1)
    d2 = ((w2.dofmap() - 1)[:, None, :] + lay).reshape(-1, 6)
    prod = (D.download()[:, 0, :].astype(T) * x[d3][:, None]).astype(T)  # one rounding each
    ref, mag = np.zeros(w2.undf, T), np.zeros(w2.undf)
    np.add.at(ref, d2, prod)
    np.add.at(mag, d2, np.abs(prod).astype(np.float64))
    got = y.export_raw()
    side = np.unique(d2[:, :4])
    np.testing.assert_array_equal(got[side], ref[side])
    assert np.all(np.abs(got.astype(np.float64) - ref) <= 2 * np.finfo(T).eps * mag)


@pytest.mark.parametrize("prec", ["R64", "R32"])
@pytest.mark.parametrize("n,nl", [(2, 1), (3, 5), (6, 43)])
def test_boundary_conditions_inside_the_mass_apply(hip, n, nl, prec):
    P = getattr(hip, prec)
    w2 = hip.FunctionSpace.cubedsphere(n, nl, hip.W2, 0)
    op = hip.LmaOperator(w2).generate_spd(n, shift=1.0)
    op = op if P == hip.R64 else op.convert(P)
    x, y, z = hip.FieldVector(w2, P).fill_uniform(1), hip.FieldVector(w2, P), hip.FieldVector(w2, P)
    hip.LinearOperator.mass_matrix(op, True).apply(x, y)
    hip.LinearOperator.mass_matrix(op, False).apply(x, z)
    z.enforce_bc()
    np.testing.assert_array_equal(y.export_raw(), z.export_raw())
    assert np.count_nonzero(y.export_raw() == 0) == 2 * w2.ncells
