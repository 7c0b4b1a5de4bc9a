"""The W2 applies over the tables of columns and neighbours.

The 6 x 6 apply in both orders of sums equals the multi-RHS kernels that walk the column lists and the colours,
bit for bit.

The transpose apply of 1 x 6 (W3 <- W2) operators over the neighbour table, and enforce_bc inside the
W2 mass apply, against numpy on the element matrices, bit for bit up to the order of two terms: a side-face
dof is fl(D1 x1) + fl(D2 x2) (commutative), a bottom/top-face dof fma(D5, x', fl(D4 x)).  numpy has no fma, so
the second is compared within one rounding of the product (2 eps of |D||x|).

Dofmaps that the tables do not describe (a side face of three cells, a bottom-face column that two cells share,
or that is another cell's side face) take the general kernels: every apply, and a solve, against numpy."""
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


# 5 cells in a row, each its own colour: the columns of faces 0..3 and of the bottom face by name, neighbours'
# side faces shared; alias replaces a (cell, face)'s column
def _row_of_cells(nl, alias):
    cols = [[("s", c), ("t", c), ("s", c + 1), ("u", c), ("b", c)] for c in range(5)]
    for c, d, name in alias:
        cols[c][d] = name
    tall = {cols[c][4] for c in range(5)}
    base, dm, undf = {}, np.zeros((5, 6), np.int32), 0
    for c in range(5):
        for d in range(5):
            name = cols[c][d]
            if name not in base:
                base[name] = undf + 1
                undf += nl + (name in tall)
            dm[c, d] = base[name]
        dm[c, 5] = dm[c, 4] + 1
    return dm, undf


@pytest.mark.parametrize("prec", ["R64", "R32"])
@pytest.mark.parametrize("alias", [[], [(4, 1, ("s", 1))], [(3, 4, ("b", 0))], [(4, 1, ("b", 2))]],
                         ids=["row", "three-cell side face", "shared bottom column", "bottom column and side face"])
@pytest.mark.parametrize("nl", [2, 5])
def test_dofmaps_beyond_the_tables(hip, nl, alias, prec):
    P, T = getattr(hip, prec), np.float64 if prec == "R64" else np.float32
    eps = np.finfo(T).eps
    dm, undf = _row_of_cells(nl, alias)
    nc = 5
    colours = np.ones(nc), np.arange(1, nc + 1)[:, None]
    w2 = hip.FunctionSpace.from_dofmap(nl, undf, dm, *colours)
    w3 = hip.FunctionSpace.from_dofmap(nl, nc * nl, np.arange(nc)[:, None] * nl + 1, *colours)
    M2, M3 = hip.LmaOperator(w2).generate_spd(1, shift=1.0), hip.LmaOperator(w3).generate_spd(2, shift=1.0)
    D = hip.LmaOperator(w3, w2).generate_uniform(3, 5, 0.5, 1.5, (-1.0, -1.0, 1.0, 1.0, -1.0, 1.0))
    if P == hip.R32:
        M2, M3, D = M2.convert(P), M3.convert(P), D.convert(P)
    d2 = ((dm - 1)[:, None, :] + np.arange(nl)[None, :, None]).reshape(-1, 6)
    A2, A3, Dm = M2.download(), M3.download().reshape(-1), D.download()[:, 0, :]
    S = np.zeros((undf, undf))
    np.add.at(S, (d2[:, :, None], d2[:, None, :]), A2)
    G = np.zeros((nc * nl, undf))
    np.add.at(G, (np.arange(nc * nl)[:, None], d2), Dm)

    def close(got, ref, mag):  # sums of at most 3 cells' two rows of 6, and one more product
        assert np.all(np.abs(got - ref) <= 48 * eps * mag), np.max(np.abs(got - ref) / mag)

    x, y = hip.FieldVector(w2, P).fill_uniform(4), hip.FieldVector(w2, P)
    xx = x.export_field()
    gathers = [M2.apply_gather, hip.LinearOperator.from_lma(M2).apply, hip.LinearOperator.mass_matrix(M2, True).apply]
    if alias == [(4, 1, ("b", 2))]:  # a column of two heights: the column lists refuse it
        for apply in gathers:
            with pytest.raises(hip.LfricError):
                apply(x, y)
        gathers = []
    for apply in [M2.apply] + gathers:
        y.set_scalar(0.0)
        apply(x, y)
        close(y.export_field(), (S @ xx), (np.abs(S) @ np.abs(xx)))
    p, u = hip.FieldVector(w3, P).fill_uniform(5), hip.FieldVector(w2, P)
    pp = p.export_field()
    u.set_scalar(0.0)
    D.apply_transpose(p, u)
    close(u.export_field(), (G.T @ pp), (np.abs(G.T) @ np.abs(pp)))
    if not gathers:
        return
    m2 = M2.mm_diagonal(hip.FieldVector(w2, P))
    mm = m2.export_field()
    q = hip.FieldVector(w3, P)
    hip.LinearOperator.helmholtz(M3, D, m2, 0.5).apply(p, q)
    H = np.diag(A3) + 0.5 * G @ np.diag(1.0 / mm) @ G.T
    Habs = np.diag(np.abs(A3)) + 0.5 * np.abs(G) @ np.diag(1.0 / mm) @ np.abs(G.T)
    close(q.export_field(), H @ pp, Habs @ np.abs(pp))
    # a solve, whose p.(A p) comes from the apply
    sol = hip.FieldVector(w2, P)
    sol.set_scalar(0.0)
    r_tol = 1e-10 if P == hip.R64 else 1e-4
    res = hip.ConjugateGradient(M2, hip.DiagonalPreconditioner(m2), r_tol, 0.0, 200).apply(sol, x)
    assert res.status == 0
    assert np.linalg.norm(xx - S @ sol.export_field()) <= 2 * r_tol * np.linalg.norm(xx)
