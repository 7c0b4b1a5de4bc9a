"""The one-launch apply of lowest-order W0 operators over the per-column table, in both of its orders of
sums, against the kernels that walk the column lists, bit for bit: the colour-ordered and the gather
forms of the multi-RHS apply, whose columns equal the one-RHS forms'.  Sizes with a partial last block,
a single block and several."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["R64", "R32"])
@pytest.mark.parametrize("n,nl", [(2, 1), (3, 2), (4, 63), (5, 7), (12, 20)])
def test_table_apply_equals_the_list_kernels(hip, n, nl, prec):
    P, T = getattr(hip, prec), np.float64 if prec == "R64" else np.float32
    fs = hip.FunctionSpace.cubedsphere(n, nl)
    op = hip.LmaOperator(fs).generate_spd(3 * n + nl)
    op = op if P == hip.R64 else op.convert(P)
    X = np.random.default_rng(nl).uniform(-1, 1, (fs.undf, 2)).astype(T)
    xm, ym = hip.FieldVector(fs, P, 2).import_raw(X.ravel()), hip.FieldVector(fs, P, 2)
    for variant, method in ((2, "apply"), (1, "apply_gather")):
        op.apply_mrhs(xm, ym, variant)
        ref = ym.export_raw().reshape(fs.undf, 2)
        for r in range(2):
            x, y = hip.FieldVector(fs, P).import_raw(X[:, r].copy()), hip.FieldVector(fs, P)
            y.set_scalar(5.0)
            getattr(op, method)(x, y)
            np.testing.assert_array_equal(y.export_raw(), ref[:, r], err_msg=method)


def test_columns_of_five_cells_take_the_lists(hip):
    """Five quadrilaterals around one vertex, a colour each: their common column has no table entry,
    and every form agrees with numpy (8 terms per element row, 5 cells: 13 eps of |A| |x|)."""
    nl, nc = 6, 5
    H = nl + 1
    rim = lambda c: [1 + 2 * c, 2 + 2 * c, 1 + 2 * ((c + 1) % nc)]  # noqa: E731
    verts = np.array([[0] + rim(c) for c in range(nc)])
    dm = np.concatenate([verts * H + 1, verts * H + 2], 1)
    fs = hip.FunctionSpace.from_dofmap(nl, (2 * nc + 1) * H, dm, np.ones(nc), np.arange(1, nc + 1)[:, None])
    op = hip.LmaOperator(fs).generate_spd(4)
    x = np.random.default_rng(0).uniform(-1, 1, fs.undf)
    xv, y = hip.FieldVector(fs).import_field(x), hip.FieldVector(fs)
    A = op.download()
    dofs = ((dm - 1)[:, None, :] + np.arange(nl)[None, :, None]).reshape(fs.ncell_3d, 8)
    ref, mag = np.zeros(fs.undf), np.zeros(fs.undf)
    np.add.at(ref, dofs, np.einsum("cij,cj->ci", A, x[dofs]))
    np.add.at(mag, dofs, np.einsum("cij,cj->ci", np.abs(A), np.abs(x[dofs])))
    for method in ("apply", "apply_gather"):
        getattr(op, method)(xv, y)
        assert np.all(np.abs(y.export_field() - ref) <= 26 * np.finfo(np.float64).eps * mag), method
