"""The colour-ordered apply of order-1 W0 operators with each unit's rows split over threads, at
sizes that leave partial blocks and partial groups of blocks, on one and on several blocks.

* Against the element matrices and the dofmap in numpy, FP64: every output is a sum of at most 4 cells' fma
  chains of 27 terms (two for a dof shared by layers), so it is within (27 + 8) eps of |A| |x|.
* Several right-hand sides equal the one-right-hand-side apply column by column, bit for bit; also on both
  sides of the colour sizes (16384 and 32768 units) where the split of a unit's rows changes and where one
  thread a unit takes over, and in the automatic choice (for 8 FP64 right-hand sides the gather form's bits)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["R64", "R32"])
@pytest.mark.parametrize("n,nl", [(2, 1), (3, 2), (5, 7), (12, 9), (13, 31)])
def test_order1_colour_apply(hip, n, nl, prec):
    P, T = getattr(hip, prec), np.float64 if prec == "R64" else np.float32
    fs = hip.FunctionSpace.cubedsphere(n, nl, hip.W0, 1)
    op = hip.LmaOperator(fs).generate_spd(n + nl)
    op = op if P == hip.R64 else op.convert(P)
    X = np.random.default_rng(n).uniform(-1, 1, (fs.undf, 8)).astype(T)
    A = op.download()
    dofs = ((fs.dofmap() - 1)[:, None, :] + np.arange(nl)[None, :, None]).reshape(fs.ncell_3d, 27)
    cols = []
    for r in range(8):
        x, y = hip.FieldVector(fs, P).import_raw(X[:, r].copy()), hip.FieldVector(fs, P)
        y.set_scalar(7.0)
        op.apply(x, y)
        cols.append(y.export_raw())
    xe = X[:, 0].astype(np.float64)[dofs]
    ref, mag = np.zeros(fs.undf), np.zeros(fs.undf)
    np.add.at(ref, dofs, np.einsum("cij,cj->ci", A, xe))
    np.add.at(mag, dofs, np.einsum("cij,cj->ci", np.abs(A), np.abs(xe)))
    # 8 eps_64 more for the reference's own sums, which matter beside FP64 only
    assert np.all(np.abs(cols[0] - ref) <= (35 * np.finfo(T).eps + 35 * np.finfo(np.float64).eps) * mag)
    for nr in (2, 4, 8):
        xm, ym = hip.FieldVector(fs, P, nr).import_raw(X[:, :nr].ravel()), hip.FieldVector(fs, P, nr)
        ym.set_scalar(-3.0)
        op.apply_mrhs(xm, ym, 2)
        np.testing.assert_array_equal(ym.export_raw().reshape(fs.undf, nr), np.stack(cols[:nr], 1))


@pytest.mark.parametrize("prec", ["R64", "R32"])
@pytest.mark.parametrize("nl,units", [(17, 15552), (18, 16416), (36, 31968), (37, 32832)])
def test_order1_colour_apply_beside_the_split_limits(hip, nl, units, prec):
    P, T = getattr(hip, prec), np.float64 if prec == "R64" else np.float32
    fs = hip.FunctionSpace.cubedsphere(24, nl, hip.W0, 1)
    assert int(fs.colouring()[0].max()) * (nl + 1) == units
    op = hip.LmaOperator(fs).generate_spd(nl)
    op = op if P == hip.R64 else op.convert(P)
    X = np.random.default_rng(nl).uniform(-1, 1, (fs.undf, 8)).astype(T)
    x, y = hip.FieldVector(fs, P), hip.FieldVector(fs, P)
    cols = []
    for r in range(8):
        op.apply(x.import_raw(X[:, r].copy()), y)
        cols.append(y.export_raw())
    for nr in (2, 4, 8):
        xm, ym = hip.FieldVector(fs, P, nr).import_raw(X[:, :nr].ravel()), hip.FieldVector(fs, P, nr)
        for variant in (2, 0):
            ym.set_scalar(-3.0)
            op.apply_mrhs(xm, ym, variant)
            got = ym.export_raw().reshape(fs.undf, nr)
            if variant == 0 and nr == 8 and prec == "R64":
                op.apply_mrhs(xm, ym, 1)
                np.testing.assert_array_equal(got, ym.export_raw().reshape(fs.undf, nr))
            else:
                np.testing.assert_array_equal(got, np.stack(cols[:nr], 1))
