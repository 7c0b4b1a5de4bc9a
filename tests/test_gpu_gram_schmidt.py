"""Gram-Schmidt of an Arnoldi column in two passes, at the edges of its groups of 8 vectors, of the lanes that
add its partial sums (16, 32, 64, 128) and of its blocks: cycle lengths on both sides of them, vectors shorter
than one block and longer, of odd length and (FP32) a multiple of the 16-byte elements.

One GMRES cycle of m columns minimises ||b - A x|| over the Krylov space of dimension m, whatever
orthogonalisation made its basis.  The residual norm therefore equals that of an orthonormal-basis
least-squares solve in numpy FP64, to what the roundings of the basis and of x leave: up to 0.05 m eps of the
vectors' type times ||b|| over these cases, and the bound is ten times that.  In FP32 a solve that loses
the last few of its columns exceeds it (33 columns: 2e-6 of ||b|| against a residual of 1.3e-6).

That bound does not see the products l of the basis vectors among themselves, since the basis stays orthogonal
there.  So a second test takes systems (a diagonal operator, few eigenvalues far from a cluster) whose basis
loses its orthogonality within the cycle, and compares the residual with that of modified Gram-Schmidt written
out in numpy with vectors of the same type.  Roundings of the same size leave residuals up to 3.4 times apart
there (numpy, the triangular form against the plain one, four seeds a case); the bound is 8.  Each mistake in l that the
kernels could make exceeds it where it can occur: tests/test_gram_schmidt_cases.py plants them in numpy."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _h(hip, n, nl, P):
    w2 = hip.FunctionSpace.cubedsphere(n, nl, hip.W2, 0)
    w3 = w2.sibling(hip.W3, 0)
    M2 = hip.LmaOperator(w2).generate_spd(0, shift=1.0).convert(P)
    D = hip.LmaOperator(w3, w2).generate_uniform(0, 5, 0.5, 1.5, (-1.0, -1.0, 1.0, 1.0, -1.0, 1.0)).convert(P)
    M3 = hip.LmaOperator(w3).generate_spd(1, shift=1.0).convert(P)
    m2 = M2.mm_diagonal(hip.FieldVector(w2, P))
    return w2, w3, M3, D, m2, hip.LinearOperator.helmholtz(M3, D, m2, 50.0)  # tau: slow enough convergence


def _dense_apply(w2, w3, M3, D, m2):
    nl = w3.nlayers
    lay = np.arange(nl)[None, :, None]
    d3 = ((w3.dofmap() - 1)[:, None, :] + lay).reshape(-1)
    d2 = ((w2.dofmap() - 1)[:, None, :] + lay).reshape(-1, 6)
    Dm, m3, md = D.download()[:, 0, :], M3.download().reshape(-1), m2.export_field()

    def apply(x):
        t = np.zeros(w2.undf)
        np.add.at(t, d2, Dm * x[d3][:, None])
        t /= md
        y = np.zeros_like(x)
        y[d3] = m3 * x[d3] + 50.0 * (Dm * t[d2]).sum(1)
        return y
    return apply


@pytest.mark.parametrize("prec", ["R64", "R32"])
@pytest.mark.parametrize("n,nl,m", [(2, 3, 1), (2, 3, 2), (3, 5, 8), (3, 5, 9), (5, 7, 16), (5, 8, 17), (7, 10, 33),
                                    (12, 10, 31), (12, 40, 64), (60, 30, 5)])
def test_one_cycle_is_the_minimal_residual(hip, n, nl, m, prec):
    P = getattr(hip, prec)
    eps = np.finfo(np.float64 if prec == "R64" else np.float32).eps
    w2, w3, M3, D, m2, H = _h(hip, n, nl, P)
    apply = _dense_apply(w2, w3, M3, D, m2)
    b = hip.FieldVector(w3, P).fill_uniform(2, 3)
    x = hip.FieldVector(w3, P)
    x.set_scalar(0.0)
    hip.GMRES(H, hip.NullPreconditioner(), m, 0.0, 0.0, 1).apply(x, b)
    bb, xx = b.export_field(), x.export_field()
    V = [bb / np.linalg.norm(bb)]
    AV = []
    for j in range(m):  # orthonormal basis, twice orthogonalised
        AV.append(apply(V[j]))
        w = AV[j].copy()
        for _ in range(2):
            w -= np.array(V).T @ (np.array(V) @ w)
        V.append(w / np.linalg.norm(w))
    AV = np.array(AV).T
    best = np.linalg.norm(bb - AV @ np.linalg.lstsq(AV, bb, rcond=None)[0])
    got = np.linalg.norm(bb - apply(xx))
    assert got <= best + 0.5 * m * eps * np.linalg.norm(bb), (got, best)


# m, share of the m columns that are eigenvalues apart, their decades, the cluster's width, (edge cells, levels)
SPECTRA = {
    "R64": [(9, 0.4, (-6, 4), 1e-4, (12, 2)), (17, 0.4, (-9, 4), 1e-2, (9, 6)), (33, 0.4, (-9, 4), 1e-2, (12, 2)),
            (64, 0.4, (-9, 2), 1e-2, (8, 9)), (17, 0.4, (-9, 4), 1e-2, (48, 20))],
    "R32": [(9, 0.4, (-3, 4), 1e-1, (5, 5)), (17, 0.4, (-3, 4), 1e-2, (9, 6)), (33, 0.8, (-3, 4), 1e-4, (12, 2)),
            (64, 0.8, (-3, 4), 1e-2, (9, 6)), (33, 0.8, (-3, 4), 1e-4, (60, 30))],
}
CASES = [(prec, *c) for prec in SPECTRA for c in SPECTRA[prec]]


def diagonal_system(prec, m, share, decades, width, mesh):
    T = np.float64 if prec == "R64" else np.float32
    n, k = 6 * mesh[0] ** 2 * mesh[1], int(share * m)
    rng = np.random.default_rng(n)
    d = np.concatenate([np.logspace(*decades, k), 1.0 + width * rng.random(n - k)])[rng.permutation(n)].astype(T)
    return d, rng.uniform(-1, 1, n).astype(T)


def one_cycle_residual(d, b, m, triangular=False, lost=None):
    """||b - A x|| / ||b|| after one GMRES cycle of m columns on A = diag(d), vectors in b's type, products in
    FP64.  Modified Gram-Schmidt, or its triangular form over the rows l_ij = v_i . v_j; lost(column, i, j) says
    which of them column `column` is to miss."""
    T, V, H, lower = b.dtype.type, [], np.zeros((m + 1, m)), np.zeros((m + 1, m + 1))

    def dot(x, y):
        return float(x.astype(np.float64) @ y.astype(np.float64))
    beta = np.sqrt(dot(b, b))
    V.append((b * T(1.0 / beta)).astype(T))
    for c in range(m):
        w = d * V[c]
        if triangular:
            h = np.array([dot(v, w) for v in V])
            lower[c, :c] = [dot(V[c], v) for v in V[:c]]
            for i in range(c + 1):
                h[i] -= sum(lower[i, j] * h[j] for j in range(i) if not (lost and lost(c, i, j)))
                H[i, c] = h[i]
            for i, v in enumerate(V):
                w = (w + T(-h[i]) * v).astype(T)
        else:
            for i, v in enumerate(V):
                H[i, c] = dot(v, w)
                w = (w + T(-H[i, c]) * v).astype(T)
        H[c + 1, c] = np.sqrt(dot(w, w))
        V.append((w * T(1.0 / H[c + 1, c])).astype(T))
    g = np.zeros(m + 1)
    g[0] = beta
    u = np.linalg.lstsq(H, g, rcond=None)[0]
    x = np.zeros_like(b)
    for c in range(m):
        x = (x + T(u[c]) * V[c]).astype(T)
    r = b.astype(np.float64) - d.astype(np.float64) * x.astype(np.float64)
    return np.linalg.norm(r) / beta


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}-m{c[1]}-{c[5][0]}x{c[5][1]}")
def test_basis_that_loses_orthogonality(hip, case):
    prec, m, mesh = case[0], case[1], case[5]
    P = getattr(hip, prec)
    d, b = diagonal_system(*case)
    w3 = hip.FunctionSpace.cubedsphere(*mesh, hip.W3, 0)
    A = hip.LmaOperator(w3, precision=P)
    dof = ((w3.dofmap() - 1) + np.arange(mesh[1])[None, :]).reshape(-1)
    A.upload(d[dof].astype(np.float64).reshape(-1, 1, 1))
    bv, x = hip.FieldVector(w3, P).import_raw(b), hip.FieldVector(w3, P)
    x.set_scalar(0.0)
    hip.GMRES(hip.LinearOperator.from_lma(A), hip.NullPreconditioner(), m, 0.0, 0.0, 1).apply(x, bv)
    r = b.astype(np.float64) - d.astype(np.float64) * x.export_field()
    got, want = np.linalg.norm(r) / np.linalg.norm(b.astype(np.float64)), one_cycle_residual(d, b, m)
    assert got <= 8 * want, (got, want)
