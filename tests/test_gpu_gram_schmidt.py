"""Gram-Schmidt of an Arnoldi column in two passes, at the edges of its groups of 8 vectors, of the lanes that
add its partial sums (16, 32, 64, 128) and of its blocks: cycle lengths on both sides of them, vectors shorter
than one block and longer, of odd length and (FP32) a multiple of the 16-byte elements.

One GMRES cycle of m columns minimises ||b - A x|| over the Krylov space of dimension m, whatever
orthogonalisation made its basis.  The residual norm therefore equals that of an orthonormal-basis
least-squares solve in numpy FP64, to what the basis' loss of orthogonality leaves: a few m eps of the
vectors' type times ||b||, here 200 m eps."""
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
    assert got <= best + 200 * m * eps * np.linalg.norm(bb), (got, best)
