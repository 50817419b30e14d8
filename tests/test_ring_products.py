"""The four-product form of the ring terms against the six products they are written with, and RCCSD's o v^3 product
on packed pairs against the whole one, in NumPy."""
import numpy as np
import pytest


def _x(M, o, v):  # M[ib,ja] at [ia,jb]
    return M.reshape(o, v, o, v).transpose(0, 3, 2, 1).reshape(o * v, o * v)


@pytest.mark.parametrize("o,v", [(1, 1), (1, 4), (3, 1), (2, 5), (4, 7)])
@pytest.mark.parametrize("singles", [False, True])
def test_four_ring_products_equal_six(o, v, singles):
    """With symmetric T and Tx (its exchanged form), U = 2T - Tx and, in RCCSD, Q = Tx + 2 tt^x, U2 = 2T - Q,
    E the T1 and Fock-like parts of WE and J1 those of WJ:
    WJ = K + K U2/2 - Kx T/2 + J1 (+ none of E), WE = -J + Kx Q/2 + E, G = T WE + U WJ + (Tx WE)^x equals
    U W + Y/2 + Y^x with W = K - J/2 + (K - Kx/2) U2/2 + J1 + E/2 and Y = Tx WE."""
    rng = np.random.default_rng(100 * o + v)
    n = o * v
    sym = lambda: (lambda A: A + A.T)(rng.normal(size=(n, n)))
    K, J, T = sym(), sym(), sym()
    Kx, Tx = _x(K, o, v), _x(T, o, v)
    assert np.array_equal(Kx, Kx.T) and np.array_equal(Tx, Tx.T)
    E, J1 = rng.normal(size=(n, n)), rng.normal(size=(n, n)) * singles
    t1 = rng.normal(size=(o, v)) * singles
    Q = Tx + 2 * np.einsum("ib,ja->iajb", t1, t1).reshape(n, n)
    U, U2 = 2 * T - Tx, 2 * T - Q
    WE = -J + 0.5 * Kx @ Q + E
    WJ = K + 0.5 * K @ U2 - 0.5 * Kx @ T + J1
    ref = T @ WE + U @ WJ + _x(Tx @ WE, o, v)
    W = K - 0.5 * J + 0.5 * (K - 0.5 * Kx) @ U2 + J1 + 0.5 * E
    Y = Tx @ WE
    got = U @ W + 0.5 * Y + _x(Y, o, v)
    # rounding only: a few products of n terms
    assert np.max(np.abs(got - ref)) < 64 * n * 2.3e-16 * np.max(np.abs(ref) + 10)


@pytest.mark.parametrize("o,v", [(1, 1), (1, 3), (2, 1), (3, 4), (4, 6)])
def test_z_on_packed_pairs(o, v):
    """Z[ij,am] = sum_ef tau[ij,ef] M[ef,am] with tau[ij,ef] = tau[ji,fe] and any M equals Zp + Zm for i <= j and
    Zp - Zm for i > j, Zp = T+ G+ and Zm = T- G- over pairs e <= f and e < f."""
    rng = np.random.default_rng(10 * o + v)
    t = rng.normal(size=(o, o, v, v))
    t = t + t.transpose(1, 0, 3, 2)
    M = rng.normal(size=(v, v, v * o))
    ref = np.einsum("ijef,efc->ijc", t, M)
    le = [(e, f) for f in range(v) for e in range(f + 1)]
    lt = [(e, f) for f in range(v) for e in range(f)]
    Gp = np.array([0.5 * (M[e, f] + M[f, e]) for e, f in le])
    Gm = np.array([0.5 * (M[e, f] - M[f, e]) for e, f in lt]).reshape(len(lt), v * o)
    for i in range(o):
        for j in range(i, o):
            Tp = np.array([t[i, j, e, f] + (t[i, j, f, e] if e != f else 0.0) for e, f in le])
            Tm = np.array([t[i, j, e, f] - t[i, j, f, e] for e, f in lt])
            zp, zm = Tp @ Gp, Tm @ Gm
            assert np.allclose(zp + zm, ref[i, j], rtol=1e-13, atol=1e-13)
            assert np.allclose(zp - zm, ref[j, i], rtol=1e-13, atol=1e-13)


@pytest.mark.parametrize("o,v", [(1, 1), (2, 3), (3, 5)])
def test_merged_singles_terms(o, v):
    """S = H + H^T does not tell H's terms from their transposes: the term t1[ie] (jb|ae) taken as A[ia,jb] =
    sum_f t1[jf] (ia|bf), and the T1^2 and T1-linear terms as one product -t1[ma] Q[mi,jb], give the same S."""
    rng = np.random.default_rng(5 * o + v)
    es = np.einsum
    t1 = rng.normal(size=(o, v))
    ovvv, ooov = rng.normal(size=(o, v, v, v)), rng.normal(size=(o, o, o, v))
    ovvv = ovvv + ovvv.transpose(0, 1, 3, 2)                         # (ia|bc) = (ia|cb)
    K, J = rng.normal(size=(o, v, o, v)), rng.normal(size=(o, v, o, v))
    K = K + K.transpose(2, 3, 0, 1)
    H = -es("ma,imjb->iajb", t1, es("ie,mejb->imjb", t1, K)) - es("mb,imaj->iajb", t1, es("ie,maje->imaj", t1, J))
    H = H + es("ie,jbae->iajb", t1, ovvv) - es("ma,mijb->iajb", t1, ooov)
    Q = ooov + es("ie,jbme->mijb", t1, K) + es("je,mbie->mijb", t1, J)
    G = es("jf,iabf->iajb", t1, ovvv) - es("ma,mijb->iajb", t1, Q)
    assert np.allclose(G + G.transpose(2, 3, 0, 1), H + H.transpose(2, 3, 0, 1), rtol=1e-12, atol=1e-12)


@pytest.mark.parametrize("o,v", [(1, 1), (2, 3), (3, 5)])
def test_singles_residual_terms(o, v):
    """The T1 residual's terms 2 t1[me] (ia|me) - t1[me] (mi|ae) as traces of the ring's T1 products, and its two
    products of T2 with (mi|ne) as one with U = 2T - Tx."""
    rng = np.random.default_rng(7 * o + v)
    es = np.einsum
    t1 = rng.normal(size=(o, v))
    K, J, ooov = rng.normal(size=(o, v, o, v)), rng.normal(size=(o, v, o, v)), rng.normal(size=(o, o, o, v))
    K = K + K.transpose(2, 3, 0, 1)
    KT, JT = es("ie,jbme->jbmi", t1, K), es("je,mbie->mbij", t1, J)
    ref = 2 * es("me,iame->ia", t1, K) - es("me,maie->ia", t1, J)
    assert np.allclose(2 * es("iamm->ia", KT) - es("maim->ia", JT), ref, rtol=1e-12, atol=1e-12)
    t2 = rng.normal(size=(o, o, v, v))
    t2 = t2 + t2.transpose(1, 0, 3, 2)
    T = t2.transpose(0, 2, 1, 3)
    U = 2 * T - es("ijba->iajb", t2)
    ref = -2 * es("nema,mine->ia", T, ooov) + es("nema,nime->ia", T, ooov)
    assert np.allclose(-es("nema,mine->ia", U, ooov), ref, rtol=1e-12, atol=1e-12)
