"""apy_aat_terms over the sizes where its kernels change: tile edges of the virtual sandwich (16 columns, W in
LDS up to 96, registers up to 160), row blocks of the occupied transforms (16, up to 36), the general path beyond
them, antisymmetric and general doubles, missing amplitudes, and jobs
that share operands (more than one pass of four per ket).  Reference: the defining sums in NumPy."""
import numpy as np
import pytest

from tests.test_gpu_aat import _c, _d, _gamma, _terms

pytestmark = pytest.mark.gpu


def _alt(t):
    return 0.25 * (t - t.transpose(0, 1, 3, 2) - t.transpose(1, 0, 2, 3) + t.transpose(1, 0, 3, 2))


def _reference(S, no, nf, b1, b2, k1, k2):
    """The 20 scalars of one overlap class from Gamma's blocks, and the sum of |terms| of the largest."""
    oa, nv = no - nf, S.shape[0] - no
    Pi = np.linalg.inv(S[:no, :no])
    x = (S[no:, :no] @ Pi).T[nf:]
    Y = Pi @ S[:no, no:]
    W = S[no:, no:] - S[no:, :no] @ Y
    y, P = Y[nf:], Pi[nf:, nf:]
    z1, z2 = np.zeros((oa, nv), complex), np.zeros((oa, oa, nv, nv), complex)
    B1, B2, K1, K2 = (z if t is None else t for t, z in ((b1, z1), (b2, z2), (k1, z1), (k2, z2)))
    m = lambda t: t.transpose(0, 2, 1, 3).reshape(oa * nv, oa * nv)
    xv, yv = x.ravel(), y.ravel()
    be, bp, bh = m(B2) @ xv, m(B2).T @ xv, m(_alt(B2)) @ xv
    kA, kB, kh = m(K2) @ yv, m(K2).T @ yv, -(m(_alt(K2)) @ yv)
    H = lambda M: (P.T @ M.reshape(oa, nv) @ W.T).ravel()
    h0, h1, h2, h3 = H(K1), H(kh), H(kA), H(kB)
    T = np.matmul(np.matmul(W, K2), W.T).reshape(oa, oa, -1)
    T = np.matmul(P.T, T)
    T = (P.T @ T.reshape(oa, -1)).reshape(oa, oa, nv, nv)
    b, k = B1.ravel(), K1.ravel()
    nt = (b2 is not None and k2 is not None) * 1.0
    out = np.array([np.linalg.det(S[:no, :no]), b @ xv, k @ yv, be @ xv, bh @ xv, kA @ yv, -(kh @ yv), b @ h0, be @ h0,
                    bh @ h0, b @ h1, b @ h2, bh @ h1, bh @ h2, be @ h1, bp @ h1, bp @ h3, be @ h2,
                    nt * np.sum(B2 * _alt(T)), nt * np.sum(B2 * T)])
    scale = np.array([1.0, *[np.linalg.norm(u) * np.linalg.norm(v) for u, v in
                             ((b, xv), (k, yv), (be, xv), (bh, xv), (kA, yv), (kh, yv), (b, h0), (be, h0), (bh, h0),
                              (b, h1), (b, h2), (bh, h1), (bh, h2), (be, h1), (bp, h1), (bp, h3), (be, h2),
                              (B2, T), (B2, T))]])
    return out, scale


@pytest.mark.parametrize("no,nv,nf,anti", [(1, 1, 0, False), (2, 16, 0, True), (3, 17, 1, False), (7, 15, 0, True),
                                           (6, 33, 0, False), (9, 50, 0, True), (4, 65, 1, False), (3, 97, 0, True),
                                           (2, 130, 0, False), (16, 5, 0, True), (18, 4, 1, False), (33, 3, 0, True),
                                           (36, 2, 0, False), (2, 161, 0, False), (37, 2, 0, True)])
def test_terms_match_the_defining_sums(dev, no, nv, nf, anti):
    rng = np.random.default_rng(no * 1000 + nv)
    n, oa = no + nv, no - nf
    S = [np.eye(n) + 0.3 / np.sqrt(n) * _c(rng, n, n) for _ in range(2)]
    g, rec = _gamma(S, no, nf, dev)
    sym = _alt if anti else (lambda t: t)
    amps = [(_c(rng, oa, nv), sym(_c(rng, oa, oa, nv, nv))) for _ in range(3)]
    amps[2] = (amps[2][0], sym(_c(rng, oa, oa, nv, nv)) if oa < 2 else _c(rng, oa, oa, nv, nv))   # never flagged
    dv = [(_d(a, dev), _d(b, dev)) for a, b in amps]
    # six jobs share the ket (gamma 0, set 1), the others share bras, leave amplitudes out or mix the symmetries
    jobs = [(0, 0, 1), (0, 2, 1), (0, 1, 1), (0, 0, 1), (0, 2, 1), (0, 1, 1), (1, 0, 2), (1, 2, 0), (0, None, 1),
            (1, 0, None)]
    pick = lambda t, k: (None, None) if k is None else t[k]
    out = _terms(g, rec, oa, nv, [(gi, *pick(dv, b), *pick(dv, k)) for gi, b, k in jobs], dev)
    for row, (gi, b, k) in zip(out, jobs):
        ref, scale = _reference(S[gi], no, nf, *pick(amps, b), *pick(amps, k))
        # rounding of sums of up to (oa nv)^2 terms in another order, against the product of the norms
        assert np.abs(row[0] - ref[0]) < 1e-12 * abs(ref[0])
        assert (np.abs(row[1:] - ref[1:]) <= 1e-13 * np.sqrt(oa * nv) * scale[1:] + 1e-300).all(), (gi, b, k)
