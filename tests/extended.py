"""Plane solves in extended precision on the CPU, from the oracle's coefficient
tables: what rounding errors are measured against."""
import numpy as np

LD = np.clongdouble


def inverse(A):
    """Inverses of a batch of matrices (S, n, n) by Gauss-Jordan with row pivoting."""
    S, n, _ = A.shape
    M = np.concatenate([A, np.broadcast_to(np.eye(n, dtype=LD), A.shape)], 2)
    at = np.arange(S)
    for k in range(n):
        p = k + np.argmax(np.abs(M[:, k:, k]), 1)
        t = M[at, p].copy()
        M[at, p] = M[:, k]
        M[:, k] = t
        M[:, k] /= M[:, k, k][:, None]
        f = M[:, :, k].copy()
        f[:, k] = 0
        M -= f[:, :, None] * M[:, k][:, None, :]
    return M[:, :, n:]


def blocks(P, nx, ny):
    """Diagonal blocks (ny lists of (slots, nx, nx)), the y couplings to the line
    below and above, and each plane's slot, of an oracle problem."""
    (xm, xp, xd), (ym, yp, yd) = (t[:3] for t in (P.tables(0), P.tables(1)))
    kappa, lam = np.asarray(P.kappa()).reshape(ny, nx), np.asarray(P.lamz())
    distinct, slot = np.unique(lam, return_inverse=True)
    X = np.zeros((nx, nx), LD)
    i = np.arange(nx)
    X[i, i], X[i[1:], i[:-1]], X[i[:-1], i[1:]] = xd, xm[1:], xp[:-1]
    D = []
    for j in range(ny):
        d = np.broadcast_to(X, (distinct.size, nx, nx)).copy()
        d[:, i, i] += (LD(yd[j]) + kappa[j].astype(LD))[None] - distinct.astype(np.longdouble)[:, None]
        D.append(d)
    return D, ym.astype(LD), yp.astype(LD), slot


def chain(D, low, up, inv=inverse):
    """The block inverses G_j = (D_j - low_j up_{j-1} G_{j-1})^-1."""
    G = []
    for j, d in enumerate(D):
        G.append(inv(d - (low[j] * up[j - 1]) * G[-1].astype(LD) if j else d))
    return G


def plane_solve(P, dims, b, adjoint=False):
    """All plane systems M_k x = b (adjoint: M_k^H x = b), b and x of length
    nx ny nz."""
    nx, ny, nz = dims
    D, low, up, slot = blocks(P, nx, ny)
    if adjoint:
        D = [d.conj().transpose(0, 2, 1) for d in D]
        low, up = np.append(LD(0), up[:-1].conj()), np.append(low[1:].conj(), LD(0))
    G = chain(D, low, up)
    B = np.asarray(b).reshape(nz, ny, nx).astype(LD)
    x = np.empty_like(B)
    for k in range(nz):
        t = [B[k, 0]]
        for j in range(1, ny):
            t.append(B[k, j] - low[j] * (G[j - 1][slot[k]] @ t[-1]))
        x[k, -1] = G[-1][slot[k]] @ t[-1]
        for j in range(ny - 2, -1, -1):
            x[k, j] = G[j][slot[k]] @ (t[j] - up[j] * x[k, j + 1])
    return x.reshape(-1)


def error(got, want):
    d = (np.asarray(got).astype(LD) - want).astype(np.complex128)
    return float(np.linalg.norm(d) / np.linalg.norm(want.astype(np.complex128)))
