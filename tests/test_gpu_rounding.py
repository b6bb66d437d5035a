"""Rounding errors of the z-FFTs, the plane factorisation and the plane solves
against extended precision: a faster kernel's may not be larger than the general
kernel's on the same data."""
import numpy as np
import pytest

import extended
from conftest import load_pkg

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def hz():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return load_pkg()


@pytest.mark.parametrize("nz", [14, 22, 26, 33, 36, 39, 48, 49, 65, 91, 100, 104, 121, 143, 144, 150, 169, 240, 256])
def test_fft_rounding(hz, monkeypatch, nz):
    """complex128 transforms in registers against the general kernel's (16 lines
    a workgroup).  Both round each of about log n levels once and take their
    constants to the last place, so their errors over 2 x 528 lines agree but for
    scatter: 15%."""
    from scipy import fft
    d = hz.problem.cube_geometry((24, 22, nz), 0, 6.0)
    S = hz.Solver(d, np.ones(d.N))
    rng = np.random.default_rng(nz)
    x = rng.standard_normal((2, nz, 528)) + 1j * rng.standard_normal((2, nz, 528))
    want = fft.fft(x.astype(extended.LD), axis=1).reshape(2, -1)
    assert want.dtype == extended.LD
    e = {}
    for lines in ("16", "0"):
        monkeypatch.setenv("HZ_FFT_LINES", lines)
        got = S.fft_z(torch.from_numpy(x.reshape(2, -1)).cuda(), -1, hz.abi.PREC_FP64).cpu().numpy()
        e[lines] = extended.error(got, want)
    print("nz=%d general %.3g registers %.3g" % (nz, e["16"], e["0"]), flush=True)
    assert e["0"] < 1.15 * e["16"]


def _layers(hz, nx, ny, nz, seed):
    """A box of 10 points per wavelength with four-point layers on every face, a
    rough medium, and a right-hand side that both precisions hold exactly."""
    pr = hz.problem
    h = 1.0 / min(nx, ny, nz)
    d = pr.cube_geometry((nx, ny, nz), 4, pr.omega_for_ppw(0.7, h, 10), beta=1.0, pml_c=3.0 * np.log(1e6) / (8.0 * h))
    rng = np.random.default_rng(seed)
    c = 0.8 + 0.5 * rng.random(d.N)
    return d, c, (rng.standard_normal(d.N) + 1j * rng.standard_normal(d.N)).astype(np.complex64)


def _solve(S, hz, b, prec, adjoint=False):
    dt = np.complex128 if prec == hz.abi.PREC_FP64 else np.complex64
    return S.plane_solve(torch.from_numpy(b.astype(dt)).cuda(), prec, adjoint=adjoint).cpu().numpy()


def _inverse_c64(A):
    """Gauss-Jordan in complex64 with partial pivoting, every update's product
    formed and then subtracted: one rounding at the size of the entry a step."""
    A = A.astype(np.complex64)
    S, n, _ = A.shape
    at, used = np.arange(S), np.zeros((S, n), bool)
    piv, kof = np.zeros((S, n), int), np.zeros((S, n), int)
    for k in range(n):
        size = np.where(used, -1, np.abs(A[:, :, k].real) + np.abs(A[:, :, k].imag))
        r = np.argmax(size, 1)
        used[at, r], piv[:, k], kof[at, r] = True, r, k
        pinv = (1.0 / A[at, r, k].astype(np.complex128)).astype(np.complex64)
        row = A[at, r].copy()
        A[at, r] = 0
        f = A[:, :, k] * pinv[:, None]
        f[at, r] = -pinv
        A -= f[:, :, None] * row[:, None, :]
        A[:, :, k] = -f
    B = np.empty_like(A)
    for s in range(S):
        B[s][np.ix_(kof[s], piv[s])] = A[s]
    return B


def test_factor_rounding(hz, oracle, monkeypatch):
    """complex64 factors of a long chain of 16-column blocks (a single panel
    each): the one-directional solve on them against the same solve on numpy's
    complex64 inverses.  Both round an entry once a step; 20% for scatter."""
    monkeypatch.setenv("HZ_SOLVE_KERNEL", "fast")
    nx, ny, nz = 16, 40, 12
    ratio = []
    for seed in range(3):
        d, c, b = _layers(hz, nx, ny, nz, seed)
        S, P = hz.Solver(d, c), oracle.Problem(d, c)
        S.factor(hz.abi.PREC_C64)
        D, low, up, slot = extended.blocks(P, nx, ny)
        G = extended.chain(D, low, up, _inverse_c64)
        x = np.empty((nz, ny, nx), np.complex64)
        B = b.reshape(nz, ny, nx)
        for k in range(nz):
            t = [B[k, 0]]
            for j in range(1, ny):
                t.append((B[k, j] - low[j] * (G[j - 1][slot[k]] @ t[-1])).astype(np.complex64))
            x[k, -1] = G[-1][slot[k]] @ t[-1]
            for j in range(ny - 2, -1, -1):
                x[k, j] = G[j][slot[k]] @ (t[j] - up[j] * x[k, j + 1]).astype(np.complex64)
        want = extended.plane_solve(P, d.n, b)
        e_gpu, e_np = extended.error(_solve(S, hz, b, hz.abi.PREC_C64), want), extended.error(x.reshape(-1), want)
        print("factor seed %d: %.3g, numpy %.3g" % (seed, e_gpu, e_np), flush=True)
        ratio.append(e_gpu / e_np)
    assert np.exp(np.mean(np.log(ratio))) < 1.2, ratio


@pytest.mark.parametrize("nx,ny,nz", [(64, 12, 12), (33, 30, 20), (16, 40, 12)])
def test_twisted_rounding(hz, oracle, monkeypatch, nx, ny, nz):
    """The twisted solve against the one-directional one, forward: the same
    operator in the same precision by half as many steps a chain, so no larger
    an error; 15% for scatter (64 x 12 x 12 is mostly layers, where the scalings
    of the symmetric factors are not 1)."""
    ratio = {}
    for seed in range(3):
        d, c, b = _layers(hz, nx, ny, nz, seed)
        S, P = hz.Solver(d, c), oracle.Problem(d, c)
        want = extended.plane_solve(P, d.n, b)
        for prec in (hz.abi.PREC_FP64, hz.abi.PREC_C64):
            S.factor(prec)
            e = {}
            for fam in ("fast", "twist"):
                monkeypatch.setenv("HZ_SOLVE_KERNEL", fam)
                e[fam] = extended.error(_solve(S, hz, b, prec), want)
            print("twisted %d %d %d prec %d seed %d: %.3g, one-directional %.3g" % (nx, ny, nz, prec, seed, e["twist"], e["fast"]), flush=True)
            ratio.setdefault(prec, []).append(e["twist"] / e["fast"])
    for prec, r in ratio.items():
        assert np.exp(np.mean(np.log(r))) < 1.15, (prec, r)


def _strong_layers(hz, n, nz, seed):
    """The reference's geometry: wide strong x/y layers, smooth medium."""
    pr = hz.problem
    d = pr.ref_geometry(n_nopml=n - 40, pml=20, spg=2, nz_nopml=nz - 4, length=(3200.0,) * 3, homo=False)
    rng = np.random.default_rng(seed)
    return d, pr.ref_sound_speed(d), (rng.standard_normal(d.N) + 1j * rng.standard_normal(d.N)).astype(np.complex64)


@pytest.mark.parametrize("nrhs", [1, 9])
def test_adjoint_sums_in_fp64(hz, oracle, monkeypatch, nrhs):
    """complex64 adjoint at a width without streaming kernels: as accurate as the
    one-directional sweep, which sums in FP64.  Half as many steps a chain, so no
    larger an error; 12% for scatter."""
    ratio = []
    for seed in range(3):
        d, c, b = _strong_layers(hz, 52, 8, seed)
        S, P = hz.Solver(d, c), oracle.Problem(d, c)
        S.factor(hz.abi.PREC_C64)
        want = extended.plane_solve(P, d.n, b, adjoint=True)
        e = {}
        for fam in ("fast", ""):
            monkeypatch.setenv("HZ_SOLVE_KERNEL", fam)
            got = _solve(S, hz, np.tile(b, (nrhs, 1)), hz.abi.PREC_C64, adjoint=True)
            e[fam] = max(extended.error(g, want) for g in got)
        print("adjoint seed %d x %d: %.3g, FP64 sums %.3g" % (seed, nrhs, e[""], e["fast"]), flush=True)
        ratio.append(e[""] / e["fast"])
    assert np.exp(np.mean(np.log(ratio))) < 1.12, ratio


def test_adjoint_batches_of_a_streaming_width(hz, monkeypatch):
    """64 columns, 17 vectors on enough planes for groups of 8: all of them with
    FP64 sums, within 12% of the error of single vectors, which have them."""
    monkeypatch.delenv("HZ_SOLVE_KERNEL", raising=False)
    d, c, b = _strong_layers(hz, 64, 40, 1)
    S = hz.Solver(d, c)
    S.factor(hz.abi.PREC_FP64)
    S.factor(hz.abi.PREC_C64)
    want = _solve(S, hz, b, hz.abi.PREC_FP64, adjoint=True)
    one = _solve(S, hz, b, hz.abi.PREC_C64, adjoint=True)
    got = _solve(S, hz, np.tile(b, (17, 1)), hz.abi.PREC_C64, adjoint=True)
    e1 = np.linalg.norm(one - want)
    assert max(np.linalg.norm(g - want) for g in got) < 1.12 * e1


@pytest.mark.parametrize("n,nrhs", [(140, 1), (140, 8), (150, 1), (150, 8), (176, 1), (206, 3), (224, 1)])
def test_adjoint_error_of_wide_planes(hz, monkeypatch, n, nrhs):
    """complex64 adjoint on both sides of the line where the sums go to FP32,
    against the complex128 solve (errors under 1e-13): within 15% of the
    one-directional sweep that sums in FP64."""
    d, c, b = _strong_layers(hz, n, 12, n)
    monkeypatch.delenv("HZ_SOLVE_KERNEL", raising=False)
    S = hz.Solver(d, c)
    S.factor(hz.abi.PREC_FP64)
    S.factor(hz.abi.PREC_C64)
    want = _solve(S, hz, b, hz.abi.PREC_FP64, adjoint=True)
    e = {}
    for fam in ("", "fast"):
        monkeypatch.setenv("HZ_SOLVE_KERNEL", fam)
        got = _solve(S, hz, np.tile(b, (nrhs, 1)), hz.abi.PREC_C64, adjoint=True)
        e[fam] = max(np.linalg.norm(g - want) / np.linalg.norm(want) for g in got)
    print("adjoint %d x %d: %.3g, FP64 sums %.3g" % (n, nrhs, e[""], e["fast"]), flush=True)
    assert e[""] < 1.15 * e["fast"]
