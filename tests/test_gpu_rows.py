"""Groups of 8 complex64 right-hand sides on the matrix cores, over the widths and
group sizes where their tiles, their wave split and a last short group have edges,
against the CPU oracle."""
import numpy as np
import pytest

from conftest import load_pkg

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


# one tile and two (ragged and full), one tile row a wave and two, the widest; an
# odd and an even number of planes (one or two of them with a slot alone)
@pytest.mark.parametrize("nx,ny,nz,nrhs", [
    (7, 2, 4, 8), (16, 5, 3, 9), (17, 4, 5, 16), (31, 6, 4, 11), (97, 4, 4, 8), (128, 5, 3, 17), (129, 3, 4, 15),
    (160, 4, 6, 8), (193, 3, 3, 9), (208, 3, 4, 8), (241, 3, 3, 10), (256, 2, 4, 8)])
def test_rows_vs_oracle(oracle, monkeypatch, nx, ny, nz, nrhs):
    """Forward and adjoint through the preconditioner within 1e-4, the
    complex64 preconditioner's bound elsewhere."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    print("case rows %d %d %d x %d" % (nx, ny, nz, nrhs), flush=True)
    hz = load_pkg()
    pr = hz.problem
    d = pr.cube_geometry((nx, ny, nz), (min(4, (nx - 1) // 2), 0, 1 if nz > 2 else 0),
                         pr.omega_for_ppw(0.8, 1.0 / max(nx, 8), 8), beta=0.5, pml_c=30.0)
    rng = np.random.default_rng(nx + nrhs)
    c = 0.8 + 0.4 * rng.random(d.N)
    monkeypatch.setenv("HZ_SOLVE_KERNEL", "mfma")
    S, P = hz.Solver(d, c), oracle.Problem(d, c)
    S.factor(hz.abi.PREC_C64)
    x = rng.standard_normal((nrhs, d.N)) + 1j * rng.standard_normal((nrhs, d.N))
    for adj in (False, True):
        got = S.precond_apply(torch.from_numpy(x).cuda(), hz.abi.PREC_C64, adjoint=adj).cpu().numpy()
        for q in range(nrhs):
            want = P.precond_apply(x[q], adjoint=adj)
            e = float(np.linalg.norm(got[q] - want) / np.linalg.norm(want))
            assert e < 1e-4, (adj, q, e)
