"""Groups of 8 complex64 right-hand sides on the dense twisted blocks, over the
widths where their tiles and wave split have edges, the shortest chains, short
last groups and a batch past one workspace, against the CPU oracle."""
import numpy as np
import pytest

from conftest import load_pkg

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


# one tile and two (ragged and full), one tile row a wave and two; the last width
# with FP64 adjoint sums and the first without, the widest; ny = 2 has no bottom end
@pytest.mark.parametrize("nx,ny,nz,nrhs", [
    (1, 3, 3, 8), (7, 2, 4, 8), (16, 5, 3, 9), (17, 4, 5, 16), (31, 6, 4, 11), (64, 3, 5, 8), (96, 5, 3, 24), (97, 4, 4, 8),
    (129, 3, 4, 15), (144, 5, 3, 8), (145, 4, 4, 10), (177, 2, 3, 9), (193, 3, 3, 9), (208, 5, 4, 8), (33, 4, 3, 66)])
def test_rows_twisted_vs_oracle(oracle, monkeypatch, nx, ny, nz, nrhs):
    """Forward and adjoint through the preconditioner within 1e-4, the complex64
    preconditioner's bound elsewhere; against the twisted solve of single
    vectors, on the same factors, within 1e-5."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    print("case rows twisted %d %d %d x %d" % (nx, ny, nz, nrhs), flush=True)
    hz = load_pkg()
    pr = hz.problem
    d = pr.cube_geometry((nx, ny, nz), (min(4, (nx - 1) // 2), 0, 1 if nz > 2 else 0),
                         pr.omega_for_ppw(0.8, 1.0 / max(nx, 8), 8), beta=0.5, pml_c=30.0)
    rng = np.random.default_rng(nx + nrhs)
    c = 0.8 + 0.4 * rng.random(d.N)
    monkeypatch.setenv("HZ_SOLVE_KERNEL", "rows")
    S, P = hz.Solver(d, c), oracle.Problem(d, c)
    S.factor(hz.abi.PREC_C64)
    x = rng.standard_normal((nrhs, d.N)) + 1j * rng.standard_normal((nrhs, d.N))
    xd = torch.from_numpy(x).cuda()
    for adj in (False, True):
        monkeypatch.setenv("HZ_SOLVE_KERNEL", "rows")
        got = S.precond_apply(xd, hz.abi.PREC_C64, adjoint=adj).cpu().numpy()
        monkeypatch.setenv("HZ_SOLVE_KERNEL", "twist")
        one = S.precond_apply(xd, hz.abi.PREC_C64, adjoint=adj).cpu().numpy()
        for q in range(nrhs):
            assert np.linalg.norm(got[q] - one[q]) < 1e-5 * np.linalg.norm(one[q]), (adj, q)
            if q < 4 or q >= nrhs - 2:
                want = P.precond_apply(x[q], adjoint=adj)
                e = float(np.linalg.norm(got[q] - want) / np.linalg.norm(want))
                assert e < 1e-4, (adj, q, e)
