"""The one-pass Gram-Schmidt dots at vector lengths of less than one block, of a
ragged last block and of more than the fewest blocks, through FGMRES against the
CPU oracle (30 steps: every count of vectors in a group)."""
import numpy as np
import pytest

from conftest import load_pkg

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n", [(7, 6, 5), (17, 16, 15), (24, 22, 28), (41, 40, 43)])
def test_fgmres_dots_vs_oracle(oracle, n):
    """Iterations +-1, residual history 1e-8 and solution 1e-8, the bounds of the
    complex128 FGMRES tests."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    print("case dots", n, flush=True)
    hz = load_pkg()
    pr = hz.problem
    d = pr.cube_geometry(n, (2, 0, 1), pr.omega_for_ppw(0.8, 1.0 / n[0], 6), beta=0.4, pml_c=30.0)
    c = 0.8 + 0.4 * np.random.default_rng(n[0]).random(d.N)
    S, P = hz.Solver(d, c), oracle.Problem(d, c)
    S.factor(hz.abi.PREC_FP64)
    f = pr.point_source(d, (n[0] // 2, n[1] // 2, n[2] // 2), amplitude=1.0)
    u_o, st_o = P.fgmres(f, m=30, rest=3, tol=1e-9)
    u, st = S.fgmres(torch.from_numpy(np.asarray(f)).cuda(), m=30, restarts=3, tol=1e-9, prec=hz.abi.PREC_FP64)
    assert abs(st.iters - st_o.iters) <= 1
    k = min(len(st.hist), len(st_o.hist), 25)
    assert np.allclose(st.hist[:k], st_o.hist[:k], rtol=1e-8)
    if st_o.converged:
        u = u.cpu().numpy()
        assert float(np.linalg.norm(u - u_o) / np.linalg.norm(u_o)) < 1e-8
