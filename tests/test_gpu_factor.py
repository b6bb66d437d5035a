"""The plane factorisation with blocks inverted in registers, at the edges of
its 16-column panels and 16 x 16 tiles and of its size classes, against the CPU
oracle's pivoted banded LU."""
import numpy as np
import pytest

from conftest import load_pkg

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def hz():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return load_pkg()


def _rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


# one tile and its edges, then both sides of every size class (64, 96, 128, 144,
# 160, 192, 208 columns; complex128 has no class past 144)
WIDTHS = [1, 2, 15, 16, 17, 31, 33, 63, 64, 65, 96, 97, 113, 128, 129, 144, 145, 160, 161, 192, 193, 207, 208, 209]


@pytest.mark.parametrize("nx", WIDTHS)
def test_factor_widths_vs_oracle(hz, oracle, nx):
    """Indefinite planes without layers or shift (every block needs pivoting
    somewhere): the preconditioner and its adjoint, 1e-9 in complex128 and 1e-3
    in complex64 (condition numbers up to about 1e4 times the unit round-off)."""
    print("case factor nx=%d" % nx, flush=True)
    pr = hz.problem
    ny, nz = 5, 4
    d = pr.cube_geometry((nx, ny, nz), 0, 37.0, beta=0.02)
    c = 0.8 + 0.4 * np.random.default_rng(nx).random(d.N)
    S, P = hz.Solver(d, c), oracle.Problem(d, c)
    rng = np.random.default_rng(100 + nx)
    x = rng.standard_normal(d.N) + 1j * rng.standard_normal(d.N)
    xd = torch.from_numpy(x).cuda()
    for prec, tol in ((hz.abi.PREC_FP64, 1e-9), (hz.abi.PREC_C64, 1e-3)):
        S.factor(prec)
        for adj in (False, True):
            e = _rel(S.precond_apply(xd, prec, adjoint=adj).cpu().numpy(), P.precond_apply(x, adjoint=adj))
            assert e < tol, (prec, adj, e)


@pytest.mark.parametrize("nx", WIDTHS)
def test_whole_chain_vs_oracle(hz, oracle, monkeypatch, nx):
    """The same planes through the one-directional factors, forward and adjoint:
    the whole top-down chain, in complex128 (and at 128, 160 and 192 columns)
    completed by the first call from the block where the factorisation stopped."""
    print("case chain nx=%d" % nx, flush=True)
    pr = hz.problem
    ny, nz = 5, 4
    d = pr.cube_geometry((nx, ny, nz), 0, 37.0, beta=0.02)
    c = 0.8 + 0.4 * np.random.default_rng(nx).random(d.N)
    S, P = hz.Solver(d, c), oracle.Problem(d, c)
    rng = np.random.default_rng(100 + nx)
    x = rng.standard_normal(d.N) + 1j * rng.standard_normal(d.N)
    xd = torch.from_numpy(x).cuda()
    for prec, tol in ((hz.abi.PREC_FP64, 1e-9), (hz.abi.PREC_C64, 1e-3)):
        monkeypatch.delenv("HZ_SOLVE_KERNEL", raising=False)
        S.factor(prec)
        monkeypatch.setenv("HZ_SOLVE_KERNEL", "fast")
        for adj in (False, True):
            e = _rel(S.precond_apply(xd, prec, adjoint=adj).cpu().numpy(), P.precond_apply(x, adjoint=adj))
            assert e < tol, (prec, adj, e)
