"""The twisted plane solve (default for few right-hand sides and in complex128,
forward and adjoint) over the widths where its 16 x 16 tiles, its wave split (even and
odd tile counts) and its chains have edges, against the CPU oracle."""
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


def _case(hz, mode, nx, ny, nz):
    pr = hz.problem
    if mode == "s7":
        d = pr.cube_geometry((nx, ny, nz), (min(4, (nx - 1) // 2), 0, 1 if nz > 2 else 0),
                             pr.omega_for_ppw(0.8, 1.0 / max(nx, 8), 8), beta=0.5, pml_c=30.0)
        return d, 0.8 + 0.4 * np.random.default_rng(nx + ny).random(d.N)
    d = pr.ref_geometry(n_nopml=nx - 8, pml=4, spg=2, nz_nopml=nz - 4, length=(240.0,) * 3, homo=False)
    d = d.replace(n=(nx, ny, nz), l=(d.l[0], d.l[0] * ny / nx, d.l[2]), h=(d.h[0], d.h[0], d.h[2]))
    return d, pr.ref_sound_speed(d)


# every tile count 1..16, on both sides of a tile edge or ragged; chains of 2
# and 3 blocks and longer ones; single-plane slots (k = 0, nz / 2), odd nz
CASES = [("s7", nx, ny, nz) for nx, ny, nz in (
    (1, 3, 3), (7, 2, 4), (16, 5, 3), (17, 6, 4), (33, 3, 5), (48, 4, 4), (49, 7, 3), (65, 6, 4), (81, 5, 3), (100, 4, 4),
    (112, 3, 3), (113, 6, 4), (130, 5, 3), (145, 4, 4), (161, 3, 3), (177, 5, 4), (193, 4, 3), (209, 3, 4), (223, 4, 3),
    (225, 5, 3), (239, 4, 4), (256, 3, 3))] + [("ref", 30, 12, 9), ("ref", 77, 14, 8), ("ref", 139, 12, 7)]


@pytest.mark.parametrize("mode,nx,ny,nz", CASES)
def test_tri_vs_oracle(hz, oracle, mode, nx, ny, nz):
    """One and three right-hand sides, forward and adjoint, through the
    preconditioner: 1e-4 in complex64 and 1e-10 in complex128, the
    preconditioners' bounds elsewhere."""
    print("case tri %s %d %d %d" % (mode, nx, ny, nz), flush=True)
    d, c = _case(hz, mode, nx, ny, nz)
    S, P = hz.Solver(d, c), oracle.Problem(d, c)
    tol = {hz.abi.PREC_C64: 1e-4, hz.abi.PREC_FP64: 1e-10}
    for prec in tol:
        S.factor(prec)
    rng = np.random.default_rng(nx)
    x = rng.standard_normal((3, d.N)) + 1j * rng.standard_normal((3, d.N))
    for adj in (False, True):
        want = [P.precond_apply(v, adjoint=adj) for v in x]
        for prec in tol:
            for nrhs in (1, 3):
                got = S.precond_apply(torch.from_numpy(x[:nrhs]).cuda(), prec, adjoint=adj).cpu().numpy()
                for q in range(nrhs):
                    assert _rel(got[q], want[q]) < tol[prec], (adj, prec, nrhs, q, _rel(got[q], want[q]))


def test_tri_widths_past_the_tiles(hz, oracle):
    """257 columns: no twisted factors, the one-directional kernels as before."""
    d, c = _case(hz, "s7", 257, 3, 3)
    S, P = hz.Solver(d, c), oracle.Problem(d, c)
    x = np.random.default_rng(1).standard_normal(d.N) + 0j
    for prec, tol in ((hz.abi.PREC_C64, 1e-4), (hz.abi.PREC_FP64, 1e-10)):
        S.factor(prec)
        for adj in (False, True):
            got = S.precond_apply(torch.from_numpy(x).cuda(), prec, adjoint=adj).cpu().numpy()
            assert _rel(got, P.precond_apply(x, adjoint=adj)) < tol


# complex64 batches: single vectors while no XCD has more than 32 workgroups,
# ceil(2 slots / 8) x vectors (slots: nz // 2 + 1), groups beyond, on the
# one-directional factors for fewer than 8 lines; always those at 128 columns
@pytest.mark.parametrize("nx,ny,nz,nrhs,fam", [
    (140, 10, 12, 8, "twist"), (100, 6, 24, 8, "twist"), (100, 8, 24, 9, "rows"), (208, 8, 40, 12, "rows"),
    (97, 5, 9, 16, "twist"), (97, 9, 9, 17, "rows"), (128, 6, 12, 8, "mfma"), (96, 6, 12, 8, "twist"), (48, 8, 40, 8, "rows"),
    (150, 7, 24, 9, "mfma"), (209, 4, 40, 8, "twist")])
def test_groups_take_the_faster_kernel(hz, monkeypatch, nx, ny, nz, nrhs, fam):
    """Untuned batches, forward and adjoint, are bit for bit the batches of the
    family the rule names."""
    d, c = _case(hz, "s7", nx, ny, nz)
    monkeypatch.delenv("HZ_SOLVE_KERNEL", raising=False)
    S = hz.Solver(d, c)
    S.factor(hz.abi.PREC_C64)
    rng = np.random.default_rng(nz)
    x = torch.from_numpy((rng.standard_normal((nrhs, d.N)) + 1j * rng.standard_normal((nrhs, d.N))).astype(np.complex64)).cuda()
    for adj in (False, True):
        monkeypatch.delenv("HZ_SOLVE_KERNEL", raising=False)
        got = S.plane_solve(x.clone(), hz.abi.PREC_C64, adjoint=adj)
        monkeypatch.setenv("HZ_SOLVE_KERNEL", fam)
        assert torch.equal(got, S.plane_solve(x.clone(), hz.abi.PREC_C64, adjoint=adj)), adj
