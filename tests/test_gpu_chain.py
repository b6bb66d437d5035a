"""The one-directional factor chain beside the twisted factors: complete after the
factorisation where a later call would else pay for the rest or be refused, and
the same blocks where it is completed later."""
import ctypes as C

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


def _box(hz, n):
    d = hz.problem.cube_geometry(n, tuple(min(6, v // 4) for v in n), 40.0, beta=0.5, pml_c=30.0)
    return d, 0.8 + 0.4 * np.random.default_rng(n[0]).random(d.N)


def _vectors(d, nrhs, prec, hz, seed=3):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((nrhs, d.N)) + 1j * rng.standard_normal((nrhs, d.N))
    return torch.from_numpy(x.astype(np.complex128 if prec == hz.abi.PREC_FP64 else np.complex64)).cuda()


def _replays(hz, S, prec, x0, want):
    """Plane solve of x0 captured on a stream of torch's and replayed four times
    between eager copies: every replay is bit for bit `want`."""
    lib, st, x = hz.abi.lib(), torch.cuda.Stream(), x0.clone()
    torch.cuda.synchronize()
    hz.abi.check(lib.hz_problem_set_stream(S.h, C.c_void_p(st.cuda_stream)), "hz_problem_set_stream")
    try:
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=st, capture_error_mode="thread_local"):
            rc = lib.hz_plane_solve(S.h, int(prec), 0, x0.shape[0], C.c_void_p(x.data_ptr()))
        hz.abi.check(rc, "hz_plane_solve under capture")
        with torch.cuda.stream(st):
            for _ in range(4):
                x.copy_(x0)
                g.replay()
                st.synchronize()
                assert torch.equal(x, want)
    finally:
        hz.abi.check(lib.hz_problem_set_stream(S.h, C.c_void_p(0)), "hz_problem_set_stream")


# complex64 groups by default: one way on a short chain, from both ends on a chain
# that stopped halfway; a forced family in either precision and a tuned one
@pytest.mark.parametrize("n,prec,nrhs,how", [
    ((112, 6, 66), 1, 8, "untuned"), ((64, 5, 128), 1, 16, "untuned"), ((112, 9, 66), 1, 8, "untuned"),
    ((100, 6, 8), 1, 8, "forced"),
    ((140, 6, 5), 0, 2, "forced"), ((140, 6, 5), 0, 2, "tuned")])
def test_first_call_after_a_factorisation_can_be_captured(hz, tmp_path, monkeypatch, n, prec, nrhs, how):
    d, c = _box(hz, n)
    monkeypatch.delenv("HZ_SOLVE_KERNEL", raising=False)
    monkeypatch.delenv("HZ_FACTOR_FULL", raising=False)
    if how == "forced":
        monkeypatch.setenv("HZ_SOLVE_KERNEL", "mfma" if prec == hz.abi.PREC_C64 else "fast")
    if how == "tuned":
        line = " | %d 1 16\n" % hz.abi.SOLVE_CHUNKED
        key = "gfx950 %d %d %d %d %d" % (*n, prec, nrhs)
        (tmp_path / "t").write_text(key + line + key + " set 2" + line)
        monkeypatch.setenv("HZ_TUNE_CACHE", str(tmp_path / "t"))
    x = _vectors(d, nrhs, prec, hz)
    E, S = hz.Solver(d, c), hz.Solver(d, c)
    for s in (E, S):
        s.factor(prec)
        if how == "tuned":
            assert s.autotune(prec, nrhs)["from_cache"]
            s.factor(prec)
    want = E.plane_solve(x.clone(), prec)  # eager, on a problem of its own
    _replays(hz, S, prec, x, want)


@pytest.mark.parametrize("prec", [0, 1])
def test_untuned_capture_on_an_incomplete_chain(hz, monkeypatch, prec):
    """128 columns: nothing has completed the chain, and an untuned captured call
    of any size takes the twisted solve."""
    d, c = _box(hz, (128, 6, 7))
    monkeypatch.delenv("HZ_FACTOR_FULL", raising=False)
    x = _vectors(d, 8, prec, hz)
    E, S = hz.Solver(d, c), hz.Solver(d, c)
    monkeypatch.setenv("HZ_SOLVE_KERNEL", "twist")
    E.factor(prec)
    want = E.plane_solve(x.clone(), prec)
    monkeypatch.delenv("HZ_SOLVE_KERNEL")
    S.factor(prec)
    _replays(hz, S, prec, x, want)


@pytest.mark.parametrize("prec,n", [(1, (160, 20, 9)), (0, (160, 20, 9)), (0, (129, 9, 6)), (0, (64, 12, 6)), (1, (230, 8, 5)), (0, (230, 7, 5))])
def test_chain_completed_later_is_the_same(hz, monkeypatch, prec, n):
    """Every one-directional family on a factorisation that stopped halfway, each
    on a problem of its own (the family's first call completes the chain), equals
    the one on a factorisation of the whole chain bit for bit."""
    d, c = _box(hz, n)
    fams = [("fast", 1, False), ("fast", 1, True), ("mr", 3, False), ("dma", 1, False), ("sym", 1, False), ("sym", 1, True)]
    if prec == hz.abi.PREC_C64:
        fams += [("mfma", 9, False), ("mfma", 9, True)]
    monkeypatch.delenv("HZ_SOLVE_KERNEL", raising=False)
    monkeypatch.setenv("HZ_FACTOR_FULL", "1")
    full = hz.Solver(d, c)
    full.factor(prec)
    monkeypatch.delenv("HZ_FACTOR_FULL")
    for fam, nrhs, adj in fams:
        monkeypatch.delenv("HZ_SOLVE_KERNEL", raising=False)
        lazy = hz.Solver(d, c)
        lazy.factor(prec)
        monkeypatch.setenv("HZ_SOLVE_KERNEL", fam)
        x = _vectors(d, nrhs, prec, hz)
        assert torch.equal(lazy.plane_solve(x.clone(), prec, adjoint=adj), full.plane_solve(x.clone(), prec, adjoint=adj)), (fam, adj)


@pytest.mark.parametrize("prec,n", [(1, (140, 10, 8)), (0, (129, 7, 9)), (0, (128, 8, 6)), (1, (60, 5, 6))])
def test_factors_where_the_twisted_ones_do_not_fit(hz, oracle, monkeypatch, prec, n):
    """With room for the dense factors but not for the twisted ones beside them
    the factorisation keeps the dense ones (and what the packed widths always
    held), and every call is that of a problem without twisted factors; with room
    again it has them."""
    d, c = _box(hz, n)
    monkeypatch.delenv("HZ_SOLVE_KERNEL", raising=False)
    monkeypatch.delenv("HZ_FACTOR_FULL", raising=False)
    monkeypatch.setenv("HZ_NO_TWIST", "1")
    plain = hz.Solver(d, c)
    plain.factor(prec)
    monkeypatch.delenv("HZ_NO_TWIST")
    nx, ny, _ = n
    dense = plain.slots()[0] * ny * nx * nx * (8 if prec == hz.abi.PREC_C64 else 16)
    S = hz.Solver(d, c)
    monkeypatch.setenv("HZ_FACTOR_BUDGET", str(int(1.5 * dense)))
    S.factor(prec)
    assert S.factor_bytes() == plain.factor_bytes()
    for adj in (False, True):
        for nrhs in (1, 3, 9):
            x = _vectors(d, nrhs, prec, hz)
            assert torch.equal(S.plane_solve(x.clone(), prec, adjoint=adj), plain.plane_solve(x.clone(), prec, adjoint=adj))
    x = np.random.default_rng(5).standard_normal(d.N) + 0j
    got = S.precond_apply(torch.from_numpy(x).cuda(), prec).cpu().numpy()
    want = oracle.Problem(d, c).precond_apply(x)
    assert np.linalg.norm(got - want) / np.linalg.norm(want) < (1e-4 if prec == hz.abi.PREC_C64 else 1e-10)
    monkeypatch.delenv("HZ_FACTOR_BUDGET")
    S.factor(prec)
    assert S.factor_bytes() > dense
    y = _vectors(d, 1, prec, hz)
    monkeypatch.setenv("HZ_SOLVE_KERNEL", "twist")
    fresh = hz.Solver(d, c)
    fresh.factor(prec)
    assert torch.equal(S.plane_solve(y.clone(), prec), fresh.plane_solve(y.clone(), prec))


def test_complex128_holds_no_idle_packed_copy(hz, monkeypatch):
    """At 128 columns untuned complex128 calls read the twisted factors alone: the
    packed copy of the one-directional ones is there from the first call of a
    family that reads it, with the same numbers as ever."""
    d, c = _box(hz, (128, 8, 6))
    prec = hz.abi.PREC_FP64
    monkeypatch.delenv("HZ_SOLVE_KERNEL", raising=False)
    monkeypatch.delenv("HZ_FACTOR_FULL", raising=False)
    S = hz.Solver(d, c)
    S.factor(prec)
    slots = S.slots()[0]
    assert S.factor_bytes() == slots * 8 * 16 * (128 * 128 + 36 * 256)  # dense blocks, 36 of 64 tiles
    x = _vectors(d, 1, prec, hz)
    monkeypatch.setenv("HZ_SOLVE_KERNEL", "sym")
    full = hz.Solver(d, c)
    full.factor(prec)
    assert torch.equal(S.plane_solve(x.clone(), prec), full.plane_solve(x.clone(), prec))
    assert S.factor_bytes() == full.factor_bytes()


@pytest.mark.parametrize("twisted", [False, True])
def test_released_factors_are_an_error(hz, monkeypatch, twisted):
    """Dense factors released by a compression and the compressed form dropped
    afterwards: nothing is left to solve with, and every call says so until the
    next factorisation."""
    d, c = _box(hz, (128, 8, 6))
    monkeypatch.delenv("HZ_SOLVE_KERNEL", raising=False)
    prec = hz.abi.PREC_C64
    S = hz.Solver(d, c)
    S.factor(prec)
    x = _vectors(d, 1, prec, hz)
    want = S.plane_solve(x.clone(), prec)
    S.compress(prec, eps=1e-4, smallsize=7, free_dense=True, twisted=twisted)
    S.compress(prec, eps=-1.0, smallsize=7)
    for call in (lambda: S.plane_solve(x.clone(), prec), lambda: S.plane_solve(x.clone(), prec, adjoint=True),
                 lambda: S.autotune(prec, 8)):
        with pytest.raises(hz.abi.HzError):
            call()
    S.factor(prec)
    assert torch.equal(S.plane_solve(x.clone(), prec), want)
