"""The autotuner over the lengths, widths and batches where its candidates
differ from what untuned calls take."""
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


def _rand(shape, seed):
    rng = np.random.default_rng(seed)
    return rng.standard_normal(shape) + 1j * rng.standard_normal(shape)


# complex128: past 288 points only the 8-line kernel fits; complex64: below 32
# the general kernel is the only one
@pytest.mark.parametrize("prec,nz", [(0, 288), (0, 300), (0, 320), (0, 324), (0, 360), (0, 400), (1, 28), (1, 30), (1, 32), (1, 400)])
def test_autotune_z_lengths(hz, monkeypatch, prec, nz):
    """Tuning offers a z-FFT only where it exists, and the tuned transform is
    numpy's (1e-14 complex128, 2e-6 complex64, the z-FFTs' bounds elsewhere)."""
    monkeypatch.delenv("HZ_TUNE_CACHE", raising=False)
    d = hz.problem.cube_geometry((6, 5, nz), 0, 6.0)
    S = hz.Solver(d, np.ones(d.N))
    S.factor(prec)
    t = S.autotune(prec, 1)
    if prec == hz.abi.PREC_FP64 and nz > 288:
        assert t["fft_lines"] == 8
    if prec == hz.abi.PREC_C64 and nz < 32:
        assert t["fft_lines"] in (8, 16, 32)
    X = _rand((nz, 30), nz)
    want = np.fft.fft(X, axis=0).reshape(-1)
    got = S.fft_z(torch.from_numpy(X.reshape(-1)).cuda(), -1, prec).cpu().numpy()
    assert np.linalg.norm(got - want) / np.linalg.norm(want) < (1e-14 if prec == hz.abi.PREC_FP64 else 2e-6)


def _box(hz, n, seed=4):
    d = hz.problem.cube_geometry(n, tuple(min(8, v // 4) for v in n), 40.0, beta=0.5, pml_c=30.0)
    return d, 0.8 + 0.4 * np.random.default_rng(seed).random(d.N)


@pytest.mark.parametrize("n,prec,nrhs", [((128, 40, 24), 0, 8), ((100, 40, 24), 0, 9), ((140, 40, 24), 1, 8), ((230, 24, 12), 1, 8)])
def test_tuned_solve_no_slower_than_untuned(hz, monkeypatch, n, prec, nrhs):
    """Eight and more vectors, where the untuned kernel is none of the families
    the tuner times for groups: the tuned call keeps it (a quarter more for the
    scatter of the timings; the families take 1.3 to 10 times as long here)."""
    monkeypatch.delenv("HZ_TUNE_CACHE", raising=False)
    d, c = _box(hz, n)
    S = hz.Solver(d, c)
    S.factor(prec)
    dt = torch.complex128 if prec == hz.abi.PREC_FP64 else torch.complex64
    x = torch.from_numpy(_rand((nrhs, d.N), 1)).to(dt).cuda()

    def best():
        t = []
        for _ in range(8):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            y = x.clone()
            e0.record()
            S.plane_solve(y, prec)
            e1.record()
            torch.cuda.synchronize()
            t.append(e0.elapsed_time(e1))
        return min(t)

    untuned = best()
    t = S.autotune(prec, nrhs)
    tuned = best()
    print("%s prec %d x %d: untuned %.3f ms, tuned %.3f (%s)" % (n, prec, nrhs, untuned, tuned, t), flush=True)
    assert tuned < 1.25 * untuned


def test_tune_cache_of_earlier_kernels(hz, tmp_path, monkeypatch):
    """An entry without the mark of the present set of kernels is tuned again;
    what is written then is taken by a new problem of the same grid, family and
    all, and gives the same numbers."""
    d, c = _box(hz, (128, 12, 8))
    cache = tmp_path / "tune.txt"
    cache.write_text("gfx950 128 12 8 0 8 | %d 1 16\n" % hz.abi.SOLVE_CHUNKED)
    monkeypatch.setenv("HZ_TUNE_CACHE", str(cache))
    x = torch.from_numpy(_rand((8, d.N), 2)).cuda()
    out = []
    for first in (True, False):
        S = hz.Solver(d, c)
        S.factor(hz.abi.PREC_FP64)
        t = S.autotune(hz.abi.PREC_FP64, 8)
        assert t["from_cache"] == (not first)
        out.append((t["solve_kernel"], t["group_cap"], t["fft_lines"], S.precond_apply(x, hz.abi.PREC_FP64).cpu().numpy()))
    assert out[0][:3] == out[1][:3] and np.array_equal(out[0][3], out[1][3])
