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


# complex128: past 292 points only the 8-line kernel fits; complex64: below 32
# the general kernel is the only one
@pytest.mark.parametrize("prec,nz", [(0, 292), (0, 300), (0, 320), (0, 324), (0, 360), (0, 400), (1, 28), (1, 30), (1, 32), (1, 400)])
def test_autotune_z_lengths(hz, monkeypatch, prec, nz):
    """Tuning offers a z-FFT only where it exists, and the tuned transform is
    numpy's (1e-14 complex128, 2e-6 complex64, the z-FFTs' bounds elsewhere)."""
    monkeypatch.delenv("HZ_TUNE_CACHE", raising=False)
    d = hz.problem.cube_geometry((6, 5, nz), 0, 6.0)
    S = hz.Solver(d, np.ones(d.N))
    S.factor(prec)
    t = S.autotune(prec, 1)
    if prec == hz.abi.PREC_FP64 and nz > 292:
        assert t["fft_lines"] == 8
    if prec == hz.abi.PREC_C64 and nz < 32:
        assert t["fft_lines"] in (8, 16, 32)
    X = _rand((nz, 30), nz)
    want = np.fft.fft(X, axis=0).reshape(-1)
    got = S.fft_z(torch.from_numpy(X.reshape(-1)).cuda(), -1, prec).cpu().numpy()
    assert np.linalg.norm(got - want) / np.linalg.norm(want) < (1e-14 if prec == hz.abi.PREC_FP64 else 2e-6)
