"""z-FFTs of two run-time factors: every factor that is built as the larger one (4
to 400 points, complex128 to the 292 that its general kernel takes) and every smaller partner of the odd primes, ragged lines, several
right-hand sides, against numpy."""
import numpy as np
import pytest

from conftest import load_pkg

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


# 4 = 2 x 2 .. 400 = 20 x 20; past them 2 x 23 and 14 x 19, which stay on the
# general kernel
@pytest.mark.parametrize("nz", [4, 6, 9, 10, 15, 20, 21, 28, 30, 33, 39, 42, 48, 49, 54, 63, 70, 77, 81, 90, 91, 100, 110,
                                121, 126, 130, 132, 143, 144, 150, 156, 169, 182, 195, 196, 208, 210, 225, 240, 256, 270,
                                280, 288, 300, 324, 360, 400, 46, 266])
def test_fft_two_factors_vs_numpy(nz):
    """Relative errors under 1e-14 (complex128) and 2e-6 (complex64), the bounds
    of the other z-FFT tests."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    print("case fft two nz=%d" % nz, flush=True)
    hz = load_pkg()
    d = hz.problem.cube_geometry((7, 5, nz), (0, 0, 0), 6.0)  # 35 lines: a full workgroup and a ragged one
    S = hz.Solver(d, np.ones(d.N))
    rng = np.random.default_rng(nz)
    X = rng.standard_normal((2, nz, 35)) + 1j * rng.standard_normal((2, nz, 35))
    x = torch.from_numpy(X.reshape(2, -1)).cuda()
    want = {-1: np.fft.fft(X, axis=1).reshape(2, -1), 1: np.fft.ifft(X, axis=1).reshape(2, -1)}
    for prec, tol in ((hz.abi.PREC_FP64, 1e-14), (hz.abi.PREC_C64, 2e-6)):
        if nz > 292 and prec == hz.abi.PREC_FP64:
            with pytest.raises(hz.abi.HzError):
                S.fft_z(x, -1, prec)
            continue
        for sign in (-1, 1):
            got = S.fft_z(x, sign, prec).cpu().numpy()
            e = float(np.linalg.norm(got - want[sign]) / np.linalg.norm(want[sign]))
            assert e < tol, (prec, sign, e)
