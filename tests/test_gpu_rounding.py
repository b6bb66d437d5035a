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
