"""The FFT kernels that hold radices up to 20, at lengths whose larger radix is
18 or 20 in the x, y and z passes; oracle, inputs and bounds of
test_gpu_fft_sizes."""
import pytest

import test_gpu_fft_sizes as sizes

pytestmark = pytest.mark.gpu

CASES = [("slit", 36, 180, 7), ("bottom", 162, 200, 6), ("nowall", 216, 126, 6), ("slit", 400, 60, 5),
         ("bottom", 324, 100, 5), ("periodic", 90, 20, 162), ("periodic", 200, 216, 9)]


@pytest.mark.parametrize("precision", ["double", "mixed"])
@pytest.mark.parametrize("case", CASES, ids=["%s_%dx%dx%d" % c for c in CASES])
def test_solve_matches_oracle(case, precision):
    sizes.test_solve_matches_oracle(case, precision)
