"""FFT3D MATVEC at every padded axis length 2N, N = 2^a 3^b 5^c 7^d with a
factor 7 from 14 to 252, on each axis in turn, and with z runs padded to half
lines (NZ = 36 to 100), against the oracle under the bar of the other axis
lengths (1e-5 relative L2)."""
import pytest

import test_gpu_axis_lengths as lengths

pytestmark = pytest.mark.gpu


def smooth7(n):
    for f in (2, 3, 5, 7):
        while n % f == 0:
            n //= f
    return n == 1


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("n", [n for n in range(14, 257, 7) if smooth7(n)])
def test_axis_length_with_a_factor_7_matches_oracle(lib, n, axis):
    lengths.test_axis_length_matches_oracle(lib, n, axis)


@pytest.mark.parametrize("n", [36, 40, 50, 54, 72, 100])
def test_half_line_padding_matches_oracle(lib, n):
    lengths.test_axis_length_matches_oracle(lib, n, 2)
