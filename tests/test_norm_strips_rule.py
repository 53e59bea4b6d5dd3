"""How many strips a workgroup of normalised rows times many columns takes: host code, held against all forms' measured times."""

import pytest

from bitwise_amd.csrc import ops

GLU, STORE = ops.EPI_SWIGLU_BF16, ops.EPI_F32

# rows, outputs, K, epilogue, microseconds: the kernel for up to 64 rows, and 5, 6, 7 and 8 strips a workgroup
MEASURED = [
    (8, 20608, 2944, GLU, 50.9, 61.6, 49.5, 53.3, 56.0),
    (5, 20812, 2432, GLU, 43.9, 51.8, 42.1, 44.8, 47.3),
    (8, 20812, 2944, GLU, 51.2, 62.6, 49.9, 53.8, 56.6),
    (2, 21000, 2944, GLU, 47.3, 58.1, 46.8, 50.1, 53.6),
    (2, 21504, 2432, GLU, 40.9, 49.4, 40.6, 42.6, 46.0),
    (2, 21760, 4096, GLU, 70.1, 80.0, 67.8, 68.7, 75.3),
    (8, 22100, 2944, GLU, 52.3, 63.5, 52.2, 54.3, 58.5),
    (8, 22100, 4096, GLU, 77.0, 84.4, 71.8, 73.0, 79.8),
    (5, 24281, 4096, GLU, 81.4, 87.4, 78.6, 78.0, 82.2),
    (5, 27000, 2432, GLU, 57.0, 55.7, 59.0, 50.4, 51.0),
    (8, 27000, 4096, GLU, 96.6, 90.5, 97.3, 84.5, 87.6),
    (8, 11008, 2432, GLU, 28.9, 34.6, 23.7, 23.6, 23.9),
    (2, 11008, 4096, GLU, 43.5, 51.2, 38.2, 37.5, 38.8),
    (2, 14336, 2944, GLU, 32.8, 39.3, 41.0, 31.6, 31.3),
    (8, 14336, 4096, GLU, 50.2, 58.0, 60.8, 49.1, 51.3),
    (2, 9728, 2432, GLU, 25.4, 20.7, 20.3, 20.5, 21.3),
    (2, 9728, 4096, GLU, 41.7, 35.4, 33.8, 33.3, 34.5),
    (5, 128192, 4096, STORE, 199.5, 199.7, 202.0, 194.1, 197.7),
    (5, 42000, 2944, STORE, 51.3, 60.8, 49.0, 52.3, 55.1),
    (5, 41624, 4096, STORE, 71.9, 84.8, 71.1, 72.6, 80.9),
]


@pytest.mark.parametrize("rows,columns,inner,epilogue,other,five,six,seven,eight", MEASURED)
def test_the_form_that_is_taken_is_about_the_fastest(rows, columns, inner, epilogue, other, five, six, seven, eight):
    taken = {0: other, 5: five, 6: six, 7: seven, 8: eight}[ops.norm_gemm_strips(rows, columns, inner, epilogue)]
    assert taken <= 1.02 * other and taken <= 1.03 * min(other, five, six, seven, eight)
