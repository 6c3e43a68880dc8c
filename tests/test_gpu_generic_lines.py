"""The element operator of blocks of any size on both sides of the lines between its two kernels:
few and many elements, short and long rows, 16 rows an element and more, rows of 16 whose
last round of workgroups is nearly empty; against the oracle, as the other cases."""
import pytest

from test_gpu_generic_rows import se, test_operator as _operator  # noqa: F401

pytestmark = pytest.mark.gpu


# the last but one before each line, or the first after it
@pytest.mark.parametrize("nr,ns,Ex,Ey", [
    (24, 8, 1399, 1), (24, 8, 35, 40), (16, 7, 20, 70), (20, 3, 3, 467), (12, 8, 89, 23),
    (12, 8, 64, 32), (9, 7, 1, 2049), (13, 5, 61, 34), (15, 4, 33, 63), (7, 6, 64, 33),
    (16, 15, 36, 39), (18, 12, 1401, 1), (30, 2, 28, 50), (8, 5, 3, 2), (20, 2, 5, 7),
    (7, 9, 48, 48), (5, 16, 64, 64), (12, 16, 80, 79), (12, 16, 64, 64), (17, 16, 38, 37)])
def test_operator_at_the_line(se, nr, ns, Ex, Ey):   # noqa: F811
    _operator(se, nr, ns, Ex, Ey)
