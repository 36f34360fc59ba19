"""The multigrid's sweeps at the line lengths where their tiles and the split over the caches change: split from 48 rows a
line on, one tile and no columns beside it up to 64, two tiles above."""
import pytest

torch = pytest.importorskip("torch")

from test_gpu_sweep_parts import check  # noqa: E402
from test_gpu_sweeps import C  # noqa: F401, E402

pytestmark = pytest.mark.gpu


# Owned boxes of 3 x 49 (64 x 4 tiles: split) lines of 47, 48, 49, 63, 64, 65 and 66 rows.  Tolerances of check().
@pytest.mark.parametrize("degree", [1, 3])
@pytest.mark.parametrize("M,p", [((2, 25, 24), 2), ((4, 50, 49), 1), ((2, 25, 25), 2), ((2, 25, 32), 2), ((4, 50, 65), 1),
                                 ((2, 25, 33), 2), ((4, 50, 67), 1)])
def test_line_lengths(C, M, p, degree):  # noqa: F811
    check(C, M, p, degree)
