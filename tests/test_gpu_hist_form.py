"""32-bit counts of a whole histogram in LDS, its window of 16-bit counts, and counts
in global memory, at the sizes where one takes over from the other.

Tiles of 32 chunks (32768 pairs) never take the window.  The bunches are those of
test_gpu_hist_window.py, whose sums are exact in any order, so that every form
gives the same bits."""
import pytest

from test_gpu_hist_window import _gaussian, _same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb", [34560, 34561, 34562, 40001, 40700, 40701, 40702])
@pytest.mark.parametrize("n", [49_152, 49_153, 2_499_998, 2_499_999])
def test_forms_agree(nb, n):
    _same(_gaussian(n), nb, 0, 2.5, (True, True, False, True, True))
