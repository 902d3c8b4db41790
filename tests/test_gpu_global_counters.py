"""Histograms counted in global memory, with gaps between their lines and without.

Tiles of 32 chunks count there; the window of 16-bit counts (31 chunks) is the
reference.  The bunches are those of test_gpu_hist_window.py, whose sums are exact
in any order, so that both give the same bits; 2200001 particles are 34 tiles
of 32 chunks (gaps by the number of bins), 200001 are 4 (none)."""
import pytest

from test_gpu_hist_window import _gaussian, _same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb", [109_999, 110_000, 110_001, 131_072, 149_999, 150_000, 150_001])
@pytest.mark.parametrize("n", [200_001, 2_200_001])
@pytest.mark.parametrize("half", [2.5, 30.0])
def test_counts_in_global_memory(nb, n, half):
    _same(_gaussian(n), nb, 31, half, (True, True, False, True, True))
