"""The backward over many small views, whose cells take one or two words of
marks each: more words than one pass over them takes, ragged grids of cells
beside a view of one block, and meshlets that show in more cells than one part
holds. Gradients against the FP64 oracle within the suite's 1e-4 and bitwise
reproducible."""
import pytest

from tests import test_gpu_diff_runs as runs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [
    [(16, 16)] * 300,                          # one cell a view, 300 words
    [(32, 32)] * 70 + [(4, 4)],
    [(68, 260)] * 6 + [(16, 16)] * 3,          # 5 x 9 cells of 1 x 2 blocks: two words
    [(260, 260), (20, 4)],                     # 9 x 9 cells of 2 x 2 blocks: three words
])
def test_gradients(gpu_ctx, sizes):
    runs.test_gradients(gpu_ctx, sizes, 0.02)
