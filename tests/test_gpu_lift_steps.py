"""Error lifting: image widths around the 1024 pixels of a step of the running sums, and numbers of cells around the 32 of a
workgroup, with few and with many rows for its waves. Counts are whole numbers; a value is a sum of float terms in double,
rounded once, as the oracle's is, so that they differ by a rounding or two."""
import numpy as np
import pytest

from tests.test_gpu_lift_rows import _both, _camera
from vet_amd import synthetic
from vet_amd.synthetic import ViewSpec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,cells", [(1023, 17, 31), (1024, 70, 32), (1025, 300, 33), (2047, 40, 1), (2048, 640, 65), (2049, 9, 64)])
def test_widths_and_cell_counts(w, h, cells, rasterizer, oracle):
    print(f"[case] lift steps {w}x{h} {cells} cells", flush=True)
    mn, ln = synthetic.cell_grid(np.array([[-1.0, -1.0, -1.0], [0.98, 0.98, 0.98]]) + 0.01, 0.25)
    keep = np.argsort(np.abs(mn[:, 1] + 0.125), kind="stable")[::2][:cells]  # the height of the image's middle first: all are seen
    poses, intr = _camera(w, h, (0.0, 0.0, 2.0), 0.2, f=0.5 * w)
    _both(rasterizer, oracle, mn[keep], ln[keep], ViewSpec(w, h), poses, intr, synthetic.error_image(5, 3, h, w), 0)
