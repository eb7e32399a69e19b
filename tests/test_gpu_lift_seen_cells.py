"""Error lifting: grids of which the image shows all, some or none, with numbers of cells around the 64 x 256 of a group of
stretches and the 4 neighbours that stay together in one. Counts are whole numbers; a value is a sum of float terms in double,
rounded once, as the oracle's is."""
import numpy as np
import pytest

from tests.test_gpu_lift_rows import _both, _camera, _lift
from vet_amd import synthetic
from vet_amd.synthetic import ViewSpec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [63, 255, 257, 1025, 16383, 16384, 16385, 16640, 33000])
@pytest.mark.parametrize("z", [3.0, 0.2])  # in front of the grid; inside it, with most cells behind the camera or beside the image
def test_cells_of_all_stretches(cells, z, rasterizer, oracle):
    print(f"[case] lift {cells} cells, camera at {z}", flush=True)
    w, h, edge = 96, 64, 0.07
    mn, ln = synthetic.cell_grid(np.array([[-1.15, -1.15, -1.15], [1.12, 1.12, 1.12]]), edge)
    assert len(mn) >= 33000
    keep = np.random.RandomState(cells).permutation(len(mn))[:cells]
    keep = np.sort(keep) if cells % 2 else keep
    poses, intr = _camera(w, h, (0.01, -0.02, z), 0.3)
    _both(rasterizer, oracle, mn[keep], ln[keep], ViewSpec(w, h), poses, intr, synthetic.error_image(cells, 2, h, w), 2)


def test_no_cell_is_seen(rasterizer):
    w, h = 64, 48
    mn, ln = synthetic.cell_grid(np.array([[-1.0, -1.0, -1.0], [0.9, 0.9, 0.9]]), 0.1)
    poses, intr = _camera(w, h, (0.0, 0.0, -5.0))
    val, cnt = _lift(rasterizer, mn, ln, ViewSpec(w, h), poses, intr, synthetic.error_image(1, 3, h, w), 0)
    assert not val.any() and not cnt.any()
