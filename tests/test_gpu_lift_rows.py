"""Error lifting by rows, where the row bounds can go wrong: faces seen edge-on (lines through pixel centres), cells that
touch the camera plane (tested pixel by pixel), image widths around the steps of the running sums, images that take
several bands, pixels that are not finite."""
import numpy as np
import pytest
import torch

from vet_amd import synthetic
from vet_amd.synthetic import ViewSpec

pytestmark = pytest.mark.gpu


def _lift(rasterizer, mn, ln, view, poses, intr, img, border):
    dev = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (mn, ln, poses, intr, img)]
    val = torch.zeros(len(mn), device="cuda")
    cnt = torch.zeros(len(mn), dtype=torch.int32, device="cuda")
    rasterizer.lift_error(dev[0], dev[1], val, cnt, view, dev[2], dev[3], dev[4], border_pixels=border)
    torch.cuda.synchronize()
    return val.cpu().numpy(), cnt.cpu().numpy()


def _both(rasterizer, oracle, mn, ln, view, poses, intr, img, border):
    val, cnt = _lift(rasterizer, mn, ln, view, poses, intr, img, border)
    want_v, want_c = np.zeros(len(mn), np.float32), np.zeros(len(mn), np.int32)
    oracle.lift_error(mn, ln, want_v, want_c, view, poses, intr, img, border_pixels=border, num_threads=16)
    assert want_c.sum() > 0
    np.testing.assert_array_equal(cnt, want_c)
    np.testing.assert_allclose(val, want_v, rtol=1e-6, atol=1e-9)


def _camera(w, h, t, yaw=0.0, f=None):
    poses = np.array([[0.0, np.sin(yaw / 2), 0.0, np.cos(yaw / 2), *t, 0.0]])
    intr = np.zeros((1, 13), np.float32)
    intr[0, :4] = [f or 0.8 * w, f or 0.8 * w, w // 2, h // 2]
    return poses, intr


# widths and heights around the 4 pixels of a load, the 512 of a step and the 4 rows of a group; one of several bands
@pytest.mark.parametrize("w,h,border", [(64, 48, 0), (511, 33, 0), (512, 30, 3), (513, 31, 0), (1027, 66, 32), (3000, 1500, 32)])
@pytest.mark.parametrize("yaw", [0.0, 0.3])
def test_edge_on_faces_and_sizes(w, h, border, yaw, rasterizer, oracle):
    print(f"[case] lift rows {w}x{h} border {border} yaw {yaw}", flush=True)
    mn, ln = synthetic.cell_grid(np.array([[-1.0, -1.0, -1.0], [0.98, 0.98, 0.98]]) + 0.01, 0.25)  # faces on x = 0, y = 0
    poses, intr = _camera(w, h, (0.0, 0.0, 2.0), yaw)
    _both(rasterizer, oracle, mn, ln, ViewSpec(w, h), poses, intr, synthetic.error_image(1, 3, h, w), border)


# the camera inside the grid: depths of a cell's nearest corners from 1e-6 on
@pytest.mark.parametrize("depth", [1e-6, 1e-4, 1e-2, 3e-2])
def test_cells_next_to_the_camera_plane(depth, rasterizer, oracle):
    print(f"[case] lift rows, nearest corners at depth {depth}", flush=True)
    w, h = 320, 200
    mn, ln = synthetic.cell_grid(np.array([[-1.0, -1.0, -1.0], [0.9, 0.9, 0.9]]), 0.3)
    poses, intr = _camera(w, h, (0.013, -0.007, depth - float(np.unique(mn[:, 2])[3])), 0.0)
    _both(rasterizer, oracle, mn, ln, ViewSpec(w, h), poses, intr, synthetic.error_image(2, 2, h, w), 0)
    poses, intr = _camera(w, h, (0.013, -0.007, depth), 0.4)
    _both(rasterizer, oracle, mn, ln, ViewSpec(w, h), poses, intr, synthetic.error_image(3, 1, h, w), 8)


def test_pixels_that_are_not_finite_stay_with_their_cells(rasterizer, oracle):
    w, h = 600, 64
    mn, ln = synthetic.cell_grid(np.array([[-2.0, -0.2, -0.1], [1.9, 0.1, 0.1]]), 0.2)
    poses, intr = _camera(w, h, (0.0, 0.0, 2.0), 0.1)
    img = synthetic.error_image(4, 3, h, w)
    img[0, 32, 100], img[1, 30, 300] = np.inf, 1e30
    val, cnt = _lift(rasterizer, mn, ln, ViewSpec(w, h), poses, intr, img, 0)
    want_v, want_c = np.zeros(len(mn), np.float32), np.zeros(len(mn), np.int32)
    oracle.lift_error(mn, ln, want_v, want_c, ViewSpec(w, h), poses, intr, img, border_pixels=0)
    np.testing.assert_array_equal(cnt, want_c)
    np.testing.assert_allclose(val, want_v, rtol=1e-5, atol=1e-9)


# cells next to the camera in an image wide enough for rows with hundreds of open columns: such a cell leaves its rows, those
# of this band and the ones behind it, and is tested pixel by pixel (two bands of rows in the two larger images)
@pytest.mark.parametrize("w,h", [(1920, 1080), (3000, 1500), (3840, 2160)])
@pytest.mark.parametrize("yaw,depth", [(0.02, 0.05), (0.3, 0.002), (-0.45, 0.01)])
def test_cells_with_many_wide_open_rows(w, h, yaw, depth, rasterizer, oracle):
    print(f"[case] lift rows {w}x{h} yaw {yaw} depth {depth}", flush=True)
    mn, ln = synthetic.cell_grid(np.array([[-0.7, -0.7, -0.7], [0.7, 0.7, 0.7]]), 0.25)
    poses, intr = _camera(w, h, (0.013, -0.007, depth - float(np.unique(mn[:, 2])[3])), yaw, f=0.52 * w)
    _both(rasterizer, oracle, mn, ln, ViewSpec(w, h), poses, intr, synthetic.error_image(5, 2, h, w), 16)


# flat cells with a face next to the camera's height: triangles with two edges so flat that they say nothing about a single
# row, beside a left or a right one
@pytest.mark.parametrize("yaw", [0.0, 0.2, -0.7])
@pytest.mark.parametrize("top", [False, True])
def test_flat_cells_with_a_face_next_to_the_camera_height(yaw, top, rasterizer, oracle):
    print(f"[case] lift rows, flat cells, yaw {yaw} top {top}", flush=True)
    w, h, n = 512, 192, 12_000
    rng = np.random.default_rng(int(100 * abs(yaw)) + top)
    width = rng.uniform(0.1, 1.0, (n, 1))
    height = width * rng.uniform(0.02, 0.4, (n, 1))
    ln = np.concatenate([width, height, width * rng.uniform(0.5, 1.0, (n, 1))], 1).astype(np.float32)
    face = np.exp(rng.uniform(np.log(1e-7), np.log(3e-5), (n, 1))) * rng.choice([-1.0, 1.0], (n, 1))
    depth = rng.uniform(0.5, 6.0, (n, 1))
    mn = np.concatenate([rng.uniform(-0.7, 0.7, (n, 1)) * depth, face - (height if top else 0.0), depth], 1).astype(np.float32)
    poses, intr = _camera(w, h, (0.0, 0.0, 0.0), yaw)
    intr[0, 2:4] = [247.3, 94.18]
    _both(rasterizer, oracle, mn, ln, ViewSpec(w, h), poses, intr, synthetic.error_image(6, 1, h, w), 0)


def _strip_of_cells(w, pixels):
    """Cells side by side, seen head-on, that each cover `pixels` columns of row 9 of an image of 19 rows."""
    h = 19
    poses, intr = _camera(w, h, (0.0, 0.0, 0.0), f=float(w))
    left = (np.arange(16, w - 16 - pixels, pixels) - w // 2 + 0.5) / w
    n = len(left)
    mn = np.stack([left, np.full(n, (8.5 - h // 2) / w), np.ones(n)], 1).astype(np.float32)
    ln = np.stack([np.full(n, pixels / w), np.full(n, 2.0 / w), np.full(n, 1e-3)], 1).astype(np.float32)
    return mn, ln, poses, intr, h


# A run of dim pixels behind bright ones of its row is a difference of large sums in 64 bits. What is left of it has to be
# good for the float that the cell's value is: with 38 bits left, one cell in 2^13 or so differs from the sequential sum's
# float, of the 59 to 246 cells here one at most. (With 26 bits left every tenth does.)
@pytest.mark.parametrize("bright,dim,w,pixels", [(1000.0, 1e-15, 1100, 10), (4e5, 1e-12, 1100, 10), (1000.0, 1000 * 2.0 ** -26, 2000, 16),
                                                 (1.0, 2.0 ** -26, 3000, 12), (1.0, 1e-3, 2000, 8), (1.0, 2.0 ** -20, 1100, 18),
                                                 (1e-3, 0.0, 1100, 10)])
def test_dim_runs_behind_bright_pixels_keep_their_bits(bright, dim, w, pixels, rasterizer, oracle):
    print(f"[case] lift rows, runs of {pixels} x {dim} behind {bright}, width {w}", flush=True)
    mn, ln, poses, intr, h = _strip_of_cells(w, pixels)
    rng = np.random.default_rng(3)
    img = (dim * rng.uniform(0.5, 1.5, (1, h, w))).astype(np.float32)
    img[0, :, :12] = bright * rng.uniform(0.5, 1.5, (h, 12))
    view = ViewSpec(w, h)
    val, cnt = _lift(rasterizer, mn, ln, view, poses, intr, img, 0)
    want_v, want_c = np.zeros(len(mn), np.float32), np.zeros(len(mn), np.int32)
    oracle.lift_error(mn, ln, want_v, want_c, view, poses, intr, img, border_pixels=0)
    assert want_c.min() >= pixels - 2
    np.testing.assert_array_equal(cnt, want_c)
    np.testing.assert_allclose(val, want_v, rtol=2.0 ** -23, atol=0.0)  # at most one unit in the last place
    assert (val != want_v).sum() <= 1
