"""GPU parity of the list-building pass where there are few bins: its launch then has no more workgroups for crowded bins than
there can be such bins or parts of them (fragments / 257), none at all up to 256 fragments. One bin takes all points here, around
the sizes at which it needs one more."""
import numpy as np
import pytest

from tests.test_gpu_wide_records import _compare
from vet_amd import abi, synthetic
from vet_amd.rasterizer import make_params

pytestmark = pytest.mark.gpu

SIDE = 16  # one tile, in bins of 4 pixels


@pytest.mark.parametrize("mode", [1, 2, 3])
@pytest.mark.parametrize("points", [1, 256, 257, 513, 514, 1024, 1025, 1536, 1537, 8192, 8193])
def test_one_bin_takes_all_points(mode, points, rasterizer, oracle):
    print(f"[case] crowded workgroups: mode {mode}, {points} points in one bin", flush=True)
    rng = np.random.default_rng(points)
    # layer 0: the four pixels (4..7, 5); with the 2x2 splat the row behind them too
    uv = np.stack([rng.uniform(3.6 if mode != 3 else 4.0, 7.4 if mode != 3 else 6.9, points), rng.uniform(5.0, 5.4, points)], 1)
    z = np.round(rng.uniform(1.0, 3.0, (points, 1)), 2)
    position = np.concatenate([uv / SIDE * z, z, np.full((points, 1), 0.01)], 1).astype(np.float32)
    texture, confidence, background = synthetic._descriptors(points, points)
    scene = synthetic.Scene("one bin", position, texture, confidence, background, synthetic._identity_pose((0, 0, 0)),
                            synthetic._intrinsics(float(SIDE), float(SIDE), 0.0, 0.0), [synthetic.ViewSpec(SIDE, SIDE)], num_layers=1,
                            max_list_length=16, seed=points)
    _, ref = _compare(scene, make_params(scene, render_mode=mode, need_point_gradient=1), rasterizer, oracle,
                      bilinear=mode == abi.RENDER_BILINEAR_BLEND)
    counts = np.diff(ref.offsets[0].astype(np.int64)).reshape(SIDE, SIDE // 4, 4).sum(axis=2)
    assert counts[5, 1] >= points and counts.sum() == points * (4 if mode == 3 else 1)
