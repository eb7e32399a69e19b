"""GPU parity of the scatter pass around the number of bins that a workgroup's 256 points may spread over.

The workgroup counts its hits in LDS, one slot per bin of the rectangle its points span in every layer, up to 5088 slots
with one hit per layer and 6144 with the 2x2 splat; in the layers that find no room its waves group their hits themselves.
The blocks here span exactly that many bins or a few more, a single bin, half of the image, or nothing that is visible;
some have hits in the coarser layers only (positions left of pixel 0), and blocks of all kinds are neighbours.
Counterpart of CountingPrepassMulti and CollectMulti, src/lib/rendering/RenderForward.cu:806-905,1011-1096.
"""
import numpy as np
import pytest

from tests.test_gpu_wide_records import _compare
from vet_amd import abi, synthetic
from vet_amd.rasterizer import make_params

pytestmark = pytest.mark.gpu

BLOCK = 256  # points of a workgroup


def _scene(w, h, layers, drop_by_radius, seed=3):
    rng = np.random.default_rng(seed)
    kinds = ["all", "bin", "all", "left", "behind", "bin", "half", "all", "left", "some", "all"]
    uv, z = [], []
    for kind in kinds:
        u, v = rng.uniform(0, w - 1, BLOCK), rng.uniform(0, h - 1, BLOCK)
        d = rng.uniform(1.0, 3.0, BLOCK)
        u[:2], v[:2] = [1.0, w - 2.0], [1.0, h - 2.0]  # the corners of the image
        if kind == "bin":
            u, v = 100 + 3 * rng.uniform(size=BLOCK), 50 + 3 * rng.uniform(size=BLOCK)
        elif kind == "half":
            u *= 0.5
        elif kind == "left":  # beside layer 0, in the first column of the layers behind it
            u = rng.uniform(-0.9, -0.6, BLOCK) - (1.0 if seed % 2 else 0.0)
        elif kind == "behind":
            d = -d
        elif kind == "some":
            d[rng.random(BLOCK) < 0.9] *= -1
        uv.append(np.stack([u, v], 1))
        z.append(d)
    uv, z = np.concatenate(uv)[:-37], np.concatenate(z)[:-37]  # the last block is not full
    position = np.concatenate([uv / w * z[:, None], z[:, None], np.exp(rng.normal(-6.5, 1.0, (len(z), 1)))], 1).astype(np.float32)
    n = len(z)
    texture, confidence, background = synthetic._descriptors(seed, n)
    scene = synthetic.Scene("slots", position, texture, confidence, background, synthetic._identity_pose((0, 0, 0)),
                            synthetic._intrinsics(float(w), float(w), 0.0, 0.0), [synthetic.ViewSpec(w, h)], num_layers=layers,
                            max_list_length=16, seed=seed)
    scene.params.update(drop_out_points_by_radius=int(drop_by_radius))
    return scene


# tiles of 16x16 pixels are the bins of these layers: 96 x 53 = 5088, 76 x 67 = 5092; 96 x 64 = 6144, 116 x 53 = 6148; up to
# 1024 slots the 2x2 splat goes by slots, beyond by first hits: 32 x 32 = 1024, 41 x 25 = 1025
@pytest.mark.parametrize("mode,tiles_x,tiles_y", [(1, 96, 53), (1, 76, 67), (2, 96, 53), (3, 96, 64), (3, 116, 53), (3, 32, 32),
                                                  (3, 41, 25)])
@pytest.mark.parametrize("layers", [1, 2, 4])
@pytest.mark.parametrize("seed", [2, 3])
def test_blocks_around_the_number_of_slots(mode, tiles_x, tiles_y, layers, seed, rasterizer, oracle):
    print(f"[case] scatter slots: mode {mode}, {tiles_x}x{tiles_y} tiles, {layers} layers, seed {seed}", flush=True)
    scene = _scene(16 * tiles_x, 16 * tiles_y, layers, drop_by_radius=seed == 2 and layers > 1, seed=seed)
    if layers == 1:
        assert int(rasterizer.layout(scene, mode).num_bins) == tiles_x * tiles_y, "the bin table changed: pick new image sizes"
    params = make_params(scene, need_point_gradient=1, render_mode=mode)
    _compare(scene, params, rasterizer, oracle, bilinear=mode == abi.RENDER_BILINEAR_BLEND)
