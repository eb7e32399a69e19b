"""GPU parity of the list-building pass around the sizes at which a bin changes hands.

A bin of up to 256 records is built by a wave, of up to 1024 by a workgroup at once, of up to 8192 by several workgroups that
take a run of its pixels each, beyond that, or where a list does not fit by itself, in memory. The spots here hold a number of
points next to these sizes, spread over a 16x16 pixel tile of layer 0 (or within a pixel: lists as long as the bin), and fall
into bins of 64, 16 and 4 pixels in the layers behind it. The cut of the longest lists takes the K smallest keys as they pass
(K <= 64) or sorts lists in full. Counterpart of SegmentedSortBitonicHelper2 and BlendMulti,
src/lib/rendering/AlphaListSort.cu:601-703, src/lib/rendering/RenderForward.cu:1303-1357.
"""
import numpy as np
import pytest

from tests.test_gpu_wide_records import _compare
from vet_amd import abi, synthetic
from vet_amd.rasterizer import make_params

pytestmark = pytest.mark.gpu

SIDE, TILE = 512, 16
SPREAD = [1, 2, 63, 64, 65, 255, 256, 257, 511, 512, 513, 1023, 1024, 1025, 1537, 2048, 3100, 8191, 8193]
IN_A_PIXEL = [64, 65, 128, 129, 256, 257, 1024, 1025]


def _scene(K, hits, seed=5):
    """With four hits per layer a spot of n points is a bin of 4 n records in layer 0: the same numbers, a quarter of the points
    each (a point a pixel away from the tile's border has all of its hits in the tile)."""
    rng = np.random.default_rng(seed)
    uv, tiles = [], rng.permutation((SIDE // TILE) ** 2)
    for k, n in enumerate(SPREAD + IN_A_PIXEL):
        corner = np.array([tiles[k] % (SIDE // TILE), tiles[k] // (SIDE // TILE)]) * TILE
        n = max(1, n // hits)
        if k < len(SPREAD):
            spot = corner + rng.uniform(1.0, TILE - 2.0, (n, 2))
        else:  # in one pixel and, for a bin of more than that list, the tile
            spot = np.concatenate([corner + 5 + rng.uniform(0.0, 0.4, (n, 2)), corner + rng.uniform(1.0, TILE - 2.0, (200, 2))])
        uv.append(spot)
    uv.append(rng.uniform(0, SIDE - 1, (3000, 2)))  # and a few everywhere
    uv = np.concatenate(uv)
    uv = uv[rng.permutation(len(uv))]
    n = len(uv)
    z = np.round(rng.uniform(1.0, 3.0, (n, 1)), 2)  # some at the same depth
    position = np.concatenate([uv / SIDE * z, z, np.full((n, 1), 0.01)], 1).astype(np.float32)
    texture, confidence, background = synthetic._descriptors(seed, n)
    return synthetic.Scene("bins", position, texture, confidence, background, synthetic._identity_pose((0, 0, 0)),
                           synthetic._intrinsics(float(SIDE), float(SIDE), 0.0, 0.0), [synthetic.ViewSpec(SIDE, SIDE)], num_layers=4,
                           max_list_length=K, seed=seed)


@pytest.mark.parametrize("mode", [1, 2, 3])
@pytest.mark.parametrize("K", [-1, 1, 16, 64, 100])
def test_bins_around_the_sizes_of_their_ways(mode, K, rasterizer, oracle):
    print(f"[case] bin sizes: mode {mode}, K {K}", flush=True)
    scene = _scene(K, 4 if mode == 3 else 1)
    _compare(scene, make_params(scene, render_mode=mode, need_point_gradient=1), rasterizer, oracle,
             bilinear=mode == abi.RENDER_BILINEAR_BLEND)
