"""GPU parity of the list-building pass around the sizes at which a bin changes hands.

A bin of up to 256 records is built by a wave, of up to 1024 by a workgroup at once, of up to 8192 by several workgroups that
take a run of its pixels each, beyond that, or where a list does not fit by itself, in memory; with a cut of up to 64 also from 1024
on where it has 4 or 16 pixels. The spots here hold a number of
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
LIMITS = [64, 256, 512, 1024, 8192]
SPREAD = [4, 8, 1540, 2048, 3100, 5000, 7300] + [n + d for n in LIMITS for d in (-1, 0, 1)]
IN_A_PIXEL = [64, 65, 128, 129, 256, 257, 1024, 1025]


def _spots(hits):
    """Points of every spot that is spread over a tile. With four hits per layer a point is four records (a pixel away from the
    tile's border all of them lie in the tile): next to a limit the nearest multiples of four."""
    return [n if hits == 1 else (n // 4 if n not in [m + 1 for m in LIMITS] else n // 4 + 1) for n in SPREAD]


def _scene(K, hits, seed=5):
    rng = np.random.default_rng(seed)
    uv, tiles = [], rng.permutation((SIDE // TILE) ** 2)
    for k, n in enumerate(_spots(hits) + [max(1, n // hits) for n in IN_A_PIXEL]):
        corner = np.array([tiles[k] % (SIDE // TILE), tiles[k] // (SIDE // TILE)]) * TILE
        if k < len(SPREAD):
            spot = corner + rng.uniform(1.0, TILE - 2.0, (n, 2))
        else:  # in one pixel and, for a bin of more than that list, the tile
            spot = np.concatenate([corner + 5 + rng.uniform(0.0, 0.4, (n, 2)), corner + rng.uniform(1.0, TILE - 2.0, (200, 2))])
        uv.append(spot)
    everywhere = rng.uniform(0, SIDE - 1, (3000, 2))  # and a few in the other tiles
    own = np.zeros((SIDE // TILE, SIDE // TILE), bool)
    own[tiles[:len(SPREAD)] // (SIDE // TILE), tiles[:len(SPREAD)] % (SIDE // TILE)] = True
    near = np.floor((everywhere[:, None] + [[-1, -1], [-1, 1.5], [1.5, -1], [1.5, 1.5]]) / TILE).astype(int).clip(0, SIDE // TILE - 1)
    uv.append(everywhere[~own[near[..., 1], near[..., 0]].any(axis=1)])
    uv = np.concatenate(uv)
    uv = uv[rng.permutation(len(uv))]
    n = len(uv)
    z = np.round(rng.uniform(1.0, 3.0, (n, 1)), 2)  # some at the same depth
    position = np.concatenate([uv / SIDE * z, z, np.full((n, 1), 0.01)], 1).astype(np.float32)
    texture, confidence, background = synthetic._descriptors(seed, n)
    return synthetic.Scene("bins", position, texture, confidence, background, synthetic._identity_pose((0, 0, 0)),
                           synthetic._intrinsics(float(SIDE), float(SIDE), 0.0, 0.0), [synthetic.ViewSpec(SIDE, SIDE)], num_layers=4,
                           max_list_length=K, seed=seed)


def _has_its_sizes(ref, hits):
    """Layer 0 is built in tiles: there is one with each of the numbers of records."""
    counts = np.diff(ref.offsets[0, :SIDE * SIDE + 1].astype(np.int64)).reshape(SIDE // TILE, TILE, SIDE // TILE, TILE).sum(axis=(1, 3))
    want = {n * hits for n in _spots(hits)}
    assert want <= set(counts.ravel().tolist()), sorted(want - set(counts.ravel().tolist()))
    for n in LIMITS:
        assert {n - hits if hits == 4 else n - 1, n, n + hits if hits == 4 else n + 1} <= want, n


@pytest.mark.parametrize("mode", [1, 2, 3])
@pytest.mark.parametrize("K", [-1, 1, 16, 64, 100])
def test_bins_around_the_sizes_of_their_ways(mode, K, rasterizer, oracle):
    print(f"[case] bin sizes: mode {mode}, K {K}", flush=True)
    hits = 4 if mode == 3 else 1
    scene = _scene(K, hits)
    _, ref = _compare(scene, make_params(scene, render_mode=mode, need_point_gradient=1), rasterizer, oracle,
                      bilinear=mode == abi.RENDER_BILINEAR_BLEND)
    _has_its_sizes(ref, hits)
