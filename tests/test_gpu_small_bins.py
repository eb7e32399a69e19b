"""GPU parity of the list-building pass in bins of 4 and 16 pixels that one wave builds: with more than 64 fragments the pixels
take turns, 16 or 4 ranks of every list at a time. Lists of one length and of very different ones, around these numbers, with and
without a cut."""
import numpy as np
import pytest

from tests.test_gpu_wide_records import _compare
from vet_amd import abi, synthetic
from vet_amd.rasterizer import make_params

pytestmark = pytest.mark.gpu


def _lists(pixels, rng):
    """Lengths of the lists of a bin, bin after bin; up to 256 fragments in each."""
    turn = 64 // pixels
    for n in (turn - 1, turn, turn + 1, 2 * turn, 4 * turn - 1, 4 * turn):
        yield [n] * pixels
    for where in (0, pixels - 1):
        for n in (63, 64, 65, 128, 129, 255, 256):
            yield [n if k == where else 0 for k in range(pixels)]
    yield [1] * (pixels - 1) + [64]
    yield [64 - pixels + 1] + [1] * (pixels - 1)
    yield [65 - pixels + 1] + [1] * (pixels - 1)
    for _ in range(20):
        total = int(rng.integers(65, 257))
        yield np.bincount(rng.choice(pixels, total, p=rng.dirichlet([0.3] * pixels)), minlength=pixels).tolist()


@pytest.mark.parametrize("mode", [1, 2, 3])
@pytest.mark.parametrize("K", [-1, 16, 17, 100])
@pytest.mark.parametrize("side,pixels", [(16, 4), (128, 16)])
def test_pixels_of_a_small_bin_take_turns(mode, K, side, pixels, rasterizer, oracle):
    print(f"[case] small bins: mode {mode}, K {K}, {pixels} pixels", flush=True)
    rng = np.random.default_rng(pixels)
    uv = []
    for b, lengths in enumerate(_lists(pixels, rng)):
        # every second row and, with the 2x2 splat, a point's four pixels in its own and the row behind it
        x0, y0 = b * pixels % side, b * pixels // side * 2 % side if side == 128 else b * pixels // side
        for k, n in enumerate(lengths):
            n = n if mode != 3 else (n + 1) // 2
            uv.append(np.stack([x0 + k + rng.uniform(0.0, 0.4, n), y0 + rng.uniform(0.0, 0.4, n)], 1))
    uv = np.concatenate(uv)
    uv = uv[rng.permutation(len(uv))]
    n = len(uv)
    z = np.round(rng.uniform(1.0, 3.0, (n, 1)), 2)  # some at the same depth
    position = np.concatenate([uv / side * z, z, np.full((n, 1), 0.01)], 1).astype(np.float32)
    texture, confidence, background = synthetic._descriptors(n, n)
    scene = synthetic.Scene("small bins", position, texture, confidence, background, synthetic._identity_pose((0, 0, 0)),
                            synthetic._intrinsics(float(side), float(side), 0.0, 0.0), [synthetic.ViewSpec(side, side)], num_layers=1,
                            max_list_length=K, seed=n)
    _, ref = _compare(scene, make_params(scene, render_mode=mode, need_point_gradient=1), rasterizer, oracle,
                      bilinear=mode == abi.RENDER_BILINEAR_BLEND)
    counts = np.diff(ref.offsets[0].astype(np.int64)).reshape(-1, pixels).sum(axis=1)
    assert ((counts > 64) & (counts <= 256)).sum() >= 20
