"""GPU parity of the gradients over the layouts of the gradient records: layer after layer and point after point, one to
four channels, one to five layers (the per-point kernel takes two at a time with one hit per layer), one point to a few
workgroups, points on the image border (fewer than four corners), a texture index, several views and camera gradients.
Counterpart of BlendBackwards2<C> / BlendBackwardsBilinear<C>, src/lib/rendering/RenderBackward.cu:1083-1513,2893-3232.
"""
import numpy as np
import pytest
import torch

from tests.helpers import max_rel_err
from vet_amd import synthetic
from vet_amd.rasterizer import DeviceScene, make_params

pytestmark = pytest.mark.gpu

GRAD_TOL = 1e-4  # 32-bit sums in another order, against the largest entry of the tensor
# The background's gradient is one sum over all pixels of transmittance x upstream gradient, in 32 bits: each term goes through
# eight additions inside its workgroup and fewer than a hundred behind it; FUZZY_BLEND works its transmittance out anew, with two
# roundings for each of the fragments in front (beyond some 40 nothing to speak of is left). 180 x 2^-24 = 1.1e-5 of the terms'
# absolute sum if all of them erred one way.
BACKGROUND_TOL = 1.1e-5


def _transmittance(ref, mode):
    """What is left for the background, per layer [B,h,w] in float64. FULL_BLEND and BILINEAR_BLEND: what the forward pass left,
    and nothing where the 2x2 splat stopped early. FUZZY_BLEND: the backward pass forms buckets all along a list
    (src/lib/rendering/RenderBackward.cu:628-720)."""
    scene, left = ref.scene, []
    for l, (w, h) in enumerate(ref.sizes):
        base = ref.layer_base(l)
        T = ref.weight[:, base:base + w * h].astype(np.float64).reshape(-1, h, w)
        if mode == 3:
            T = np.where(T < 0.001, 0.0, T)
        if mode == 2:
            K = ref.params.debug_max_list_length
            for b, y, x in np.argwhere(np.diff(ref.offsets[:, base:base + w * h + 1].astype(np.int64)).reshape(-1, h, w) > 1):
                keys = ref.pixel_list(b, l, x, y)[:K if K > 0 else None]
                depth = (keys >> np.uint64(32)).astype(np.uint32).view(np.float32)
                conf = scene.confidence[scene.index[(keys & np.uint64(0xFFFFFFFF)).astype(np.int64)]].astype(np.float64)
                T[b, y, x], j = 1.0, 0
                while j < len(keys):
                    e = j + int(np.argmin(np.append(depth[j:] - depth[j] < np.float32(ref.params.depth_accept_blend), False)))
                    T[b, y, x] *= 1.0 - conf[j:e].mean()
                    j = e
        left.append(T)
    return left


@pytest.mark.parametrize("mode", [1, 2, 3])
@pytest.mark.parametrize("points,size,layers,channels,cut,views,point_major", [
    (1, (16, 16), 1, 4, -1, 1, False), (255, (17, 33), 2, 1, 3, 1, False), (257, (40, 31), 3, 2, 1, 2, True),
    (3000, (97, 49), 4, 3, 4, 5, False), (3000, (97, 49), 4, 4, -1, 1, True), (3001, (130, 70), 5, 4, 8, 3, True),
    (5000, (64, 64), 5, 4, 2, 1, False)])
def test_gradients_for_every_record_layout(mode, points, size, layers, channels, cut, views, point_major, rasterizer, oracle):
    print(f"[case] gradient records: mode {mode}, {points} points, {size}, {layers} layers, {channels} channels, cut {cut}", flush=True)
    rng = np.random.default_rng(points + layers)
    scene = synthetic.tiny_scene(num_points=points, w=size[0], h=size[1], num_layers=layers, K=cut, seed=points)
    scene.texture, scene.background = scene.texture[:channels].copy(), scene.background[:channels].copy()
    scene.views = [synthetic.ViewSpec(size[0], size[1], image_index=b, crop_transform=(1.0, 1.0, 3.0 * b, -2.5 * b, 0.0)) for b in range(views)]
    scene.poses_se3 = np.repeat(scene.poses_se3[:1], views, axis=0).copy()
    scene.index = np.arange(points, dtype=np.int32)
    scene.index[::5] //= 2
    scene.dropout = (rng.random((views, points)) < 0.2).astype(np.float32)
    params = make_params(scene, render_mode=mode, need_point_gradient=1)
    ref = oracle.forward(scene, params)
    grad_out = scene.grad_out()
    want = oracle.backward(ref, grad_out, want_cameras=True)
    if point_major:  # what makes the call lay the records out point after point
        for l in range(layers):
            params.expected_fragments[l] = max(0.2 * points, 0.01)
    res = rasterizer.forward(DeviceScene(scene), params, save_for_backward=True)
    got = rasterizer.backward(res, [torch.from_numpy(g).cuda() for g in grad_out], want_cameras=True)
    torch.cuda.synchronize()
    for l in range(layers):
        np.testing.assert_array_equal(res.out[l].cpu().numpy(), ref.out[l])
    for key in ("texture", "confidence", "points", "pose", "intrinsics"):
        err = max_rel_err(got[key].cpu().numpy(), want[key])
        assert err <= (1e-3 if key == "intrinsics" else GRAD_TOL), (key, err)  # (intrinsics: the oracle's sums are in float32)
    terms = [(T[:, None] * g.astype(np.float64)) for T, g in zip(_transmittance(ref, mode), grad_out)]
    off = got["background"].cpu().numpy() - sum(t.sum(axis=(0, 2, 3)) for t in terms)
    assert (np.abs(off) <= BACKGROUND_TOL * sum(np.abs(t).sum(axis=(0, 2, 3)) for t in terms)).all(), off
