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
    # (the background's gradient is one sum over all pixels that no record takes part in; in the oracle's float32 the order of
    # its some 6000 terms of both signs alone moves it by up to 6000 x 2^-24 = 3.6e-4 of their size)
    for key in ("texture", "confidence", "points", "pose", "intrinsics"):
        err = max_rel_err(got[key].cpu().numpy(), want[key])
        assert err <= (1e-3 if key == "intrinsics" else GRAD_TOL), (key, err)  # (intrinsics: the oracle's sums are in float32)
