"""GPU parity of the per-pixel backward kernels where the regions of the screen are cut into parts that different XCDs take, and where
they stay whole (test_region_rule_cpu.py has the rule). Every pixel's records must be there, and the sums over pixels must come out
whichever workgroup added them up."""
import numpy as np
import pytest
import torch

from tests.helpers import max_rel_err
from vet_amd import synthetic
from vet_amd.rasterizer import DeviceScene, make_params

pytestmark = pytest.mark.gpu


# (width, height, layers, points, cut): 1 region of 5, 3, 2 and 1 layers; 8, 9, 64 and 65 regions; long lists, 66 regions; four layers with 4, 12
# and 16 regions (parts, parts, whole), 16 in rows of eight with lists below and from the line on, five layers with strips of split tiles
@pytest.mark.parametrize("mode", [1, 2, 3])
@pytest.mark.parametrize("w,h,layers,points,cut", [(171, 133, 5, 20_000, -1), (61, 57, 3, 3_000, 40), (31, 30, 2, 3_000, -1), (16, 9, 1, 500, 16),
                                                   (250, 118, 3, 20_000, 16), (180, 190, 3, 20_000, -1), (512, 511, 3, 30_000, 16),
                                                   (832, 316, 3, 30_000, 16), (350, 176, 2, 260_000, 3), (350, 176, 2, 260_000, 20),
                                                   (203, 155, 4, 40_000, -1), (500, 371, 4, 20_000, 16), (500, 386, 4, 20_000, 16), (1021, 131, 4, 30_000, 16),
                                                   (1021, 131, 4, 150_000, 16), (290, 270, 5, 120_000, 12)])
def test_every_region_is_taken(mode, w, h, layers, points, cut, rasterizer, oracle):
    print(f"[case] region parts: mode {mode}, {w}x{h}, {layers} layers, {points} points, cut {cut}", flush=True)
    scene = synthetic.config2(num_points=points, seed=w, w=w, h=h, num_layers=layers, K=cut)
    params = make_params(scene, render_mode=mode, need_point_gradient=1)
    ref = oracle.forward(scene, params, num_threads=8)
    grad_out = scene.grad_out()
    want = oracle.backward(ref, grad_out, num_threads=8)
    res = rasterizer.forward(DeviceScene(scene), params, save_for_backward=True)
    got = rasterizer.backward(res, [torch.from_numpy(g).cuda() for g in grad_out])
    torch.cuda.synchronize()
    np.testing.assert_array_equal(got["point_count"].cpu().numpy(), want["point_count"])
    for key in ("texture", "confidence", "points"):
        assert max_rel_err(got[key].cpu().numpy(), want[key]) <= 1e-4, key  # 32-bit sums in another order
    # A pixel adds T g to the background's gradient (not where the 2x2 splat's blend has stopped in front of it), in fewer than 64
    # additions one after the other (10 inside a workgroup, then rows), so it is off by at most 64 roundings of 2^-24 of sum |T g|.
    # FUZZY_BLEND's T is not the forward pass's: there the check's own sum stands in, of T g with T <= 1, one pixel after the other.
    weights = [ref.weight[0, ref.layer_base(l): ref.layer_base(l) + gw * gh].reshape(gh, gw).astype(np.float64) for l, (gw, gh) in enumerate(ref.sizes)]
    weights = [np.ones_like(t) if mode == 2 else np.where(t < np.float32(0.001), 0.0, t) if mode == 3 else t for t in weights]
    additions = 64 + (sum(t.size for t in weights) if mode == 2 else 0)
    for c in range(scene.num_channels):
        terms = [t * g[0, c] for t, g in zip(weights, grad_out)]
        exact = float(want["background"][c]) if mode == 2 else sum(t.sum() for t in terms)
        assert abs(float(got["background"][c]) - exact) <= additions * 2.0**-24 * sum(np.abs(t).sum() for t in terms)
