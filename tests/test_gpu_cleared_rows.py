"""GPU parity of gradient rows behind a texture index, which start at zero whatever was in them: cleared by one workgroup of the
per-pixel kernel (up to 16384 words), by all of them (up to that many words each), or by launches of their own where the image is
too small for so many rows. A 16x16 image has 8 workgroups: 131072 words."""
import ctypes as C

import numpy as np
import pytest
import torch

from tests.helpers import max_rel_err
from vet_amd import abi, synthetic
from vet_amd.rasterizer import DeviceScene, make_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [1, 2, 3])
@pytest.mark.parametrize("points", [1, 4096, 4097, 16385, 32768, 32769, 131073])
def test_rows_start_at_zero(mode, points, rasterizer, oracle):
    print(f"[case] cleared rows: mode {mode}, {points} points", flush=True)
    scene = synthetic.tiny_scene(num_points=points, w=16, h=16, num_layers=1, K=4, seed=points)
    scene.index = np.arange(points, dtype=np.int32)[::-1].copy()
    scene.index[::3] //= 2
    params = make_params(scene, render_mode=mode, need_point_gradient=1)
    ref = oracle.forward(scene, params)
    grad_out = scene.grad_out()
    want = oracle.backward(ref, grad_out, want_cameras=True)
    res = rasterizer.forward(DeviceScene(scene), params, save_for_backward=True)
    got = rasterizer.backward(res, [torch.from_numpy(g).cuda() for g in grad_out], want_cameras=True)
    args = got.pop("_args")
    for t in got.values():
        t.fill_(float("nan"))
    abi.check(rasterizer.lib.vetrast_backward(rasterizer.ctx, C.byref(args), rasterizer._stream()), "backward")
    torch.cuda.synchronize()
    for key in ("texture", "confidence"):
        g = got[key].cpu().numpy()
        assert (g[want[key] == 0] == 0).all(), key  # rows no fragment belongs to
    np.testing.assert_array_equal(got["point_count"].cpu().numpy(), want["point_count"])
    for key in ("texture", "confidence", "points", "pose"):
        assert max_rel_err(got[key].cpu().numpy(), want[key]) <= 1e-4, key  # 32-bit sums in another order
