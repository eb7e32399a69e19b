"""The backward scratch of the workspace: 32 bytes for a point and layer in every mode (the four corners of the 2x2 splat share
them) and, with the 2x2 splat only, a float4 for every pixel behind them; there the block is no smaller than 32 bytes for each
corner, and no larger unless the pixels do not fit into what the corners leave."""
import ctypes as C

import pytest

from vet_amd import abi


def _align(n):
    return (n + 255) // 256 * 256


@pytest.mark.parametrize("mode", [abi.RENDER_FULL_BLEND, abi.RENDER_FUZZY_BLEND, abi.RENDER_BILINEAR_BLEND])
@pytest.mark.parametrize("points,views,layers,w,h", [(0, 1, 1, 16, 16), (1, 1, 4, 17, 33), (60_007, 1, 4, 203, 155), (2_000_000, 4, 4, 512, 512),
                                                     (5_000_001, 2, 5, 1920, 1080)])
def test_backward_scratch(mode, points, views, layers, w, h):
    lay = abi.WorkspaceLayout()
    assert abi.load_library().vetrast_workspace_layout_for_mode(points, views, layers, w, h, mode, C.byref(lay)) == 0
    pixels = 256 * lay.layer_tile_base[layers]
    want = _align(points * layers * 32)
    if mode == abi.RENDER_BILINEAR_BLEND:
        want = max(want + pixels * 16, _align(4 * points * layers * 32))
    assert lay.background_partial_base - lay.partial_base == want
    # what is folded into the records' place behind the per-point kernel: 64 rows of 160 bytes for each view of a round, where there
    # are more than 256 workgroups of points
    if points > 256 * 256:
        assert points * layers * 32 >= lay.view_lanes * 64 * 160


@pytest.mark.parametrize("mode", [abi.RENDER_FULL_BLEND, abi.RENDER_FUZZY_BLEND, abi.RENDER_BILINEAR_BLEND])
@pytest.mark.parametrize("points,views,layers,w,h", [(0, 1, 1, 16, 16), (1, 1, 4, 17, 33), (777_777, 2, 4, 1237, 701), (60_007, 1, 4, 203, 155),
                                                     (100_000, 3, 5, 1000, 700), (2_000_000, 4, 4, 1920, 1080)])
def test_background_rows_take_what_callers_have_reserved(mode, points, views, layers, w, h):
    """The rows of background-gradient sums have 128 bytes for each workgroup there can be (a tile of each layer in regions of one
    coarsest tile, eight regions at a time, four workgroups to a tile), and 8 KiB: buffers of that size have to stay large enough."""
    lay = abi.WorkspaceLayout()
    assert abi.load_library().vetrast_workspace_layout_for_mode(points, views, layers, w, h, mode, C.byref(lay)) == 0
    span = 16 << (layers - 1)
    regions = ((w + span - 1) // span) * ((h + span - 1) // span)
    groups = (regions + 7) // 8 * 8 * 4 * sum(4**l for l in range(layers))
    backward_block = lay.background_partial_base - lay.partial_base + _align(groups * 128 + 256 * 32)
    forward_block = lay.forward_only_bytes - lay.log_base - lay.lane_scratch_stride * (lay.view_lanes - 1)
    assert lay.lane_scratch_stride == max(forward_block, backward_block)
