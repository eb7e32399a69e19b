"""Which launches of the per-pixel backward kernels cut the screen's regions into parts: calls that were measured, each on its faster
side, and either side of every line of the rule."""
import ctypes as C
import os
import subprocess

import pytest

from vet_amd import build


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    folder = tmp_path_factory.mktemp("region_rule")
    source = folder / "rule.cpp"
    source.write_text('#include "region_rule.h"\n'
                      'extern "C" int in_parts(int layers, int w, int h, double fragments, float expected, int cut)\n'
                      "{\n"
                      "    const uint32_t span = 16u << (layers - 1), x = (w + span - 1) / span, y = (h + span - 1) / span;\n"
                      "    return vetrast::regions_in_parts(layers, x, x * y, vetrast::fragments_a_pixel_may_blend(fragments, expected, w, h, cut));\n"
                      "}\n")
    library = folder / "rule.so"
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-shared", "-fPIC", "-I", build.CSRC, str(source), "-o", str(library)], check=True)
    f = C.CDLL(str(library)).in_parts
    f.argtypes = [C.c_int, C.c_int, C.c_int, C.c_double, C.c_float, C.c_int]
    return f


@pytest.mark.parametrize("layers,w,h,fragments,expected,cut,want", [
    # a cloud of which a view sees a fifteenth: what is seen counts where the caller has said it
    (4, 1920, 1080, 10_000_000, 660_000, 16, 0), (4, 1920, 1080, 22_000_000, 1_290_000, 16, 0),
    # few regions, but short lists, or small regions: parts cost more than they give
    (4, 1237, 701, 777_777, 0, 16, 0), (4, 700, 500, 315_000, 164_000, 16, 0), (3, 480, 270, 200_000, 96_000, 16, 0),
    (3, 500, 380, 180_000, 0, -1, 0), (2, 500, 380, 3_000_000, 0, -1, 0), (1, 1920, 1080, 20_000_000, 0, 16, 0),
    # the same list where a row of regions gives an XCD columns, diagonals, or regions from all over
    (4, 960, 540, 2_000_000, 640_000, 16, 1), (4, 1920, 1080, 8_000_000, 2_560_000, -1, 0), (4, 1237, 701, 3_000_000, 1_070_000, 16, 0),
    (4, 1920, 1080, 8_000_000, 4_800_000, -1, 1), (4, 700, 500, 1_300_000, 665_000, 16, 0), (4, 700, 500, 2_100_000, 1_100_000, 16, 1),
    # long lists, shipped crops, large regions, no more regions than XCDs or few more
    (4, 1920, 1080, 10_000_000, 9_700_000, 16, 1), (4, 512, 512, 8_000_000, 506_000, -1, 1), (5, 1920, 1080, 1_800_000, 800_000, 16, 1),
    (5, 228, 228, 2_300_000, 40_000, -1, 1), (4, 203, 155, 240_000, 34_000, -1, 1), (4, 384, 384, 4_000_000, 70_000, -1, 1),
    # the cut bounds a list; either side of the lines
    (4, 1920, 1080, 10_000_000, 0, 3, 0), (4, 1920, 1080, 10_000_000, 0, 4, 1), (4, 1024, 1024, 1.0 * 2**20, 0, 0, 1), (4, 1024, 1024, 0.99 * 2**20, 0, 0, 0),
    (4, 512, 512, 3.5 * 2**18, 0, -1, 1), (4, 512, 512, 3.49 * 2**18, 0, -1, 0), (4, 640, 384, 5.99 * 640 * 384, 0, -1, 0), (4, 640, 384, 6 * 640 * 384, 0, -1, 1),
    (4, 512, 384, 0, 0, -1, 1), (4, 512, 385, 0, 0, -1, 0), (5, 2048, 2048, 0, 0, -1, 1), (5, 2048, 2049, 0, 0, -1, 0)])
def test_regions_in_parts(rule, layers, w, h, fragments, expected, cut, want):
    assert rule(layers, w, h, fragments, expected, cut) == want
