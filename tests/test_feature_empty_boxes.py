"""Boxes without pixels in the feature pass.  On the CPU: every label that the walk over a box's cells reads
(nscale_amd/csrc/features_rules.hpp and the clamps of k_object_features, restated) lies inside the box, for boxes of
all small shapes, empty and inverted ones among them, and the empty boxes of nsc_bounding_boxes.  On the GPU: an
empty box has no pixels, and its neighbours' features are what they are without it."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from tests._lib import ROOT

PROGRAM = r"""
#include <algorithm>
#include <climits>
#include <cstdio>
#include "features_rules.hpp"
using std::max;
using std::min;
int main() {
    const int boxes[][4] = {{INT_MAX, -1, INT_MAX, -1}, {0, -1, 0, 4}, {0, 4, 0, -1}, {3, 2, 3, 2}};
    int bad = 0, reads = 0;
    auto walk = [&](int minx, int maxx, int miny, int maxy) {
        const int bw = maxx - minx + 1, bh = maxy - miny + 1;
        const nsc::CellWalk c = nsc::cell_walk(bw, bh);
        if (c.cw <= 0) { ++bad; return; }
        for (int cy = 0; cy < c.ch; ++cy)
            for (int cx = 0; cx < c.cw; ++cx) {
                const int x = minx + cx, y = miny + cy, xs[2] = {min(x, maxx), max(x - 1, minx)},
                          ys[2] = {min(y, maxy), max(y - 1, miny)};
                for (int px : xs)
                    for (int py : ys) {
                        ++reads;
                        bad += px < minx || px > maxx || py < miny || py > maxy;
                    }
            }
    };
    for (auto& b : boxes) walk(b[0], b[1], b[2], b[3]);
    for (int bw = -3; bw <= 9; ++bw)
        for (int bh = -3; bh <= 9; ++bh) walk(2, 2 + bw - 1, 5, 5 + bh - 1);
    std::printf("%d of %d reads leave their box\n", bad, reads);
    return bad != 0;
}
"""


def test_no_read_leaves_its_box(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("no host compiler")
    src = tmp_path / "rule.cpp"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "nscale_amd", "csrc"), "-o", str(tmp_path / "rule"), str(src)],
                   check=True)
    r = subprocess.run([str(tmp_path / "rule")], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout


@pytest.mark.gpu
def test_empty_boxes_hold_nothing():
    torch = pytest.importorskip("torch")
    from nscale_amd import gpu
    rng = np.random.default_rng(1)
    lab = np.zeros((40, 50), np.int32)
    lab[3:12, 0:9] = 1
    lab[20:31, 30:50] = 3
    gray = torch.from_numpy(rng.integers(0, 256, lab.shape).astype(np.uint8)).cuda()
    d = torch.from_numpy(lab).cuda()
    boxes, _ = gpu.bounding_boxes(d, 4)  # labels 2 and 4 are absent
    boxes = torch.cat([boxes, torch.tensor([[5], [0], [-1], [0], [7]], dtype=torch.int32, device="cuda")], 1).contiguous()
    print("empty boxes", flush=True)
    got = {k: v.cpu().numpy() for k, v in gpu.object_features(d, boxes, gray).items()}
    both = boxes[:, [0, 2]].contiguous()
    exp = {k: v.cpu().numpy() for k, v in gpu.object_features(d, both, gray).items()}
    for k in exp:
        assert np.array_equal(got[k][[0, 2]], exp[k]), k
    for k in ("area", "perimeter"):
        assert not got[k][[1, 3, 4]].any(), k
